// copy_out.h -- large device arrays to pageable host memory.
//
// hipMemcpyAsync to pageable memory goes through one thread that copies out of
// a staging buffer and takes the destination's page faults: 16 GB/s into
// touched pages, 9 into fresh ones, of the 40 that pinned memory receives.
// Here the array comes in 2 MB chunks through 8 pinned slots, and 4 threads
// copy them out (ms for 8 / 33 / 100 MB, fresh pages: 0.81 / 3.74 / 10.1 ->
// 0.37 / 1.07 / 2.72; touched ones 0.49 / 2.03 / 6.2 -> 0.29 / 0.90 / 2.62).
// 1 MB chunks took 1.41 and 3.43 ms (33 and 100 MB), 8 threads what 4 do.
//
// The slots are the process's, not a context's: pinning them and the first
// touch of their pages cost 1 to 2 ms, more than one copy into touched pages
// gains up to 24 MB (a new context's first copy of 8 / 16 / 24 / 33 MB with
// slots of its own 1.43 / 2.65 / 2.71 / 4.82, with these 0.34 / 0.54 / 0.73 /
// 3.00, without any 0.50 / 0.94 / 1.41 / 8.77; 33 MB into fresh pages).
#ifndef PHASECON_COPY_OUT_H
#define PHASECON_COPY_OUT_H
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <exception>
#include <mutex>
#include <thread>

namespace phasecon {

// A context's large copies.  The pinned slots are shared by the process (by
// the contexts of a library): a set of 16 MB is pinned at the first large copy
// and another for each copy at the same time, up to kSets (further ones go
// without), and all are freed with the last context that has used them.  The
// events are the context's, of its device.
class CopyOut {
 public:
  CopyOut() = default;
  CopyOut(const CopyOut&) = delete;
  CopyOut& operator=(const CopyOut&) = delete;
  ~CopyOut() {
    for (hipEvent_t e : ev_)
      if (e) (void)hipEventDestroy(e);
    if (!user_) return;
    Pool& p = pool();
    std::lock_guard<std::mutex> lock(p.m);
    if (--p.users) return;
    for (char*& b : p.buf) {
      if (b) (void)hipHostFree(b);
      b = nullptr;
    }
  }

  // src (device) to dst (host), after the work on `s`.  The caller
  // synchronizes `s` before it reads dst, as after hipMemcpyAsync.  Below
  // kMin, into memory the runtime knows (pinned or device), or where no slots
  // can be had, it is hipMemcpyAsync.
  hipError_t operator()(void* dst, const void* src, size_t bytes, hipStream_t s) {
    if (bytes < kMin || known(dst) || !make())
      return hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, s);
    char** const set = acquire();
    if (!set) return hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, s);
    const hipError_t rc = staged(*set, dst, src, bytes, s);
    Pool& p = pool();
    std::lock_guard<std::mutex> lock(p.m);
    p.busy[set - p.buf] = false;
    return rc;
  }

 private:
  static constexpr size_t kMin = 8u << 20, kChunk = 2u << 20;
  static constexpr int kSlots = 8, kThreads = 4, kSets = 4;
  static_assert(kSlots % kThreads == 0, "a slot belongs to one thread");

  struct Pool {
    std::mutex m;
    char* buf[kSets] = {};
    bool busy[kSets] = {};
    int users = 0;  // contexts that have used the slots
  };
  // never destroyed: contexts may be, when the process ends
  static Pool& pool() {
    static Pool* p = new Pool;
    return *p;
  }

  // Returns with the slots at buf empty and nothing of them in flight.
  hipError_t staged(char* buf, void* dst, const void* src, size_t bytes, hipStream_t s) {
    int dev = 0;
    hipError_t rc = hipGetDevice(&dev);
    if (rc != hipSuccess) return rc;
    const int n = (int)((bytes + kChunk - 1) / kChunk);
    const auto issue = [&](int c) {
      const size_t o = kChunk * c;
      const hipError_t e =
          hipMemcpyAsync(buf + kChunk * (c % kSlots), (const char*)src + o,
                         std::min(kChunk, bytes - o), hipMemcpyDeviceToHost, s);
      return e == hipSuccess ? hipEventRecord(ev_[c % kSlots], s) : e;
    };
    for (int c = 0; c < std::min(n, kSlots); ++c)
      if ((rc = issue(c)) != hipSuccess) {
        (void)hipStreamSynchronize(s);  // the slots are free again
        return rc;
      }
    // thread t has the chunks c = t mod kThreads and so, kSlots being a
    // multiple of kThreads, its own slots: it refills each when it is empty
    hipError_t err[kThreads] = {};
    const auto work = [&](int t) {
      err[t] = hipSetDevice(dev);
      for (int c = t; c < n && err[t] == hipSuccess; c += kThreads) {
        if ((err[t] = hipEventSynchronize(ev_[c % kSlots])) != hipSuccess) break;
        const size_t o = kChunk * c;
        std::memcpy((char*)dst + o, buf + kChunk * (c % kSlots), std::min(kChunk, bytes - o));
        if (c + kSlots < n) err[t] = issue(c + kSlots);
      }
    };
    std::thread th[kThreads];
    int started = 1;
    try {
      for (; started < kThreads; ++started) th[started] = std::thread(work, started);
    } catch (const std::exception&) {
      // no thread or no memory for one: the shares without are this one's
    }
    work(0);
    for (int t = started; t < kThreads; ++t) work(t);
    for (int t = 1; t < started; ++t) th[t].join();
    for (hipError_t e : err)
      if (e != hipSuccess) rc = e;
    if (rc != hipSuccess) (void)hipStreamSynchronize(s);
    return rc;
  }

  static bool known(const void* p) {
    hipPointerAttribute_t a;
    if (hipPointerGetAttributes(&a, p) == hipSuccess) return a.type != hipMemoryTypeUnregistered;
    (void)hipGetLastError();  // plain host memory
    return false;
  }

  bool make() {
    for (hipEvent_t& e : ev_)
      if (!e && hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) {
        e = nullptr;
        (void)hipGetLastError();
        return false;
      }
    return true;
  }

  // A set of slots for this copy alone; null where all are taken or another
  // cannot be pinned.
  char** acquire() {
    Pool& p = pool();
    std::lock_guard<std::mutex> lock(p.m);
    int i = 0;
    while (i < kSets && p.buf[i] && p.busy[i]) ++i;  // pinned in order
    if (i == kSets) return nullptr;
    if (!p.buf[i]) {
      void* b = nullptr;
      if (hipHostMalloc(&b, kSlots * kChunk, hipHostMallocPortable) != hipSuccess) {
        (void)hipGetLastError();
        return nullptr;
      }
      p.buf[i] = static_cast<char*>(b);
    }
    if (!user_) ++p.users;
    user_ = true;
    p.busy[i] = true;
    return &p.buf[i];
  }

  bool user_ = false;
  hipEvent_t ev_[kSlots] = {};
};

}  // namespace phasecon
#endif
