// copy_out.h -- large device arrays to pageable host memory.
//
// hipMemcpyAsync to pageable memory goes through one thread that copies out of
// a staging buffer and takes the destination's page faults: 16 GB/s into
// touched pages, 9 into fresh ones, of the 40 that pinned memory receives.
// Here the array comes in 2 MB chunks through 8 pinned slots, and 4 threads
// copy them out (ms for 8 / 33 / 100 MB, fresh pages: 0.81 / 3.74 / 10.1 ->
// 0.37 / 1.07 / 2.72; touched ones 0.49 / 2.03 / 6.2 -> 0.29 / 0.90 / 2.62).
// 1 MB chunks took 1.41 and 3.43 ms (33 and 100 MB), 8 threads what 4 do.
#ifndef PHASECON_COPY_OUT_H
#define PHASECON_COPY_OUT_H
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <system_error>
#include <thread>

namespace phasecon {

// A context's staging slots: made at its first large copy, freed with it.
class CopyOut {
 public:
  CopyOut() = default;
  CopyOut(const CopyOut&) = delete;
  CopyOut& operator=(const CopyOut&) = delete;
  ~CopyOut() {
    for (hipEvent_t e : ev_)
      if (e) (void)hipEventDestroy(e);
    if (buf_) (void)hipHostFree(buf_);
  }

  // src (device) to dst (host), after the work on `s`.  The caller
  // synchronizes `s` before it reads dst, as after hipMemcpyAsync.  Below
  // kMin, into memory the runtime knows (pinned or device), or where no slots
  // can be had, it is hipMemcpyAsync.
  hipError_t operator()(void* dst, const void* src, size_t bytes, hipStream_t s) {
    if (bytes < kMin || known(dst) || !make())
      return hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, s);
    int dev = 0;
    hipError_t rc = hipGetDevice(&dev);
    if (rc != hipSuccess) return rc;
    const int n = (int)((bytes + kChunk - 1) / kChunk);
    const auto issue = [&](int c) {
      const size_t o = kChunk * c;
      const hipError_t e =
          hipMemcpyAsync(buf_ + kChunk * (c % kSlots), (const char*)src + o,
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
        std::memcpy((char*)dst + o, buf_ + kChunk * (c % kSlots), std::min(kChunk, bytes - o));
        if (c + kSlots < n) err[t] = issue(c + kSlots);
      }
    };
    std::thread th[kThreads];
    int started = 1;
    try {
      for (; started < kThreads; ++started) th[started] = std::thread(work, started);
    } catch (const std::system_error&) {
      // the shares without a thread are this one's
    }
    work(0);
    for (int t = started; t < kThreads; ++t) work(t);
    for (int t = 1; t < started; ++t) th[t].join();
    for (hipError_t e : err)
      if (e != hipSuccess) rc = e;
    if (rc != hipSuccess) (void)hipStreamSynchronize(s);
    return rc;
  }

 private:
  static constexpr size_t kMin = 8u << 20, kChunk = 2u << 20;
  static constexpr int kSlots = 8, kThreads = 4;
  static_assert(kSlots % kThreads == 0, "a slot belongs to one thread");

  static bool known(const void* p) {
    hipPointerAttribute_t a;
    if (hipPointerGetAttributes(&a, p) == hipSuccess) return a.type != hipMemoryTypeUnregistered;
    (void)hipGetLastError();  // plain host memory
    return false;
  }

  bool make() {
    if (buf_) return true;
    for (hipEvent_t& e : ev_)
      if (!e && hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) {
        e = nullptr;
        (void)hipGetLastError();
        return false;
      }
    void* p = nullptr;
    if (hipHostMalloc(&p, kSlots * kChunk) != hipSuccess) {
      (void)hipGetLastError();
      return false;
    }
    buf_ = static_cast<char*>(p);
    return true;
  }

  char* buf_ = nullptr;
  hipEvent_t ev_[kSlots] = {};
};

}  // namespace phasecon
#endif
