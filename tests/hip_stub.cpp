// Host stand-in for the HIP runtime: device memory is reserved address space
// (zero, private to the process), kernel launches are recorded and not run.
// Linked with the host side of a .hip file (hip_stub.py) it shows on the CPU
// which allocations, copies and launches an entry point makes.
#include <hip/hip_runtime.h>
#include <sys/mman.h>

#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>

namespace {
std::mutex g_m;
std::map<void*, size_t> g_dev, g_pin;         // live allocations
std::map<const char*, size_t> g_dead;         // freed ones: never handed out again
long long g_mallocs, g_launches, g_pins, g_events;
long long g_live_events, g_fail_at = -1;  // hipMalloc that fails from now on (0: the next)
std::string g_log;                        // "name x y z threads\n" per launch
thread_local dim3 t_grid, t_block;
thread_local size_t t_lds;
thread_local hipStream_t t_stream;
int g_pin_fails;

// host stub -> device name; filled by constructors that may run before this file's
std::map<const void*, std::string>& kernels() {
  static std::map<const void*, std::string> k;
  return k;
}

void* reserve(size_t n) {
  void* p = mmap(nullptr, n ? n : 1, PROT_READ | PROT_WRITE,
                 MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
  return p == MAP_FAILED ? nullptr : p;
}

void retire(void* p, size_t n) {
  madvise(p, n ? n : 1, MADV_DONTNEED);
  g_dead[static_cast<const char*>(p)] = n ? n : 1;
}

// whether a copy may use p: not null, not freed
bool usable(const void* p) {
  std::lock_guard<std::mutex> l(g_m);
  auto i = g_dead.upper_bound(static_cast<const char*>(p));
  if (i == g_dead.begin()) return p != nullptr;
  --i;
  return p && static_cast<const char*>(p) >= i->first + i->second;
}
}  // namespace

extern "C" {

// ------------------------------------------------ what the tests read and set
void stub_fail_malloc(long long after) { g_fail_at = after < 0 ? -1 : g_mallocs + after; }
void stub_fail_pin(int on) { g_pin_fails = on; }
long long stub_launches() { return g_launches; }
long long stub_mallocs() { return g_mallocs; }
long long stub_pins() { return g_pins; }
long long stub_live() { return (long long)g_dev.size(); }
long long stub_live_pins() { return (long long)g_pin.size(); }
long long stub_live_events() { return g_live_events; }
const char* stub_log() { return g_log.c_str(); }
void stub_clear_log() { g_log.clear(); }

// ------------------------------------------------------------------- runtime
hipError_t hipMalloc(void** p, size_t n) {
  std::lock_guard<std::mutex> l(g_m);
  *p = nullptr;
  if (g_fail_at >= 0 && g_mallocs >= g_fail_at) return hipErrorOutOfMemory;
  ++g_mallocs;
  if (!(*p = reserve(n))) return hipErrorOutOfMemory;
  g_dev[*p] = n;
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  std::lock_guard<std::mutex> l(g_m);
  const auto i = g_dev.find(p);
  if (i == g_dev.end()) return p ? hipErrorInvalidValue : hipSuccess;
  retire(p, i->second);
  g_dev.erase(i);
  return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  std::lock_guard<std::mutex> l(g_m);
  *p = nullptr;
  if (g_pin_fails || !(*p = reserve(n))) return hipErrorOutOfMemory;
  ++g_pins;
  g_pin[*p] = n;
  return hipSuccess;
}
hipError_t hipHostFree(void* p) {
  std::lock_guard<std::mutex> l(g_m);
  const auto i = g_pin.find(p);
  if (i == g_pin.end()) return hipErrorInvalidValue;
  retire(p, i->second);
  g_pin.erase(i);
  return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) {
  if (!usable(d) || !usable(s)) return hipErrorInvalidValue;
  memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind k, hipStream_t) {
  return hipMemcpy(d, s, n, k);
}
hipError_t hipMemset(void*, int, size_t) { return hipSuccess; }
hipError_t hipMemsetAsync(void*, int, size_t, hipStream_t) { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "stub error"; }
hipError_t hipStreamCreate(hipStream_t* s) {
  *s = reinterpret_cast<hipStream_t>(8);
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) {
  std::lock_guard<std::mutex> l(g_m);
  *e = reinterpret_cast<hipEvent_t>(16 * ++g_events);
  ++g_live_events;
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t) {
  std::lock_guard<std::mutex> l(g_m);
  --g_live_events;
  return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) {
  *ms = 0.f;
  return hipSuccess;
}
hipError_t hipGetDevice(int* d) {
  *d = 0;
  return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipPointerGetAttributes(hipPointerAttribute_t*, const void*) {
  return hipErrorInvalidValue;  // plain host memory
}
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) {
  *v = 160 * 1024;  // the only one asked for: LDS per workgroup
  return hipSuccess;
}
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int threads, size_t) {
  *n = 2048 / threads;
  return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void* s) {
  *p = const_cast<void*>(s);
  return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipErrorNotSupported; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t*) { return hipErrorNotSupported; }
hipError_t hipGraphInstantiate(hipGraphExec_t*, hipGraph_t, hipGraphNode_t*, char*, size_t) {
  return hipErrorNotSupported;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipErrorNotSupported; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }

// ------------------------------------------------------------ compiler's side
void** __hipRegisterFatBinary(const void*) {
  static void* h;
  return &h;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* f, char*, const char* name, unsigned, uint3*,
                           uint3*, dim3*, dim3*, int*) {
  kernels()[f] = name;
}
void __hipRegisterVar(void**, void*, char*, const char*, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, hipStream_t s) {
  t_grid = g;
  t_block = b;
  t_lds = lds;
  t_stream = s;
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* lds, hipStream_t* s) {
  *g = t_grid;
  *b = t_block;
  *lds = t_lds;
  *s = t_stream;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3 g, dim3 b, void**, size_t, hipStream_t) {
  std::lock_guard<std::mutex> l(g_m);
  ++g_launches;
  g_log += kernels()[f] + " " + std::to_string(g.x) + " " + std::to_string(g.y) + " " +
           std::to_string(g.z) + " " + std::to_string(b.x * b.y * b.z) + "\n";
  return hipSuccess;
}
}  // extern "C"
