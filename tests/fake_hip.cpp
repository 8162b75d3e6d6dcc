// A stand-in for the HIP runtime, preloaded before the library so that its host code runs
// without a GPU: device memory is host memory under a budget, copies are done at once,
// kernels do nothing.  Tests of the library's memory handling use it.
#define __HIP_PLATFORM_AMD__
#include <hip/hip_runtime_api.h>
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <new>

namespace {
std::mutex mu;
struct Block {
  size_t bytes;
  int device;
};
std::map<void*, Block> blocks;
size_t used[2] = {0, 0}, budget[2] = {~size_t(0), ~size_t(0)};
int double_frees = 0;
thread_local int current = 0;
thread_local hipError_t last = hipSuccess;
hipError_t done(hipError_t e) {
  if (e != hipSuccess) last = e;
  return e;
}
char symbol[1 << 20];
thread_local int new_fails_in = -1;
}  // namespace

// host memory that runs out: the n-th operator new from now on (and no other) throws
void* operator new(size_t n) {
  if (new_fails_in >= 0 && new_fails_in-- == 0) throw std::bad_alloc();
  void* p = std::malloc(n ? n : 1);
  if (!p) throw std::bad_alloc();
  return p;
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }

extern "C" {
// test controls
size_t fake_hip_used(int device) { return used[device]; }
void fake_hip_set_budget(int device, size_t bytes) { budget[device] = bytes; }
void fake_hip_fail_new(int n) { new_fails_in = n; }
int fake_hip_bad_frees() { return double_frees; }

hipError_t hipMalloc(void** p, size_t n) {
  std::lock_guard<std::mutex> lk(mu);
  *p = nullptr;
  if (used[current] + n > budget[current]) return done(hipErrorOutOfMemory);
  *p = std::calloc(n ? n : 1, 1);
  if (!*p) return done(hipErrorOutOfMemory);
  const int keep = new_fails_in;
  new_fails_in = -1;
  blocks[*p] = Block{n, current};
  new_fails_in = keep;
  used[current] += n;
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  if (!p) return hipSuccess;
  std::lock_guard<std::mutex> lk(mu);
  auto it = blocks.find(p);
  if (it == blocks.end()) {
    ++double_frees;
    return done(hipErrorInvalidValue);
  }
  used[it->second.device] -= it->second.bytes;
  blocks.erase(it);
  std::free(p);
  return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) {
  std::memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
  std::memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) {
  std::memset(d, v, n);
  return hipSuccess;
}
hipError_t hipMemsetD32Async(hipDeviceptr_t d, int v, size_t n, hipStream_t) {
  for (size_t i = 0; i < n; ++i) static_cast<int*>(d)[i] = v;
  return hipSuccess;
}
hipError_t hipGetDeviceCount(int* n) { return *n = 2, hipSuccess; }
hipError_t hipGetDevice(int* d) { return *d = current, hipSuccess; }
hipError_t hipSetDevice(int d) {
  if (d < 0 || d > 1) return done(hipErrorInvalidDevice);
  return current = d, hipSuccess;
}
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t a, int) {
  *v = a == hipDeviceAttributeMultiprocessorCount ? 256 : 64;
  return hipSuccess;
}
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
  std::memset(p, 0, sizeof(*p));
  p->multiProcessorCount = 256;
  p->warpSize = 64;
  p->maxThreadsPerBlock = 1024;
  std::strcpy(p->gcnArchName, "gfx950");
  return hipSuccess;
}
int hipGetStreamDeviceId(hipStream_t) { return current; }
hipError_t hipStreamCreate(hipStream_t* s) { return *s = reinterpret_cast<hipStream_t>(symbol), hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { return hipStreamCreate(s); }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { return *e = reinterpret_cast<hipEvent_t>(symbol), hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { return *ms = 0.f, hipSuccess; }
const char* hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "error"; }
hipError_t hipGetLastError() {
  const hipError_t e = last;
  last = hipSuccess;
  return e;
}
hipError_t hipGetSymbolAddress(void** p, const void*) { return *p = symbol, hipSuccess; }
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void*) {
  std::memset(a, 0, sizeof(*a));
  a->type = hipMemoryTypeDevice;
  return hipSuccess;
}
// a launch is refused, as by the runtime, when it is empty, when a block has more than
// 1024 threads or when a grid has 2^32 threads or more in one dimension
hipError_t hipLaunchKernel(const void*, dim3 g, dim3 b, void**, size_t, hipStream_t) {
  const uint64_t n[3] = {uint64_t(g.x) * b.x, uint64_t(g.y) * b.y, uint64_t(g.z) * b.z};
  if (uint64_t(b.x) * b.y * b.z > 1024) return done(hipErrorInvalidConfiguration);
  for (uint64_t v : n)
    if (v == 0 || v >= (uint64_t(1) << 32)) return done(hipErrorInvalidConfiguration);
  return hipSuccess;
}
static thread_local dim3 pushed_grid, pushed_block;
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t, hipStream_t) {
  pushed_grid = g;
  pushed_block = b;
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* s, hipStream_t* st) {
  *g = pushed_grid;
  *b = pushed_block;
  *s = 0;
  *st = nullptr;
  return hipSuccess;
}
void** __hipRegisterFatBinary(const void*) {
  static void* handle = nullptr;
  return &handle;
}
void __hipRegisterFunction(void**, const void*, char*, const char*, unsigned, void*, void*, dim3*, dim3*, int*) {}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
void __hipUnregisterFatBinary(void**) {}
}
