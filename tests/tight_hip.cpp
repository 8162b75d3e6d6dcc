// Preloaded before the HIP runtime: device allocations are counted and fail beyond a budget,
// so that a test reaches the library's out-of-memory paths without filling the device.
#define __HIP_PLATFORM_AMD__
#include <dlfcn.h>
#include <hip/hip_runtime_api.h>
#include <map>
#include <mutex>

namespace {
std::mutex mu;
std::map<void*, size_t> blocks;
size_t used = 0, peak = 0, budget = ~size_t(0);
int refused = 0;
}  // namespace

extern "C" {
void tight_hip_set_budget(size_t bytes) { budget = bytes; }
void tight_hip_reset_peak() { peak = used; }
size_t tight_hip_used() { return used; }
size_t tight_hip_peak() { return peak; }
int tight_hip_refused() { return refused; }

hipError_t hipMalloc(void** p, size_t n) {
  static auto real = reinterpret_cast<hipError_t (*)(void**, size_t)>(dlsym(RTLD_NEXT, "hipMalloc"));
  {
    std::lock_guard<std::mutex> lk(mu);
    if (used + n > budget) {
      ++refused;
      *p = nullptr;
      return hipErrorOutOfMemory;
    }
  }
  const hipError_t e = real(p, n);
  if (e == hipSuccess) {
    std::lock_guard<std::mutex> lk(mu);
    blocks[*p] = n;
    used += n;
    if (used > peak) peak = used;
  }
  return e;
}
hipError_t hipFree(void* p) {
  static auto real = reinterpret_cast<hipError_t (*)(void*)>(dlsym(RTLD_NEXT, "hipFree"));
  {
    std::lock_guard<std::mutex> lk(mu);
    auto it = blocks.find(p);
    if (it != blocks.end()) {
      used -= it->second;
      blocks.erase(it);
    }
  }
  return real(p);
}
}
