// A GPU of little memory: hipMalloc, hipFree and hipMemGetInfo of whatever is
// loaded after this library, within a budget of bytes; and a host whose pinned
// memory is used up (hipHostMalloc).
#include <dlfcn.h>
#include <hip/hip_runtime_api.h>

#include <map>
#include <mutex>

namespace {
std::mutex mu;
std::map<void*, size_t> blocks;
size_t budget = 0, used = 0;
bool pinned = true;
template <class F>
F real(const char* name) {
  return reinterpret_cast<F>(dlsym(RTLD_NEXT, name));
}
}  // namespace

extern "C" {
void budget_set(size_t bytes) { budget = bytes; }
size_t budget_used() { return used; }
void pinned_set(int left) { pinned = left != 0; }

hipError_t hipMalloc(void** p, size_t bytes) {
  static const auto f = real<hipError_t (*)(void**, size_t)>("hipMalloc");
  std::lock_guard<std::mutex> lock(mu);
  if (used + bytes > budget) return hipErrorOutOfMemory;
  const hipError_t e = f(p, bytes);
  if (e == hipSuccess && *p) {
    blocks[*p] = bytes;
    used += bytes;
  }
  return e;
}
hipError_t hipFree(void* p) {
  static const auto f = real<hipError_t (*)(void*)>("hipFree");
  std::lock_guard<std::mutex> lock(mu);
  const auto it = blocks.find(p);
  if (it != blocks.end()) {
    used -= it->second;
    blocks.erase(it);
  }
  return f(p);
}
hipError_t hipMemGetInfo(size_t* free_b, size_t* total) {
  std::lock_guard<std::mutex> lock(mu);
  *free_b = budget - used;
  *total = budget;
  return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t bytes, unsigned flags) {
  static const auto f = real<hipError_t (*)(void**, size_t, unsigned)>("hipHostMalloc");
  return pinned ? f(p, bytes, flags) : hipErrorOutOfMemory;
}
}
