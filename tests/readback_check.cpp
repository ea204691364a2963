// Read-back (csrc/readback.hip) over a stand-in for the HIP calls it makes:
// every byte exactly once and in place, whole units, with and without pinned
// memory or heap, a failing copy, and nothing kept once the last user has gone.
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <new>
#include <set>
#include <vector>

#include "readback.hpp"

namespace {
std::mutex mu;
std::set<void*> pinned;
std::atomic<int> events{0}, copies{0};
bool no_pinned = false;
bool no_heap = false;
int fail_copy = -1;
hipError_t last = hipSuccess;

void check(bool ok, const char* what) {
  if (ok) return;
  std::printf("failed: %s\n", what);
  std::fflush(stdout);
  std::_Exit(1);
}
#define CHECK(x) check(x, #x)
}  // namespace

void* operator new(size_t n) {
  void* p = no_heap ? nullptr : std::malloc(n);
  if (!p) throw std::bad_alloc();
  return p;
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }

extern "C" {
hipError_t hipHostMalloc(void** p, size_t bytes, unsigned) {
  if (no_pinned) return last = hipErrorOutOfMemory;
  std::lock_guard<std::mutex> lock(mu);
  const bool was = no_heap;
  no_heap = false;
  *p = std::malloc(bytes);
  pinned.insert(*p);
  no_heap = was;
  return hipSuccess;
}
hipError_t hipHostFree(void* p) {
  std::lock_guard<std::mutex> lock(mu);
  check(pinned.erase(p) == 1, "pinned memory freed once");
  std::free(p);
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  *e = reinterpret_cast<hipEvent_t>(uintptr_t(++events));
  return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t) {
  --events;
  return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipMemcpyAsync(void* to, const void* from, size_t n, hipMemcpyKind, hipStream_t) {
  if (copies++ == fail_copy) return last = hipErrorUnknown;
  std::memcpy(to, from, n);
  return hipSuccess;
}
hipError_t hipGetLastError(void) {
  const hipError_t e = last;
  last = hipSuccess;
  return e;
}
}

using lbmx::ReadBack;

// arrays of these sizes, each in units of 12 bytes
static hipError_t run(const std::vector<size_t>& units, bool whole) {
  std::vector<std::vector<unsigned char>> src, dst;
  std::vector<std::vector<std::atomic<unsigned char>>> seen;
  for (size_t k = 0; k < units.size(); ++k) {
    src.emplace_back(12 * units[k]);
    dst.emplace_back(12 * units[k], 0);
    seen.emplace_back(units[k]);
    for (size_t i = 0; i < src[k].size(); ++i) src[k][i] = (unsigned char)(i * 2654435761u >> 13) ^ k;
  }
  std::vector<ReadBack> r;
  for (size_t k = 0; k < units.size(); ++k)
    r.push_back({src[k].data(), src[k].size(), 12, [&, k](const char* data, size_t at, size_t n) {
                   check(at % 12 == 0 && n % 12 == 0, "whole units");
                   std::memcpy(dst[k].data() + at, data, n);
                   for (size_t i = at / 12; i < (at + n) / 12; ++i) ++seen[k][i];
                 }});
  const hipError_t e = lbmx::read_back(0, nullptr, r.data(), int(r.size()));
  if (whole) {
    CHECK(e == hipSuccess && src == dst);
    for (auto& s : seen)
      for (auto& c : s) CHECK(c == 1);
  }
  return e;
}

int main() {
  lbmx::read_back_user(1);
  {  // where the heap is used up: small reads need none, larger ones say so
    std::vector<unsigned char> from(12 << 20, 3), to(12 << 20);
    unsigned char* out = to.data();
    ReadBack r{from.data(), 1000, 1, [out](const char* data, size_t at, size_t n) { std::memcpy(out + at, data, n); }};
    no_heap = true;
    const hipError_t small = lbmx::read_back(0, nullptr, &r, 1);
    r.bytes = from.size();
    const hipError_t large = lbmx::read_back(0, nullptr, &r, 1);
    no_heap = false;
    CHECK(small == hipSuccess && to[999] == 3 && large == hipErrorOutOfMemory);
  }
  for (bool none : {false, true}) {
    no_pinned = none;
    for (size_t n : {size_t(1), size_t(1000), size_t(699050), size_t(699051), size_t(2000003)}) {
      (void)run({n}, true);
      (void)run({n, 3, 2 * n + 1}, true);
    }
    (void)run({}, true);
    for (int k : {0, 2, 9}) {
      copies = 0;
      fail_copy = k;
      CHECK(run({4000000}, false) == hipErrorUnknown);
      fail_copy = -1;
      (void)hipGetLastError();
    }
    CHECK(hipGetLastError() == hipSuccess);
  }
  lbmx::read_back_user(-1);
  CHECK(pinned.empty() && events == 0);
  std::printf("ok\n");
  return 0;
}
