// Spare buffers and allocations (csrc/memory.hip) over a stand-in for the HIP
// calls they make: two devices of 1000 bytes each.
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <map>
#include <mutex>
#include <string>
#include <thread>
#include <vector>

#include "memory.hpp"

namespace {
std::mutex mu;
struct Block {
  int device;
  size_t bytes;
};
std::map<void*, Block> blocks;
size_t used[2] = {0, 0};
thread_local int device = 0;
thread_local hipError_t last = hipSuccess;
std::vector<std::string> calls;  // synchronisations and frees, in order
uintptr_t next_address = 0x1000;

void check(bool ok, const char* what) {
  if (ok) return;
  std::printf("failed: %s\n", what);
  std::fflush(stdout);
  std::_Exit(1);
}
#define CHECK(x) check(x, #x)
}  // namespace

extern "C" {
hipError_t hipMalloc(void** p, size_t bytes) {
  std::lock_guard<std::mutex> lock(mu);
  if (used[device] + bytes > 1000) return last = hipErrorOutOfMemory;
  used[device] += bytes;
  *p = reinterpret_cast<void*>(next_address += 0x1000);
  blocks[*p] = {device, bytes};
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  std::lock_guard<std::mutex> lock(mu);
  if (!p) return hipSuccess;
  check(blocks.count(p) == 1, "freed once");
  used[blocks[p].device] -= blocks[p].bytes;
  blocks.erase(p);
  calls.push_back("free");
  return hipSuccess;
}
hipError_t hipMemGetInfo(size_t* free_b, size_t* total) {
  std::lock_guard<std::mutex> lock(mu);
  *free_b = 1000 - used[device];
  *total = 1000;
  return hipSuccess;
}
hipError_t hipGetDevice(int* d) {
  *d = device;
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s) {
  std::lock_guard<std::mutex> lock(mu);
  calls.push_back("sync " + std::to_string(reinterpret_cast<uintptr_t>(s)));
  return hipSuccess;
}
hipError_t hipGetLastError(void) {
  const hipError_t e = last;
  last = hipSuccess;
  return e;
}
}

using lbmx::device_alloc;
using lbmx::Spare;
using lbmx::SpareHold;

static hipStream_t stream(uintptr_t k) { return reinterpret_cast<hipStream_t>(k); }

int main() {
  void* p = nullptr;
  {  // taken only where a quarter stays free, once, and given back for an allocation
    Spare a, b, c;
    a.ask(760, stream(1));
    CHECK(!a.taken() && !a.hold());
    a.ask(10, stream(1));
    CHECK(!a.taken());
    b.ask(300, stream(2));
    c.ask(400, stream(3));
    CHECK(b.taken() && c.taken());
    calls.clear();
    CHECK(device_alloc(&p, 500) == hipSuccess);
    CHECK(!c.taken() && b.taken());  // as many as it needs
    CHECK(calls.size() == 2 && calls[0] == "sync 3" && calls[1] == "free");
    CHECK(hipGetLastError() == hipSuccess);
    void* q = nullptr;
    CHECK(device_alloc(&q, 600) == hipErrorOutOfMemory);  // all of them are not enough
    CHECK(!b.taken() && hipGetLastError() == hipSuccess);
    CHECK(hipFree(p) == hipSuccess);
    c.ask(100, stream(3));
    CHECK(!c.taken());  // (not again by itself)
    c.give_back();
    c.ask(100, stream(3));
    CHECK(c.taken());
    c.give_back();
    CHECK(!c.taken() && used[0] == 0);
  }
  {  // another device's stays
    Spare a;
    a.ask(700, stream(1));
    device = 1;
    CHECK(device_alloc(&p, 1000) == hipSuccess);
    void* q = nullptr;
    CHECK(device_alloc(&q, 1) == hipErrorOutOfMemory && a.taken());
    CHECK(hipFree(p) == hipSuccess);
    device = 0;
  }
  {  // what this thread holds stays, and the allocation fails at once
    Spare a;
    a.ask(700, stream(1));
    const SpareHold h(a);
    CHECK(h.p && device_alloc(&p, 500) == hipErrorOutOfMemory && a.taken());
  }
  CHECK(used[0] == 0);  // (a Spare gives back at its end)
  {  // what another thread holds is waited for, call after call of its owner
    Spare a;
    a.ask(700, stream(1));
    std::vector<std::thread> th;
    void* got[2] = {nullptr, nullptr};
    bool done = false;
    {
      const SpareHold h(a);
      for (int i = 0; i < 2; ++i)
        th.emplace_back([&, i] { CHECK(device_alloc(&got[i], 450) == hipSuccess); });
      std::this_thread::sleep_for(std::chrono::milliseconds(100));
      CHECK(a.taken() && h.p && blocks.count(h.p) == 1);
    }
    for (int k = 0; k < 1000000 && !done; ++k) {
      const SpareHold h(a);
      done = !h.p;
    }
    CHECK(done);
    for (auto& t : th) t.join();
    CHECK(got[0] && got[1] && !a.taken() && used[0] == 900);
  }
  std::printf("ok\n");
  return 0;
}
