#include "memory.hpp"

#include <atomic>
#include <condition_variable>
#include <cstdint>
#include <mutex>

namespace lbmx {
namespace {

std::mutex g_mu;               // every Spare's state
std::condition_variable g_cv;  // one was taken, let go or given back; none waits any more
Spare* g_first = nullptr;
std::atomic<uint64_t> g_freed{0};  // spares freed so far
constexpr int kDevices = 64;
int g_waiting[kDevices] = {};    // per device, allocations that wait for a held one
thread_local int t_holding = 0;  // spares this thread holds

}  // namespace

void Spare::ask(size_t bytes, hipStream_t s) {
  if (asked_) return;
  asked_ = true;
  size_t free_b = 0, total = 0;
  void* p = nullptr;
  if (hipMemGetInfo(&free_b, &total) != hipSuccess || free_b < bytes || free_b - bytes < total / 4 ||
      hipGetDevice(&device_) != hipSuccess || hipMalloc(&p, bytes) != hipSuccess) {
    (void)hipGetLastError();
    return;
  }
  {
    std::lock_guard<std::mutex> lock(g_mu);
    p_ = p;
    s_ = s;
    next_ = g_first;
    g_first = this;
  }
  g_cv.notify_all();
}

bool Spare::taken() const {
  std::lock_guard<std::mutex> lock(g_mu);
  return p_ != nullptr;
}

void* Spare::hold() {
  std::unique_lock<std::mutex> lock(g_mu);
  // (an allocation that waits has this one freed first if it is not held)
  g_cv.wait(lock, [&] { return !p_ || g_waiting[device_ % kDevices] == 0; });
  if (!p_) return nullptr;
  ++held_;
  ++t_holding;
  return p_;
}

void Spare::let_go() {
  {
    std::lock_guard<std::mutex> lock(g_mu);
    if (held_ == 0) return;
    --held_;
    --t_holding;
  }
  g_cv.notify_all();
}

// (under g_mu)
void Spare::release() {
  for (Spare** q = &g_first; *q; q = &(*q)->next_)
    if (*q == this) {
      *q = next_;
      break;
    }
  (void)hipStreamSynchronize(s_);
  (void)hipFree(p_);
  ++g_freed;
  p_ = nullptr;
  next_ = nullptr;
}

void Spare::give_back() {
  {
    std::lock_guard<std::mutex> lock(g_mu);
    asked_ = false;
    if (p_) release();
  }
  g_cv.notify_all();
}

// Frees one spare of the device, or waits until one was let go; false if there is
// none to free or wait for and none has been freed since `seen`.
bool Spare::free_one(int device, uint64_t seen) {
  std::unique_lock<std::mutex> lock(g_mu);
  if (g_freed != seen) return true;
  bool held = false;
  for (Spare* q = g_first; q; q = q->next_) {
    if (q->device_ != device) continue;
    if (q->held_ == 0) {
      q->release();
      return true;
    }
    held = true;
  }
  if (!held || t_holding) return false;
  int& waiting = g_waiting[device % kDevices];
  ++waiting;
  g_cv.wait(lock);
  for (Spare* q = g_first; q; q = q->next_)
    if (q->device_ == device && q->held_ == 0) {
      q->release();
      break;
    }
  if (--waiting == 0) g_cv.notify_all();
  return true;
}

hipError_t device_alloc(void** p, size_t bytes) {
  for (;;) {
    const uint64_t seen = g_freed;
    const hipError_t e = hipMalloc(p, bytes);
    if (e == hipSuccess) return e;
    (void)hipGetLastError();
    int device = 0;
    if (e != hipErrorOutOfMemory || hipGetDevice(&device) != hipSuccess || !Spare::free_one(device, seen)) return e;
  }
}

}  // namespace lbmx
