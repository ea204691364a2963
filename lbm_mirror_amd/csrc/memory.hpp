// Device memory: allocations that give back spare buffers before they fail.
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>

namespace lbmx {

// hipMalloc on the current device.  Where it is out of memory, the spare buffers
// there are freed one at a time, each as soon as no call uses it, until the
// allocation succeeds or none is left.  A failure leaves no error behind for
// the next launch to report.  Not for a thread that holds a spare buffer itself
// (it would free only those nobody uses).
hipError_t device_alloc(void** p, size_t bytes);
template <class T>
hipError_t device_alloc(T** p, size_t bytes) {
  return device_alloc(reinterpret_cast<void**>(p), bytes);
}

// A buffer with which its owner is faster and without which it still works.
class Spare {
 public:
  Spare() = default;
  ~Spare() { give_back(); }
  Spare(const Spare&) = delete;
  Spare& operator=(const Spare&) = delete;

  // Takes `bytes` on the current device, unless that would leave less than a
  // quarter of its memory free.  Asked once, and again only after give_back().
  // Work that uses the buffer is queued on `s` alone.
  void ask(size_t bytes, hipStream_t s);
  bool taken() const;  // (another thread's allocation may free it next)
  // The buffer for the work of one call, or null where there is none.  Until
  // let_go() by the same thread no allocation frees it.  A call that uses or
  // captures its stream holds it, needed or not.
  void* hold();
  void let_go();
  // Frees it, behind the work queued on its stream.
  void give_back();

 private:
  friend hipError_t device_alloc(void** p, size_t bytes);
  void release();
  static bool free_one(int device, uint64_t seen);

  void* p_ = nullptr;
  int device_ = 0;
  hipStream_t s_ = nullptr;
  bool asked_ = false;
  int held_ = 0;
  Spare* next_ = nullptr;  // the list of those that have a buffer
};

// hold() until the end of a scope
class SpareHold {
 public:
  explicit SpareHold(Spare& s) : p(s.hold()), s_(s) {}
  ~SpareHold() {
    if (p) s_.let_go();
  }
  SpareHold(const SpareHold&) = delete;
  SpareHold& operator=(const SpareHold&) = delete;

  void* const p;

 private:
  Spare& s_;
};

}  // namespace lbmx
