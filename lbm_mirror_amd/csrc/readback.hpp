// Device arrays into caller memory, through pinned staging and several threads.
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>
#include <functional>

namespace lbmx {

// One array to read: `bytes` from device address `src`.  `use(data, offset,
// n)` takes the bytes [offset, offset + n) at host address `data`; offset and n
// are multiples of `unit` (the end aside).  It is called from several threads
// at once for different ranges, and must not throw.
struct ReadBack {
  const void* src;
  size_t bytes, unit;
  std::function<void(const char* data, size_t offset, size_t n)> use;
};

// Reads the arrays behind what is queued on `s` and returns when every byte has
// been used.
hipError_t read_back(int device, hipStream_t s, const ReadBack* what, int count);

// A context or network that may read back lives: the staging kept between calls
// is given back with the last one.
void read_back_user(int change);

}  // namespace lbmx
