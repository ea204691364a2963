// The network's initial weights (host).
#pragma once
#include <cstddef>
#include <cstdint>

namespace lbmnet {

// w[0 .. count) := normal values of variance 2 / (9 cin), for each layer in turn
// from one generator.
struct HeLayer {
  float* w;
  size_t count;
  int cin;
};
void he_normal(uint64_t seed, const HeLayer* layers, int n);

}  // namespace lbmnet
