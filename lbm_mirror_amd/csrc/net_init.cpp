// In a file for the host compiler: std::normal_distribution takes two logarithms
// of constants per value in long double, which g++ folds and clang calls.  A network
// of 916,451 parameters is made in 35 or 63 ms with clang's code, by where it
// happens to lie in the library, and in 13 ms with this; the values are the same bits.
#include "net_init.hpp"

#include <cmath>
#include <random>

namespace lbmnet {

void he_normal(uint64_t seed, const HeLayer* layers, int n) {
  std::mt19937_64 rng(seed);
  for (const HeLayer* l = layers; l != layers + n; ++l) {
    std::normal_distribution<double> nd(0.0, std::sqrt(2.0 / (9.0 * l->cin)));
    for (size_t i = 0; i < l->count; ++i) l->w[i] = float(nd(rng));
  }
}

}  // namespace lbmnet
