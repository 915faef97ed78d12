// Host build of the product's x^1.5 (finitewave_amd/csrc/fw_math.hpp) for the
// CPU tests.
#include <math.h>
#include <stdint.h>

#include "fw_math.hpp"

extern "C" void fw_pow15(const double* x, int64_t n, double* out) {
  for (int64_t i = 0; i < n; ++i) out[i] = fw::pow15(x[i]);
}
