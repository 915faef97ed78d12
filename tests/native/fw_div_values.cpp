// Host build of the product's division by a reciprocal pair
// (finitewave_amd/csrc/fw_math.hpp): the quotients themselves.
#include <math.h>
#include <stdint.h>

#include "fw_math.hpp"

extern "C" void fw_div_values(const double* a, int64_t n, double b, double* out) {
  const fw::Recip y = fw::recip(b);
  for (int64_t i = 0; i < n; ++i) out[i] = fw::div_recip(a[i], y);
}
