// Host build of the product's division by a literal's and by a parameter's
// reciprocal pair (finitewave_amd/csrc/fw_math.hpp): the quotients.
#include <math.h>
#include <stdint.h>

#include "fw_math.hpp"

extern "C" void fw_div_pair(const double* a, int64_t n, double b, int32_t literal, double* out) {
  const fw::Recip y = literal ? fw::literal_recip(b) : fw::recip(b);
  for (int64_t i = 0; i < n; ++i) out[i] = fw::div_recip(a[i], y);
}
