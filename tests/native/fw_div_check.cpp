// Host build of the product's division by a reciprocal pair
// (finitewave_amd/csrc/fw_math.hpp) for the CPU tests.
#include <math.h>
#include <stdint.h>

#include "fw_math.hpp"

// counts the quotients a[i] / b that differ from the machine's division
extern "C" int64_t fw_div_check(const double* a, int64_t n, double b) {
  const fw::Recip y = fw::recip(b);
  int64_t bad = 0;
  for (int64_t i = 0; i < n; ++i) bad += fw::div_recip(a[i], y) != a[i] / b;
  return bad;
}
