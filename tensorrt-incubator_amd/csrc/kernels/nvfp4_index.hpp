// Where blocks along the second-to-last axis keep what a vector of the tensor needs; plain arithmetic, for the device and the host.
#pragma once
#include <stdint.h>

namespace nvfp4_cluster {

// All vectors of a launch have 32-bit numbers (64 GiB of output do not).
constexpr bool numbers_fit(int64_t nvec) { return uint64_t(nvec) >> 32 == 0; }

// The place, among the scales [d0 / 16, d1], of the first scale of vector v (G elements of one row) of a [d0, d1] tensor.  NARROW: where
// the numbers fit they are divided in 32 bits (a 64-bit division is a hundred instructions).
template <bool NARROW, int G>
constexpr int64_t scale_of_vector(int64_t v, int64_t d1) {
  const int64_t groups = d1 / G;
  const int64_t row = NARROW ? int64_t(uint32_t(v) / uint32_t(groups)) : int64_t(uint64_t(v) / uint64_t(groups));
  return row / 16 * d1 + (v - row * groups) * G;
}

}  // namespace nvfp4_cluster
