// chromo_index.hpp -- index arithmetic that has to hold up to the largest chain taken
// (2^31 - 1 beads).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace chromo {

// Place of component j of bead b in an N x 3 array: past 2^31 from 715,827,883 beads on.
__host__ __device__ __forceinline__ int64_t row3(int32_t b, int j) { return 3 * (int64_t)b + j; }

}  // namespace chromo
