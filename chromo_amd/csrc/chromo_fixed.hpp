// chromo_fixed.hpp -- corner weights as integers, for density sums that do not depend on
// the order of the beads (chromo_energy.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <math.h>
#include <stdint.h>

#include "chromo_hip.h"

namespace chromo {

// A weight w in [0, 1] as (hi 2^30 + lo) 2^-60, the multiple of 2^-60 nearest to w.  hi is
// the integer nearest to w 2^30, lo the one nearest to the rest times 2^30; the rest lies
// in [-1/2, 1/2], ends included, so |lo| <= 2^29.  Adding 1.5 2^52 leaves an integer in
// the low word.
// Words of 30 bits: times a binder state (up to 3) hi still fits 32 unsigned bits and lo
// 32 signed ones, and the sums over 2^31 beads of one voxel fit 64 bits.
struct Fixed60 {
    uint32_t hi;
    int32_t lo;
};
static_assert(CHROMO_MAX_SITES <= 3, "a word times a binder state fits 32 bits");
constexpr double FIXED60_SCALE = 0x1p30;

// w30 = w FIXED60_SCALE
__host__ __device__ __forceinline__ Fixed60 fixed60(double w30)
{
    const double mh = w30 + 0x1.8p52;
    const double ml = fma(w30 - (mh - 0x1.8p52), 0x1p30, 0x1.8p52);
    return Fixed60{(uint32_t)__builtin_bit_cast(uint64_t, mh), (int32_t)__builtin_bit_cast(uint64_t, ml)};
}

// The double nearest to (hi 2^30 + lo) 2^-60, sums of words; exact before the one rounding
// for sums below 2^53 (more than 2^21 beads in one voxel, whose state is 3, round hi first).
__host__ __device__ __forceinline__ double from_fixed60(uint64_t hi, uint64_t lo)
{
    return fma((double)hi, 0x1p30, (double)(int64_t)lo) * 0x1p-60;
}

}  // namespace chromo
