// chromo_spec.hip -- the speculative persistent kernel k_mc_spec<W, NB, TW> for one
// NB = CHROMO_NB (binder types); built once per NB so that the instantiations compile
// in parallel.
#include <hip/hip_runtime.h>

#include "chromo_spec.hpp"

#ifndef CHROMO_NB
#error "compile with -DCHROMO_NB=1 .. 4"
#endif

#define CHROMO_CAT2(a, b) a##b
#define CHROMO_CAT(a, b) CHROMO_CAT2(a, b)

namespace {

// Persistent mc_sim with W wavefronts per replica (one workgroup per replica), for the
// replicas with NB binder types; the others are left to the launch of their own NB.
// One wavefront per SIMD: the full register file.  TW: the twisting chains' kernel,
// which passes over the others; the other kernel refuses a twisting chain with
// ERR_TWIST_WAVES (the caller asked for more wavefronts than such a chain may be given).
template <int W, int NB, bool TW>
__global__ void __launch_bounds__(WAVE * W) __attribute__((amdgpu_waves_per_eu(1)))
k_mc_spec(const chromo_replica *__restrict__ reps, int n_reps, int64_t steps)
{
    const int r = blockIdx.x;
    if (r >= n_reps) return;
    __shared__ chromo_replica Rs;
    __shared__ EvConst EC;
    load_record(&Rs, &reps[r]);
    __syncthreads();
    const chromo_replica *R = &Rs;
    if (R->B != NB) return;
    if (R->counters[CHROMO_CNT_ERROR] != 0) return;
    if ((R->twist != 0) != TW) {
        if (!TW) counters_error(R, ERR_TWIST_WAVES);
        return;
    }
    ev_const(&EC, R);
    __syncthreads();
    spec_run<NB, W, TW>(R, EC, steps);
}

template <int W, int NB, bool TW>
hipError_t launch(const chromo_replica *d_reps, int n_reps, int64_t steps, hipStream_t st)
{
    const size_t bytes = spec_layout<W>(NB + 1).total;
    // the attribute is set once per process: setting it costs far more than a launch
    static bool attr_set = false;
    if (!attr_set) {
        int dev = 0, lim = 0;
        hipError_t e = hipGetDevice(&dev);
        if (e == hipSuccess) e = hipDeviceGetAttribute(&lim, hipDeviceAttributeMaxSharedMemoryPerBlock, dev);
        if (e != hipSuccess) return e;
        if (bytes > (size_t)lim) return hipErrorInvalidValue;
        e = hipFuncSetAttribute((const void *)k_mc_spec<W, NB, TW>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
        if (e != hipSuccess) return e;
        attr_set = true;
    }
    hipLaunchKernelGGL((k_mc_spec<W, NB, TW>), dim3(n_reps), dim3(WAVE * W), bytes, st, d_reps, n_reps, steps);
    return hipGetLastError();
}

// Four wavefronts per replica where every replica can have a compute unit of its own
// (the block of three evaluators takes most of a unit's LDS), two otherwise.  128
// replicas of 1,500-9,000 beads, B = 3, the first 10 sweeps: 13.8 ms with one wavefront
// each, 5.4 with four (6.3 for later ones, at wider windows); one twisting chain, steady-state windows: 19.2 ms with
// one, 9.3 with four.
template <bool TW>
hipError_t launch_shape(const chromo_replica *d_reps, int n_reps, int64_t steps, hipStream_t st)
{
    static int units = 0;
    if (units == 0) {
        int dev = 0, n = 0;
        hipError_t e = hipGetDevice(&dev);
        if (e == hipSuccess) e = hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev);
        if (e != hipSuccess) return e;
        units = n;
    }
    return n_reps <= units ? launch<4, CHROMO_NB, TW>(d_reps, n_reps, steps, st)
                           : launch<2, CHROMO_NB, TW>(d_reps, n_reps, steps, st);
}

}  // namespace

namespace chromo {

hipError_t CHROMO_CAT(spec_launch_, CHROMO_NB)(const chromo_replica *d_reps, int n_reps, int64_t steps, bool twist,
                                               hipStream_t st)
{
    return twist ? launch_shape<true>(d_reps, n_reps, steps, st) : launch_shape<false>(d_reps, n_reps, steps, st);
}

}  // namespace chromo
