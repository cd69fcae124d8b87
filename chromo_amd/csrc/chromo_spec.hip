// chromo_spec.hip -- the speculative persistent kernel k_mc_spec<W, NB> for one
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

// Persistent mc_sim with W wavefronts per replica (one workgroup per replica),
// for the replicas with NB binder types; the others are left to the launch of
// their own NB.  One wavefront per SIMD: the full register file.
template <int W, int NB>
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
    if (R->twist) {
        // the speculative evaluator has no twist terms: a twisting chain runs
        // with one wavefront (k_mc_run_nb)
        counters_error(R, ERR_TWIST_WAVES);
        return;
    }
    ev_const(&EC, R);
    __syncthreads();
    spec_run<NB, W>(R, EC, steps);
}

template <int W, int NB>
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
        e = hipFuncSetAttribute((const void *)k_mc_spec<W, NB>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
        if (e != hipSuccess) return e;
        attr_set = true;
    }
    hipLaunchKernelGGL((k_mc_spec<W, NB>), dim3(n_reps), dim3(WAVE * W), bytes, st, d_reps, n_reps, steps);
    return hipGetLastError();
}

}  // namespace

namespace chromo {

hipError_t CHROMO_CAT(spec_launch_, CHROMO_NB)(const chromo_replica *d_reps, int n_reps, int64_t steps,
                                               hipStream_t st)
{
    return launch<2, CHROMO_NB>(d_reps, n_reps, steps, st);
}

}  // namespace chromo
