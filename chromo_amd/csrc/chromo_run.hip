// chromo_run.hip -- the one-wavefront persistent kernel k_mc_run_nb<NB> for one
// NB = CHROMO_NB (binder types); built once per NB so that the instantiations compile
// in parallel.
#include <hip/hip_runtime.h>

#include "chromo_mc.hpp"

#ifndef CHROMO_NB
#error "compile with -DCHROMO_NB=1 .. 4"
#endif

#define CHROMO_CAT2(a, b) a##b
#define CHROMO_CAT(a, b) CHROMO_CAT2(a, b)

namespace {

// Persistent mc_sim, one workgroup of one wavefront per replica, for the replicas with
// NB binder types and no twist; the others are left to the launch of their own kind.
// One instantiation per kernel, so that its registers are allocated for that one alone.
template <int NB>
__global__ void __launch_bounds__(64) k_mc_run_nb(const chromo_replica *__restrict__ reps, int n_reps,
                                                  int64_t steps)
{
    const int r = blockIdx.x;
    if (r >= n_reps) return;
    __shared__ chromo_replica Rs;
    __shared__ EvConst EC;
    load_record(&Rs, &reps[r]);
    wave_sync();
    const chromo_replica *R = &Rs;
    if (R->B != NB || R->twist) return;
    if (R->counters[CHROMO_CNT_ERROR] != 0) return;
    constexpr int Bp1 = NB + 1;
    ev_const(&EC, R);
    const EvLds S = ev_lds(lds_dyn, Bp1, 0);
    ev_clear(S);
    uint32_t *mt_lds = (uint32_t *)(lds_dyn + wide_lds_bytes(Bp1));
    const bool need_mt = any_binding(R);
    WaveRng rng;
    rng_load(R, rng, mt_lds, need_mt);
    Counters K;
    counters_load(R, K);
    const int nc = R->n_ctrl < MAX_CTRL ? R->n_ctrl : MAX_CTRL;
    __shared__ chromo_ctrl sctrl[MAX_CTRL];
    if (lane_id() == 0)
        for (int i = 0; i < nc; ++i) sctrl[i] = R->ctrl[i];
    __syncthreads();
    int err = 0;
    run_steps<NB>(R, EC, rng, K, sctrl, nc, steps, err, S);
    rng_store(R, rng, need_mt);
    if (lane_id() == 0)
        for (int i = 0; i < nc; ++i) R->ctrl[i] = sctrl[i];
    counters_store(R, K, err);
}

template <int NB>
hipError_t launch_nb(const chromo_replica *d_reps, int n_reps, int64_t steps, hipStream_t st)
{
    // the attribute is set once per process: setting it costs far more than a launch
    static bool attr_set = false;
    const size_t bytes = mc_lds_bytes(NB + 1);
    if (!attr_set) {
        hipError_t e = hipFuncSetAttribute((const void *)k_mc_run_nb<NB>,
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
        if (e != hipSuccess) return e;
        attr_set = true;
    }
    hipLaunchKernelGGL((k_mc_run_nb<NB>), dim3(n_reps), dim3(WAVE), bytes, st, d_reps, n_reps, steps);
    return hipGetLastError();
}

}  // namespace

namespace chromo {

hipError_t CHROMO_CAT(run_launch_, CHROMO_NB)(const chromo_replica *d_reps, int n_reps, int64_t steps, hipStream_t st)
{
    return launch_nb<CHROMO_NB>(d_reps, n_reps, steps, st);
}

}  // namespace chromo
