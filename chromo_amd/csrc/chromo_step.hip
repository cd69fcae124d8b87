// chromo_step.hip -- the kernels that take a replica of any kind: one proposal per
// launch (mc_step and the plain path) and the persistent kernel behind chromo_mc_run.
#include <hip/hip_runtime.h>

#include "chromo_spec.hpp"

using namespace chromo;

namespace {

// Persistent mc_sim: one workgroup (one wave) per replica.
__global__ void __launch_bounds__(64) k_mc_run(const chromo_replica *__restrict__ reps, int n_reps, int64_t steps,
                                               int max_bp1)
{
    const int r = blockIdx.x;
    if (r >= n_reps) return;
    __shared__ chromo_replica Rs;
    __shared__ EvConst EC;
    load_record(&Rs, &reps[r]);
    wave_sync();
    const chromo_replica *R = &Rs;
    if (R->counters[CHROMO_CNT_ERROR] != 0) return;
    if (R->B < 1 || R->B + 1 > max_bp1) {
        counters_error(R, ERR_NBINDERS);
        return;
    }
    const int Bp1 = R->B + 1;
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
    if (R->twist) {
        switch (R->B) {
        case 1: run_steps<1, true>(R, EC, rng, K, sctrl, nc, steps, err, S); break;
        case 2: run_steps<2, true>(R, EC, rng, K, sctrl, nc, steps, err, S); break;
        case 3: run_steps<3, true>(R, EC, rng, K, sctrl, nc, steps, err, S); break;
        case 4: run_steps<4, true>(R, EC, rng, K, sctrl, nc, steps, err, S); break;
        default: err = ERR_NBINDERS; break;
        }
    } else {
        switch (R->B) {
        case 1: run_steps<1>(R, EC, rng, K, sctrl, nc, steps, err, S); break;
        case 2: run_steps<2>(R, EC, rng, K, sctrl, nc, steps, err, S); break;
        case 3: run_steps<3>(R, EC, rng, K, sctrl, nc, steps, err, S); break;
        case 4: run_steps<4>(R, EC, rng, K, sctrl, nc, steps, err, S); break;
        default: err = ERR_NBINDERS; break;
        }
    }
    rng_store(R, rng, need_mt);
    if (lane_id() == 0)
        for (int i = 0; i < nc; ++i) R->ctrl[i] = sctrl[i];
    counters_store(R, K, err);
}

// One mc_step per launch (the plain path / mc_step API).
__global__ void __launch_bounds__(64) k_mc_step(const chromo_replica *__restrict__ reps, int rep, int ci,
                                                int max_bp1)
{
    __shared__ chromo_replica Rs;
    __shared__ EvConst EC;
    __shared__ SpecSlot slot;
    __shared__ uint32_t words[GLIBC_BUF + 1];
    load_record(&Rs, &reps[rep]);
    wave_sync();
    const chromo_replica *R = &Rs;
    // the replica's state travels while the constants and the hash are set up; nothing
    // is written before the error check
    const int64_t failed = R->counters[CHROMO_CNT_ERROR];
    chromo_ctrl C = R->ctrl[ci];
    Counters K;
    counters_load(R, K);
    const int Bp1 = R->B < 1 || R->B + 1 > max_bp1 ? max_bp1 : R->B + 1;
    uint32_t *mt_lds = (uint32_t *)(lds_dyn + wide_lds_bytes(Bp1));
    const bool need_mt = (C.move == CHROMO_CHANGE_BINDING_STATE);
    WaveRng rng;
    rng_load(R, rng, mt_lds, need_mt);
    ev_const(&EC, R);
    const EvLds S = ev_lds(lds_dyn, Bp1, 0);
    ev_clear(S);
    if (failed != 0) return;
    if (R->B < 1 || R->B + 1 > max_bp1) {
        counters_error(R, ERR_NBINDERS);
        return;
    }
    MoveOut o;
    if (R->twist) {
        switch (R->B) {
        case 1: mc_step_slot<1, true>(R, EC, rng, C, o, S, slot, words); break;
        case 2: mc_step_slot<2, true>(R, EC, rng, C, o, S, slot, words); break;
        case 3: mc_step_slot<3, true>(R, EC, rng, C, o, S, slot, words); break;
        case 4: mc_step_slot<4, true>(R, EC, rng, C, o, S, slot, words); break;
        default: o.err = ERR_NBINDERS; o.n = 0; break;
        }
    } else {
        switch (R->B) {
        case 1: mc_step_slot<1, false>(R, EC, rng, C, o, S, slot, words); break;
        case 2: mc_step_slot<2, false>(R, EC, rng, C, o, S, slot, words); break;
        case 3: mc_step_slot<3, false>(R, EC, rng, C, o, S, slot, words); break;
        case 4: mc_step_slot<4, false>(R, EC, rng, C, o, S, slot, words); break;
        default: o.err = ERR_NBINDERS; o.n = 0; break;
        }
    }
    if (!o.err && o.n > 0) record(R, C, o, K);
    rng_store(R, rng, need_mt);
    if (lane_id() == 0) R->ctrl[ci] = C;
    counters_store(R, K, o.err);
}

// The largest block of any binder count.
size_t mc_bytes()
{
    size_t b = 0;
    for (int bp1 = 2; bp1 <= CHROMO_MAX_BINDERS + 1; ++bp1) b = mc_lds_bytes(bp1) > b ? mc_lds_bytes(bp1) : b;
    return b;
}

}  // namespace

namespace chromo {

hipError_t step_setup(int lds_limit)
{
    if (mc_bytes() + 2048 > (size_t)lds_limit) return hipErrorInvalidValue;
    hipError_t e = hipFuncSetAttribute((const void *)k_mc_run, hipFuncAttributeMaxDynamicSharedMemorySize,
                                       (int)mc_bytes());
    if (e != hipSuccess) return e;
    return hipFuncSetAttribute((const void *)k_mc_step, hipFuncAttributeMaxDynamicSharedMemorySize, (int)mc_bytes());
}

hipError_t step_launch(const chromo_replica *d_reps, int rep, int ctrl, hipStream_t st)
{
    hipLaunchKernelGGL(k_mc_step, dim3(1), dim3(64), mc_bytes(), st, d_reps, rep, ctrl, CHROMO_MAX_BINDERS + 1);
    return hipGetLastError();
}

hipError_t run_any_launch(const chromo_replica *d_reps, int n_reps, int64_t steps, hipStream_t st)
{
    hipLaunchKernelGGL(k_mc_run, dim3(n_reps), dim3(64), mc_bytes(), st, d_reps, n_reps, steps,
                       CHROMO_MAX_BINDERS + 1);
    return hipGetLastError();
}

}  // namespace chromo
