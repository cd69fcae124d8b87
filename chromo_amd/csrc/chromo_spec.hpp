// chromo_spec.hpp -- device code of the speculative persistent kernel.
#pragma once

#include "chromo_mc.hpp"

namespace {

// ===========================================================================
// Speculative rounds: several proposals of one controller block evaluated at once.
//
// Inside a controller block the amplitudes are fixed, so the random draws of each
// proposal -- the proposal itself and its Metropolis draw -- do not depend on the
// accept/reject outcomes before it.  (The exception, a crank-shaft axis shorter
// than 1e-5 which draws a random axis, is detected and redone one at a time.)
// One wavefront (Shape::GEN) draws proposals ahead into a ring of slots; wavefront w <
// Shape::EV evaluates slot w of the round against the current state with ev_eval, in
// its own LDS block.  Resolution walks the slots in order: slot s keeps its evaluated
// dE unless an accepted slot s' < s of the same round wrote a bead or a voxel that s
// reads; then s and all later slots go to the next round and are evaluated again.
// Each chain therefore is the reference's sequential chain; only the number of rounds
// depends on conflicts.  What a slot cannot hold runs one at a time through
// mc_step_dev.
//
// Two shapes.  W = 2 (more replicas than compute units): wavefront 0 both draws and
// evaluates, two workgroups share a compute unit.  W = 4 (a compute unit per replica):
// three evaluators and one wavefront that only draws and keeps the books, so drawing
// leaves the evaluators' critical path.
// ===========================================================================

template <int W>
struct Shape {
    static_assert(W == 2 || W == 4, "two or four wavefronts");
    static constexpr int EV = W == 2 ? 2 : 3;       // evaluating wavefronts
    static constexpr int GEN = W == 2 ? 0 : 3;      // the wavefront that draws
    static constexpr int BOOK = W == 2 ? 1 : 3;     // the wavefront that books a round
    static constexpr int RING = W == 2 ? 4 : 8;     // slots
};

constexpr int SPEC_NMAX = SEG_MAX;    // tangent picks or binding beads of a slot
constexpr int SPEC_BEADS = 192;       // beads of a crank-shaft, end-pivot or slide slot
constexpr int SPEC_EVMAX = 3;
enum : int { SLOT_SMALL = 0, SLOT_EMPTY = 1, SLOT_SEQ = 2 };
constexpr int CK_WORDS = 40;

struct SpecSlot {
    int32_t kind, move, binder, lhs;
    int32_t ud, s1, s2, pad0;
    int64_t n, ind0, indf;
    double ang;                               // angle; slide: amplitude
    int64_t picks[SPEC_NMAX];                 // tangent rotation beads
    int32_t ps1[SPEC_NMAX], ps2[SPEC_NMAX];   // their unit-sphere draws
    int32_t newst[SPEC_NMAX];                 // binding: new states
    uint32_t ck[CK_WORDS];                    // RNG state before the proposal
};

struct SpecRes {
    double dEp, dEf, u, expdE;
    int32_t accepted, nbins, resample, overflow;
    int64_t rlo, rhi, wlo, whi;               // beads read [rlo, rhi], written [wlo, whi)
    uint32_t cmask;                           // earlier slots whose writes this one reads
    int32_t pad1;
};

struct SpecCtl {
    int32_t cnt, remaining, err;
    int32_t head;                             // ring position of the round's first slot
    int32_t tag;                              // the round's number in the launch (never repeats)
    int32_t stall;                            // = tag when a wait passed its bound
    int32_t done[SPEC_EVMAX];                 // = tag once slot s's result and voxels are published
    int32_t chk[SPEC_EVMAX];                  // = tag once slot s's conflict mask is set
};

// LDS exchange area of the one-at-a-time path (seq_step).
struct SeqIO {
    uint32_t ck[CK_WORDS];
    int32_t mti, pad0;
    chromo_ctrl C;
    MoveOut out;
};

struct SpecLayout {
    size_t seg, seg_bytes, mt, slots, res, ctl, seq, total;
};

// LDS: one evaluator block per evaluating wavefront (together they serve as the
// one-at-a-time block), the MT19937 block, the slot ring, per-slot results, the
// control words.
template <int W>
__host__ __device__ inline SpecLayout spec_layout(int Bp1)
{
    SpecLayout S;
    S.seg = 0;
    S.seg_bytes = ev_layout(Bp1, false).total;
    size_t o = S.seg_bytes * (size_t)Shape<W>::EV;
    S.mt = o;
    o = align_up(o + MT_LDS_BYTES, 16);
    S.slots = o;
    o += sizeof(SpecSlot) * (size_t)Shape<W>::RING;
    S.res = o;
    o += sizeof(SpecRes) * (size_t)Shape<W>::EV;
    S.ctl = o;
    o += sizeof(SpecCtl);
    o = align_up(o, 16);
    S.seq = o;
    o += sizeof(SeqIO);
    S.total = align_up(o, 256);
    return S;
}

struct SpecLds {
    SpecSlot *ring;
    SpecRes *res;
    SpecCtl *ctl;
    SeqIO *seq;
    uint32_t *mt;
    char *blocks;   // the evaluator blocks
};
// A stream checkpoint in LDS: the glibc words and indices, and the Philox position
// (counter, index in block; words 35-38 are not used: rng_restore needs the
// position only).
__device__ __forceinline__ void rng_save(const WaveRng &g, uint32_t *ck)
{
    const int lane = lane_id();
    uint64_t ctr = 0;
    int bi = 4;
    if (g.mode == CHROMO_RNG_PHILOX) philox_pos(g, ctr, bi);
    if (lane < 31) ck[lane] = g.g;
    if (lane == 0) {
        ck[31] = (uint32_t)g.gf;
        ck[32] = (uint32_t)g.gr;
        ck[33] = (uint32_t)ctr;
        ck[34] = (uint32_t)(ctr >> 32);
        ck[39] = (uint32_t)bi;
    }
    wave_sync();
}

// Restores the glibc and Philox streams (the MT19937 stream is never rewound:
// no proposal that is redone consumed MT19937 draws).
__device__ __forceinline__ void rng_restore(WaveRng &g, const uint32_t *ck)
{
    wave_sync();
    const int lane = lane_id();
    g.g = lane < 31 ? ck[lane] : 0u;
    g.gf = uni_i32((int)ck[31]);
    g.gr = uni_i32((int)ck[32]);
    if (g.mode == CHROMO_RNG_PHILOX) philox_set(g, (uint64_t)ck[33] | ((uint64_t)ck[34] << 32), (int)ck[39]);
}

// capped_exponential (bead_selection.pyx:19-66) with the one draw x: ok is
// cleared when the reference would draw again (r > cap) or loop for ever.
__device__ __forceinline__ int64_t cexp_once(int32_t x, int64_t window, int64_t cap, bool &ok)
{
    if (cap < 1) {
        ok = false;
        return 0;
    }
    const int64_t r = cexp_trunc(x, window);
    if (r > cap) ok = false;
    return r;
}

// from_point (bead_selection.pyx) with the side draw x_side and one exponential
// draw x_exp.
__device__ __forceinline__ int64_t from_point_once(int32_t x_side, int32_t x_exp, int64_t w, int64_t nb,
                                                   int64_t ind0, bool &ok)
{
    if (w > nb || w < 1) {
        ok = false;
        return 0;
    }
    if ((x_side & 1) == 0) {
        const int64_t ws = imax64(imin64(w, ind0), 1), ub = imax64(ind0, 1);
        if (ws > ub) ok = false;
        return ub - cexp_once(x_exp, ws, ws, ok);
    }
    const int64_t ws = imax64(imin64(w, nb - ind0), 1), ub = imax64(nb - ind0, 1);
    if (ws > ub) ok = false;
    return cexp_once(x_exp, ws, ws, ok) + ind0;
}

// Whether a slot holds a crank-shaft, end-pivot or slide window of n beads: windows the
// replica's arena does not hold are left to mc_step_dev, which reports them.
__device__ __forceinline__ bool slot_holds(const chromo_replica *R, int64_t n)
{
    return n <= SEG_MAX || (n <= SPEC_BEADS && n <= R->bead_cap && (!R->field_on || n <= R->seg_cap));
}

// Philox, crank-shaft / end-pivot / slide: the usual proposal -- every capped
// exponential accepted at its first draw, a window that a slot holds, no extra
// axis draws -- from the next eight words of the batch, read in one LDS round
// trip instead of one per draw.  The same words, in the same order and with the
// same arithmetic, as gen_slot's draw-at-a-time code.  Consumes nothing and returns
// false for any other case, which gen_slot then draws one word at a time.
template <int NB>
__device__ __forceinline__ bool gen_fast(const chromo_replica *R, WaveRng &rng, const chromo_ctrl &C, SpecSlot &S)
{
    const int mv = C.move;
    if (rng.mode != CHROMO_RNG_PHILOX ||
        (mv != CHROMO_CRANK_SHAFT && mv != CHROMO_END_PIVOT && mv != CHROMO_SLIDE))
        return false;
    const int p = uni_i32(rng.pidx);
    if (p + 8 > 4 * WAVE) return false;
    int32_t d[8];
#pragma unroll
    for (int t = 0; t < 8; ++t) d[t] = (int32_t)(uni_u32(rng.mt[p + t]) >> 1);
    const int64_t N = R->N;
    const double amp_move = C.amp_move;
    const int64_t amp_bead = C.amp_bead;
    bool ok = true;
    int used = 0;
    int64_t ind0 = 0, indf = 0;
    double ang = 0;
    int32_t s1 = 0, s2 = 0, lhs = 0, ud = 0;
    if (mv == CHROMO_CRANK_SHAFT) {
        ang = amp_move * (((double)d[0] / RMAX) - 0.5);
        const int64_t b0 = (int64_t)(int32_t)(((double)d[1] / RMAX) * (double)N);
        const int64_t b1 = imax64(from_point_once(d[2], d[3], amp_bead, N, b0, ok), 1);
        check_bead_bounds(b0, b1, N, ind0, indf);
        ud = d[4];
        used = 5;
    } else if (mv == CHROMO_END_PIVOT) {
        ang = amp_move * (((double)d[0] / RMAX) - 0.5);
        lhs = (int32_t)(d[1] & 1);
        if (amp_bead > N) ok = false;
        const int64_t r = cexp_once(d[2], amp_bead, amp_bead, ok);
        if (lhs == 1) {
            ind0 = 0;
            indf = r + 1;
        } else {
            ind0 = N - r;
            indf = N;
        }
        if (indf > N) ok = false;
        s1 = d[3];
        s2 = d[4];
        ud = d[5];
        used = 6;
    } else {
        ang = amp_move * ((double)d[0] / RMAX);
        s1 = d[1];
        s2 = d[2];
        const int64_t b0 = draw_mod(d[3], N);
        const int64_t b1 = from_point_once(d[4], d[5], amp_bead, N, b0, ok);
        check_bead_bounds(b0, b1, N, ind0, indf);
        ud = d[6];
        used = 7;
    }
    const int64_t n = indf - ind0;
    if (!ok || n < 1 || !slot_holds(R, n)) return false;
    rng.pidx = p + used;
    if (lane_id() == 0) {
        S.kind = SLOT_SMALL;
        S.move = mv;
        S.binder = 0;
        S.lhs = lhs;
        S.ud = ud;
        S.s1 = s1;
        S.s2 = s2;
        S.n = n;
        S.ind0 = ind0;
        S.indf = indf;
        S.ang = ang;
    }
    wave_sync();
    return true;
}

// Draws one proposal into slot S (wavefront 0), in the draw order of
// mc_step_dev.  A proposal that is too large for one wavefront, or that fails,
// is marked SLOT_SEQ with its draws given back: mc_step_dev redoes it.
template <int NB>
__device__ __forceinline__ int gen_slot(const chromo_replica *R, WaveRng &rng, const chromo_ctrl &C, SpecSlot &S)
{
    const int lane = lane_id();
    const int64_t N = R->N;
    rng_save(rng, S.ck);
    if (gen_fast<NB>(R, rng, C, S)) return SLOT_SMALL;
    const double amp_move = C.amp_move;
    const int64_t amp_bead = C.amp_bead;
    const int mv = C.move;
    int err = 0;
    bool seq = false;
    int64_t n = 0, ind0 = 0, indf = 0;
    double ang = 0;
    int32_t s1 = 0, s2 = 0, lhs = 0, binder = 0;
    if (mv == CHROMO_CRANK_SHAFT) {
        ang = amp_move * (((double)rnd31(rng) / RMAX) - 0.5);
        int64_t b0 = (int64_t)(int32_t)(((double)rnd31(rng) / RMAX) * (double)N);
        int64_t b1 = from_point(rng, amp_bead, N, b0, err);
        if (!err) {
            b1 = imax64(b1, 1);
            check_bead_bounds(b0, b1, N, ind0, indf);
            n = indf - ind0;
            // an empty window has coinciding axis beads (ind0 == indf == N): the
            // reference draws a random axis before it returns
            if (n == 0) {
                rnd31(rng);
                rnd31(rng);
            }
        }
        seq = err || !slot_holds(R, n);
    } else if (mv == CHROMO_END_PIVOT) {
        ang = amp_move * (((double)rnd31(rng) / RMAX) - 0.5);
        lhs = (int32_t)(rnd31(rng) & 1);
        if (lhs == 1) {
            ind0 = 0;
            indf = from_left(rng, amp_bead, N, err) + 1;
        } else {
            ind0 = from_right(rng, amp_bead, N, err);
            indf = N;
        }
        if (!err && indf > N) err = ERR_WINDOW;
        n = indf - ind0;
        seq = err || !slot_holds(R, n);
        if (!seq) {
            s1 = rnd31(rng);
            s2 = rnd31(rng);
        }
    } else if (mv == CHROMO_SLIDE) {
        ang = amp_move * ((double)rnd31(rng) / RMAX);
        s1 = rnd31(rng);
        s2 = rnd31(rng);
        int64_t b0 = draw_mod(rnd31(rng), N);
        int64_t b1 = from_point(rng, amp_bead, N, b0, err);
        if (!err) {
            check_bead_bounds(b0, b1, N, ind0, indf);
            n = indf - ind0;
        }
        seq = err || !slot_holds(R, n);
    } else if (mv == CHROMO_TANGENT_ROTATION) {
        ang = amp_move * (((double)rnd31(rng) / RMAX) - 0.5);
        int64_t k = draw_mod(rnd31(rng), amp_bead) + 1;
        n = k;
        seq = (k > N) || (k > SPEC_NMAX);
        int64_t fpick = 0;
        int32_t fd1 = 0, fd2 = 0;
        if (!seq && tangent_draws_at_once(rng, k, N, fpick, fd1, fd2)) {
            if (lane < k) {
                S.picks[lane] = fpick;
                S.ps1[lane] = fd1;
                S.ps2[lane] = fd2;
            }
        } else if (!seq) {
            int64_t mine = 0;
            for (int64_t i = 0; i < k && !seq; ++i) {
                for (int it = 0;; ++it) {
                    // a pick that does not end is left to mc_step_dev, which reports it
                    if (it >= SPIN_LIMIT) {
                        seq = true;
                        break;
                    }
                    int64_t c = draw_mod(rnd31(rng), N);
                    if (!wave_any(lane < i && mine == c)) {
                        if (lane == i) mine = c;
                        break;
                    }
                }
            }
            if (lane < k) S.picks[lane] = mine;
            for (int64_t i = 0; i < k && !seq; ++i) {
                int32_t a = rnd31(rng);
                int32_t b = rnd31(rng);
                if (lane == 0) {
                    S.ps1[i] = a;
                    S.ps2[i] = b;
                }
            }
        }
    } else {
        binder = (int32_t)(rnd31(rng) % NB);
        const int64_t ntails = R->sites[binder];
        int64_t b0 = draw_mod(rnd31(rng), N);
        int64_t b1 = from_point(rng, amp_bead, N, b0, err);
        if (!err) {
            check_bead_bounds(b0, b1, N, ind0, indf);
            n = indf - ind0;
        }
        seq = err || n > SPEC_NMAX;
        if (!seq) {
            for (int64_t i = 0; i < n; ++i) {
                int st = (int)rnd_randint(rng, ntails + 1);
                if (lane == 0) S.newst[i] = st;
            }
        }
    }
    int kind;
    int32_t ud = 0;
    if (seq) {
        rng_restore(rng, S.ck);
        kind = SLOT_SEQ;
    } else if (n == 0) {
        kind = SLOT_EMPTY;
    } else {
        ud = rnd31(rng);
        kind = SLOT_SMALL;
    }
    if (lane == 0) {
        S.kind = kind;
        S.move = mv;
        S.binder = binder;
        S.lhs = lhs;
        S.ud = ud;
        S.s1 = s1;
        S.s2 = s2;
        S.n = n;
        S.ind0 = ind0;
        S.indf = indf;
        S.ang = ang;
    }
    wave_sync();
    return kind;
}

// One proposal of a sequential round by the drawing wavefront alone, in the
// one-at-a-time block (the slot blocks' LDS: every slot hash is empty again on
// return).  The RNG, the controller and the result pass through LDS, io.
template <int NB, int W, bool TW>
__device__ __forceinline__ void seq_step(const chromo_replica *R, const EvConst &EC, SeqIO *io, uint32_t *mt,
                                         char *blocks)
{
    const int lane = lane_id();
    WaveRng rng;
    rng.mode = uni_i32(R->rng_mode);
    rng.k0 = uni_u32(R->rng[CHROMO_RNG_PHILOX_KEY]);
    rng.k1 = uni_u32(R->rng[CHROMO_RNG_PHILOX_KEY + 1]);
    rng.pbase = PHILOX_NONE;
    rng.pidx = 0;
    rng.mt = mt;
    rng_restore(rng, io->ck);
    rng.mti = uni_i32(io->mti);
    chromo_ctrl C = io->C;
    MoveOut o;
    o.err = 0;
    o.n = 0;
    Proposal P;
    double u = 0;
    const bool go = mc_propose<NB>(R, rng, C, o, P, u);
    // the RNG goes back to LDS now, so that it is not held through the evaluation
    rng_save(rng, io->ck);
    if (lane == 0) io->mti = rng.mti;
    const EvLds S = ev_lds(blocks, NB + 1, true);
    ev_clear(S);
    if (go) mc_evaluate<NB, TW>(R, EC, C, o, P, u, S);
    const size_t bytes = ev_layout(NB + 1, false).total;
    for (int b = 0; b < Shape<W>::EV; ++b) ev_clear(ev_lds(blocks + bytes * b, NB + 1, false));
    if (lane == 0) {
        io->C = C;
        io->out = o;
    }
    wave_sync();
}

// The proposal of slot S from its stored draws: the arithmetic of mc_step_dev's
// proposal part (move_funcs.pyx).  The axis and fulcrum beads lie in the window or
// next to it: their coordinates come from B.  False when a crank-shaft's axis
// beads coincide: the reference then draws a random axis, which only the
// one-at-a-time path can do in stream order.
template <int NB>
__device__ __forceinline__ bool slot_proposal(const chromo_replica *R, const SpecSlot &S, Proposal &P,
                                              const EvBeads<NB> &B)
{
    const int lane = lane_id();
    const int64_t N = R->N;
    const int mv = S.move;
    const int64_t n = S.n, ind0 = S.ind0, indf = S.indf;
    P.move = mv;
    P.n = n;
    P.ind0 = ind0;
    P.indf = indf;
    P.binder = S.binder;
    P.mypick = 0;
    P.mynew = 0;
#pragma unroll
    for (int q = 0; q < 12; ++q) P.T[q] = 0;
#pragma unroll
    for (int q = 0; q < 9; ++q) P.myT[q] = 0;
    if (mv == CHROMO_CRANK_SHAFT) {
        // get_crank_shaft_axis / _fulcrum, move_funcs.pyx:157-280
        int64_t ia, ib;
        const int64_t indf_m1 = indf - 1, ind0_m1 = ind0 - 1;
        if (ind0 == indf_m1 && ind0 == 0) { ia = indf; ib = ind0; }
        else if (ind0 == indf_m1 && ind0 == N - 1) { ia = ind0; ib = ind0_m1; }
        else if (ind0 == 0 && indf == N) { ia = indf_m1; ib = ind0; }
        else if (ind0 == 0) { ia = indf; ib = ind0; }
        else if (indf == N) { ia = indf_m1; ib = ind0_m1; }
        else { ia = indf; ib = ind0_m1; }
        int64_t ifc;
        if (ind0 == 0 && indf != N) ifc = indf;
        else if (ind0 != 0 && indf == N) ifc = ind0_m1;
        else if (ind0 == 0 && indf == N) ifc = ind0;
        else ifc = ind0_m1;
        const double sa = sin(S.ang), ca = cos(S.ang);
        double ra[3], rb[3], pt[3], dir[3];
        ev_r3(R, B, ia, ind0, indf, ra);
        ev_r3(R, B, ib, ind0, indf, rb);
        ev_r3(R, B, ifc, ind0, indf, pt);
        for (int i = 0; i < 3; ++i) dir[i] = ra[i] - rb[i];
        double mag = sqrt(dir[0] * dir[0] + dir[1] * dir[1] + dir[2] * dir[2]);
        if (mag < 1E-5) return false;
        double sc = 1.0 / mag;
        for (int i = 0; i < 3; ++i) dir[i] = dir[i] * sc;
        axis_rotation_cs(dir, pt, ca, sa, P.T);
    } else if (mv == CHROMO_END_PIVOT) {
        // get_end_pivot_fulcrum, move_funcs.pyx:349-398
        int64_t ifc;
        if (ind0 == 0 && indf != N) ifc = indf;
        else if (ind0 != 0 && indf == N) ifc = ind0 - 1;
        else if (ind0 == 0 && indf == N && S.lhs == 1) ifc = indf - 1;
        else ifc = ind0;
        double pt[3], axis[3], sa, ca;
        sphere_from_uni(S.s1, S.s2, S.ang, axis, sa, ca);
        ev_r3(R, B, ifc, ind0, indf, pt);
        axis_rotation_cs(axis, pt, ca, sa, P.T);
    } else if (mv == CHROMO_SLIDE) {
        double dir[3], sa, ca;
        sphere_from_uni(S.s1, S.s2, 0.0, dir, sa, ca);
        for (int i = 0; i < 3; ++i) dir[i] *= S.ang;
        P.T[3] = dir[0];
        P.T[7] = dir[1];
        P.T[11] = dir[2];
    } else if (mv == CHROMO_TANGENT_ROTATION) {
        const double sa = sin(S.ang), ca = cos(S.ang);
        if (lane < n) {
            double dir[3], T[12];
            const double origin[3] = {0., 0., 0.};
            P.mypick = S.picks[lane];
            sphere_from(S.ps1[lane], S.ps2[lane], dir);
            axis_rotation_cs(dir, origin, ca, sa, T);
            for (int j = 0; j < 3; ++j)
                for (int q = 0; q < 3; ++q) P.myT[3 * j + q] = T[4 * j + q];
        }
    } else {
        if (lane < n) P.mynew = S.newst[lane];
    }
    return true;
}

// Evaluates slot S into res, its trial state in K, P and the block G, whose hash then
// holds the slot's voxels (returned: how many; 0 and an empty hash when the slot has to
// be redone one at a time).
template <int NB, bool TW>
__device__ __forceinline__ int eval_slot(const chromo_replica *R, const EvConst &EC, const SpecSlot &S, SpecRes &res,
                                         Proposal &P, EvKeep &K, const EvLds &G)
{
    const int lane = lane_id();
    const int64_t ind0 = S.ind0, indf = S.indf;
    if (lane == 0) {
        res.cmask = 0;
        res.resample = 0;
        res.overflow = 0;
        res.nbins = 0;
        res.rlo = ind0 - 1;
        res.rhi = indf;
        res.wlo = ind0;
        res.whi = indf;
    }
    // every load of the first chunk but the densities', issued before the proposal's
    // arithmetic
    EvBeads<NB> B;
    const int64_t pick = (S.move == CHROMO_TANGENT_ROTATION && (lane & 31) < S.n) ? S.picks[lane & 31] : 0;
    ev_load<NB, TW>(R, S.move, S.n, ind0, indf, 0, pick, B);
    if (!slot_proposal<NB>(R, S, P, B)) {
        if (lane == 0) res.resample = 1;
        wave_sync();
        return 0;
    }
    EvRes sr;
    const double u = (double)S.ud / RMAX;
    ev_eval<NB, TW>(R, EC, P, u, G, sr, K, B);
    if (sr.overflow) {
        // more voxels than the block holds: the one-at-a-time path evaluates it
        if (lane == 0) res.overflow = 1;
        wave_sync();
        return 0;
    }
    if (lane == 0) {
        res.dEp = sr.dEp;
        res.dEf = sr.dEf;
        res.u = u;
        res.expdE = sr.expdE;
        res.accepted = sr.accepted;
        res.nbins = sr.U;
    }
    wave_sync();
    return sr.U;
}

template <int RING>
__device__ __forceinline__ const SpecSlot &ring_at(const SpecSlot *ring, int head, int s)
{
    return ring[(head + s) & (RING - 1)];
}

// Whether slot s (its voxels numbered in block G, U of them) reads what the accepted
// slot a < s of the round writes: a shared bead (tangent rotation: picks within one
// bead of each other), or a shared voxel, looked up in a's own hash (block A).
template <int RING>
__device__ __forceinline__ bool spec_conflict(const SpecSlot *ring, int head, const SpecRes *res, const EvLds &G, int U,
                                              int s, const EvLds &A, int a)
{
    const int lane = lane_id();
    const SpecSlot &S = ring_at<RING>(ring, head, s), &Q = ring_at<RING>(ring, head, a);
    bool hit = false;
    if (S.move == CHROMO_TANGENT_ROTATION) {
        if (lane < S.n) {
            const int64_t mine = S.picks[lane];
            for (int64_t q = 0; q < Q.n; ++q) {
                const int64_t d = Q.picks[q] - mine;
                hit |= d >= -1 && d <= 1;
            }
        }
    } else {
        hit = res[a].wlo <= res[s].rhi && res[s].rlo < res[a].whi;
        if (res[a].nbins > 0)
            for (int q = lane; q < U; q += WAVE) {
                const int2 v = G.uv[q];
                int h = (int)((uint32_t)v.y >> 16);
                for (int probes = 0; probes < A.hsize; ++probes) {
                    const int key = A.hkey[h];
                    hit |= key == v.x;
                    if (key == v.x || key == HKEY_EMPTY) break;
                    h = (h + 1) & (A.hsize - 1);
                }
            }
    }
    return wave_any(hit);
}

// The drawing wavefront: appends proposals to the queue of `q` slots starting at ring
// position head until it holds `limit`, or `remaining` (the block's unresolved
// proposals), or ends with a SLOT_SEQ one.  Returns the new queue length.
template <int NB, int RING>
__device__ __forceinline__ int spec_gen(const chromo_replica *R, WaveRng &rng, const chromo_ctrl &C, SpecSlot *ring,
                                        int head, int q, int limit, int remaining)
{
    if (q >= limit || q >= remaining) return q;
    bool stop = q > 0 && ring_at<RING>(ring, head, q - 1).kind == SLOT_SEQ;
    while (!stop && q < limit && q < remaining) {
        const int kind = gen_slot<NB>(R, rng, C, ring[(head + q) & (RING - 1)]);
        ++q;
        stop = kind == SLOT_SEQ;
    }
    return q;
}

// One wavefront: AcceptanceTracker updates (mc_stat.py:190-208), controller counts,
// replica counters and log records of the resolved slots 0..F-1, one slot per
// lane; the same totals as record() called once per slot in order.
template <int RING>
__device__ __forceinline__ void spec_book(const chromo_replica *R, chromo_ctrl &C, Counters &K,
                                          const SpecSlot *ring, int head, const SpecRes *res, int F)
{
    const int lane = lane_id();
    const bool live = lane < F && ring_at<RING>(ring, head, lane < F ? lane : 0).kind != SLOT_EMPTY;
    int64_t n = 0, nb = 0, bytes = 0;
    int acc = 0, tie = 0;
    if (live) {
        const SpecSlot &S = ring_at<RING>(ring, head, lane);
        const SpecRes &q = res[lane];
        n = S.n;
        nb = q.nbins;
        acc = q.accepted;
        tie = fabs(q.u - q.expdE) < 1E-12;
        bytes = move_bytes(S.move, n, nb, R->B, acc);
    }
    const uint64_t live_m = __ballot(live);
    const uint64_t acc_m = __ballot(live && acc);
    const uint64_t tie_m = __ballot(live && tie);
    static_assert(SPEC_EVMAX <= 8, "bookkeeping sums over the first eight lanes");
    const int64_t sn = sum_lanes8_i64(n), sb = sum_lanes8_i64(nb), sy = sum_lanes8_i64(bytes);
    const int64_t logged = K.logged;
    const int nlive = __popcll(live_m);
    if (R->log != nullptr && live) {
        const int64_t at = logged + __popcll(live_m & ((1ull << lane) - 1));
        if (at < R->log_cap) {
            const SpecSlot &S = ring_at<RING>(ring, head, lane);
            const SpecRes &q = res[lane];
            chromo_move_log &Lg = R->log[at];
            Lg.move = S.move;
            Lg.accepted = q.accepted;
            Lg.n = S.n;
            Lg.ind0 = S.move == CHROMO_TANGENT_ROTATION ? S.picks[0] : S.ind0;
            Lg.indf = S.move == CHROMO_TANGENT_ROTATION ? S.picks[0] + 1 : S.indf;
            Lg.dE_poly = q.dEp;
            Lg.dE_field = q.dEf;
            Lg.u = q.u;
            Lg.exp_dE = q.expdE;
            Lg.n_bins = q.nbins;
        }
    }
    wave_sync();
    if (lane == 0) {
        // every field is read before any is written: the compiler cannot tell C from
        // K, and interleaved reads and writes would wait on LDS one at a time
        const double alpha = C.alpha;
        double rate = C.rate;
        const auto na = C.num_attempt, nsu = C.num_success;
        const int64_t kp = K.prop, ka = K.acc, kn = K.sumn, kb = K.sumb, kt = K.ties, ky = K.bytes;
        for (int s = 0; s < F; ++s)
            if ((live_m >> s) & 1) rate = (alpha * (double)((acc_m >> s) & 1)) + (1 - alpha) * rate;
        const int nacc = __popcll(acc_m);
        C.rate = rate;
        C.num_attempt = na + F;
        C.num_success = nsu + nacc;
        K.prop = kp + nlive;
        K.acc = ka + nacc;
        K.sumn = kn + sn;
        K.sumb = kb + sb;
        K.ties = kt + __popcll(tie_m);
        K.bytes = ky + sy;
        if (R->log != nullptr && logged < R->log_cap)
            K.logged = logged + nlive < R->log_cap ? logged + nlive : R->log_cap;
    }
    wave_sync();
}

// Raises a flag of the round for the other wavefronts: what this wavefront wrote to
// LDS before is visible to who sees it.
__device__ __forceinline__ void flag_raise(int32_t *f, int32_t tag)
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    if (lane_id() == 0) __hip_atomic_store(f, tag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// Waits for a flag; false when it did not come within SPIN_LIMIT looks.
__device__ __forceinline__ bool flag_wait(const int32_t *f, int32_t tag)
{
    int spins = 0;
    while (uni_i32(__hip_atomic_load(f, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP)) != tag)
        if (++spins >= SPIN_LIMIT) break;
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    return spins < SPIN_LIMIT;
}

// One controller block.  C and K live in LDS: only the booking wavefront touches them
// between two barriers, and keeping them out of registers leaves those to the
// evaluation.
//
// A round, between two barriers:
//  * wavefront s < cnt evaluates slot s and raises done[s]; slot 0 stands whatever the
//    others do (nothing precedes it), so it is committed at once -- a later slot that
//    reads what it writes is redone anyway;
//  * slot s waits for done[a] of every a < s, looks its voxels and beads up in the
//    accepted ones', and raises chk[s];
//  * the drawing wavefront meanwhile draws the following proposals into the ring;
//  * every wavefront resolves the slots it needs from the published results, in the
//    same way: slot s commits if nothing before it ends the round.
// A slot's hash is emptied at the start of its wavefront's next evaluation, when
// nobody looks into it any more.  The flag waits are bounded; a wait that passes its
// bound stops the replica with ERR_SPIN at the next round's top.
template <int NB, int W, bool TW>
__device__ __forceinline__ void spec_block(const chromo_replica *R, const EvConst &EC, WaveRng &rng, chromo_ctrl &C,
                                           Counters &K, const SpecLds &L, int &held)
{
    using SH = Shape<W>;
    constexpr int RING = SH::RING, EV = SH::EV, Bp1 = NB + 1;
    static_assert((RING & (RING - 1)) == 0, "ring positions wrap by mask");
    const int wv = wave_id(), lane = lane_id();
    const size_t seg_bytes = ev_layout(Bp1, false).total;
    const EvLds G = ev_lds(L.blocks + seg_bytes * (wv < EV ? wv : 0), Bp1, false);
    SpecSlot *ring = L.ring;
    // the drawing wavefront's
    int head = 0;                      // ring position of the first queued slot
    int nq = 0;                        // slots queued
    int remaining = C.num_per_cycle;   // proposals of the block not yet resolved
    int pend = 0;                      // error to publish before the next barrier
    int32_t tag = uni_i32(L.ctl->tag); // the round's number in the launch
    int64_t rounds = 0;
    // every round resolves a proposal or turns its first slot into a sequential one
    const int64_t max_rounds = 2 * (int64_t)C.num_per_cycle + 64;
    // drawing ahead is off where a redone proposal would have to rewind MT19937
    const bool ahead = !(rng.mode == CHROMO_RNG_GLIBC && C.move == CHROMO_CHANGE_BINDING_STATE);
    for (;;) {
        if (wv == SH::GEN) {
            // L.ctl->err is written only here, before the barrier after which every
            // wavefront reads it
            if (++rounds > max_rounds) pend = ERR_SPIN;
            if (uni_i32(L.ctl->stall) >= 0) pend = ERR_SPIN;
            if (pend && lane == 0) L.ctl->err = pend;
            if (!pend) {
                tag += 1;
                nq = spec_gen<NB, RING>(R, rng, C, ring, head, nq, EV, remaining);
                const int nr = nq < EV ? nq : EV;
                // leading slots that are not SLOT_SEQ, all kinds read at once
                const int kd = lane < nr ? ring_at<RING>(ring, head, lane).kind : SLOT_SEQ;
                const uint64_t seqm = __ballot(kd == SLOT_SEQ);
                const int cnt = seqm ? (int)__builtin_ctzll(seqm) : nr;
                if (lane == 0) {
                    L.ctl->cnt = cnt;
                    L.ctl->remaining = remaining;
                    L.ctl->head = head;
                    L.ctl->tag = tag;
                }
            }
        }
        __syncthreads();
        if (L.ctl->err || L.ctl->remaining <= 0) break;
        const int cnt = uni_i32(L.ctl->cnt), h = uni_i32(L.ctl->head);
        if (ring_at<RING>(ring, h, 0).kind == SLOT_SEQ) {
            held = 0;   // the one-at-a-time block lies over the slot blocks and leaves them empty
            if (wv == SH::GEN) {
                // the slot hashes may still hold the last round's voxels: seq_step clears
                // what it uses, before and after
                SeqIO *io = L.seq;
                const SpecSlot &S0 = ring_at<RING>(ring, h, 0);
                for (int i = lane; i < CK_WORDS; i += WAVE) io->ck[i] = S0.ck[i];
                if (lane == 0) {
                    io->mti = rng.mti;
                    io->C = C;
                }
                wave_sync();
                seq_step<NB, W, TW>(R, EC, io, L.mt, L.blocks);
                rng_restore(rng, io->ck);
                rng.mti = uni_i32(io->mti);
                if (lane == 0) C = io->C;
                wave_sync();
                const MoveOut o = io->out;
                if (o.err) {
                    pend = o.err;
                } else if (o.n > 0) {
                    record(R, C, o, K);
                }
                remaining -= 1;
                // nothing is drawn past a SLOT_SEQ slot
                head = (head + 1) & (RING - 1);
                nq = 0;
            }
        } else {
            const int32_t now = uni_i32(L.ctl->tag);
            const bool evaluates = wv < EV && wv < cnt;
            const SpecSlot &mys = ring_at<RING>(ring, h, evaluates ? wv : 0);
            const bool mine = evaluates && mys.kind == SLOT_SMALL;
            bool stalled = false, committed = false;
            EvKeep keep;
            Proposal P;
            if (mine) {
                ev_release(G, held);
                held = eval_slot<NB, TW>(R, EC, mys, L.res[wv], P, keep, G);
            }
            if (evaluates) flag_raise(&L.ctl->done[wv], now);
            if (wv == 0 && mine && L.res[0].accepted && !L.res[0].resample && !L.res[0].overflow) {
                ev_commit<NB>(R, P, keep, G, held);
                committed = true;
            }
            if (evaluates && wv > 0) {
                uint32_t m = 0;
                const bool look = mine && !L.res[wv].resample && !L.res[wv].overflow;
                for (int a = 0; a < wv; ++a) {
                    if (!flag_wait(&L.ctl->done[a], now)) {
                        stalled = true;
                        break;
                    }
                    if (!look || ring_at<RING>(ring, h, a).kind != SLOT_SMALL) continue;
                    const SpecRes &q = L.res[a];
                    if (!q.accepted || q.resample || q.overflow) continue;
                    if (spec_conflict<RING>(ring, h, L.res, G, held, wv, ev_lds(L.blocks + seg_bytes * a, Bp1, false), a))
                        m |= 1u << a;
                }
                if (lane == 0) L.res[wv].cmask = m;
                if (stalled && lane == 0) L.ctl->stall = now;
                flag_raise(&L.ctl->chk[wv], now);
            }
            // the following proposals
            if (wv == SH::GEN && ahead && !pend) nq = spec_gen<NB, RING>(R, rng, C, ring, head, nq, RING, remaining);
            // the results this wavefront resolves: all for the drawing and booking ones,
            // the slots before its own for the others
            const bool all = wv == SH::GEN || wv == SH::BOOK;
            const int upto = all ? cnt : (evaluates ? wv + 1 : 0);
            if (upto > 0 && !evaluates) stalled |= !flag_wait(&L.ctl->done[0], now);
            for (int s = 1; s < upto; ++s)
                if (s != wv) stalled |= !flag_wait(&L.ctl->chk[s], now);
            if (stalled && lane == 0) L.ctl->stall = now;
            // resolution, identical in every wavefront; lane s reads slot s's result,
            // all slots in one LDS round trip
            uint32_t kd = SLOT_EMPTY, cmk = 0, ov = 0, rs = 0, ac = 0;
            if (lane < upto) {
                const SpecRes &q = L.res[lane];
                kd = (uint32_t)ring_at<RING>(ring, h, lane).kind;
                cmk = q.cmask;
                ov = (uint32_t)q.overflow;
                rs = (uint32_t)q.resample;
                ac = (uint32_t)q.accepted;
            }
            int F = upto, rew = 0;
            uint32_t accm = 0;
            for (int s = 0; s < upto; ++s) {
                if ((int)readlane_u32(kd, s) == SLOT_EMPTY) continue;
                const uint32_t q_cmask = readlane_u32(cmk, s), q_overflow = readlane_u32(ov, s);
                if (q_cmask & accm) {
                    F = s;
                    break;
                }
                // an axis to be drawn again, or more voxels than a block holds: the
                // sequential path redoes it
                if (readlane_u32(rs, s) || q_overflow) {
                    F = s;
                    rew = 1;
                    break;
                }
                if (readlane_u32(ac, s)) accm |= 1u << s;
            }
            if (mine && !committed && wv < F && L.res[wv].accepted) ev_commit<NB>(R, P, keep, G, held);
            // only the barrier below orders C and K for the next reader
            if (wv == SH::BOOK) spec_book<RING>(R, C, K, ring, h, L.res, F);
            if (wv == SH::GEN) {
                if (rew) {
                    // slot F is redone one at a time; what was drawn after it is
                    // dropped (the sequential path rewinds the streams to it)
                    if (lane == 0) ring[(head + F) & (RING - 1)].kind = SLOT_SEQ;
                    nq = F + 1;
                }
                head = (head + F) & (RING - 1);
                nq -= F;
                remaining -= F;
            }
        }
        __syncthreads();
    }
}

template <int NB, int W, bool TW>
__device__ __forceinline__ void spec_run(const chromo_replica *R, const EvConst &EC, int64_t steps)
{
    using SH = Shape<W>;
    constexpr int Bp1 = NB + 1;
    const SpecLayout SL = spec_layout<W>(Bp1);
    const int wv = wave_id(), lane = lane_id();
    SpecLds L;
    L.blocks = lds_dyn + SL.seg;
    L.ring = (SpecSlot *)(lds_dyn + SL.slots);
    L.res = (SpecRes *)(lds_dyn + SL.res);
    L.ctl = (SpecCtl *)(lds_dyn + SL.ctl);
    L.seq = (SeqIO *)(lds_dyn + SL.seq);
    L.mt = (uint32_t *)(lds_dyn + SL.mt);
    if (wv < SH::EV) ev_clear(ev_lds(L.blocks + SL.seg_bytes * wv, Bp1, false));
    __shared__ chromo_ctrl sctrl[MAX_CTRL];
    __shared__ Counters sK;
    const int nc = R->n_ctrl < MAX_CTRL ? R->n_ctrl : MAX_CTRL;
    WaveRng rng;
    rng.mode = uni_i32(R->rng_mode);
    bool need_mt = false;
    if (wv == SH::GEN) {
        need_mt = any_binding(R);
        rng_load(R, rng, L.mt, need_mt);
        if (lane == 0) {
            counters_load(R, sK);
            for (int i = 0; i < nc; ++i) sctrl[i] = R->ctrl[i];
            L.ctl->err = 0;
            L.ctl->tag = 0;
            L.ctl->stall = -1;
            for (int s = 0; s < SPEC_EVMAX; ++s) L.ctl->done[s] = L.ctl->chk[s] = -1;
        }
    }
    __syncthreads();
    int held = 0;   // voxels in this wavefront's hash
    for (int64_t s = 0; s < steps; ++s) {
        for (int ci = 0; ci < nc; ++ci) {
            if (sctrl[ci].on == 1) spec_block<NB, W, TW>(R, EC, rng, sctrl[ci], sK, L, held);
            if (wv == 0 && lane == 0 && !L.ctl->err) update_amplitudes_dev(sctrl[ci]);
            __syncthreads();
            if (L.ctl->err) break;
        }
        if (L.ctl->err) break;
    }
    if (wv == SH::GEN) {
        rng_store(R, rng, need_mt);
        if (lane == 0)
            for (int i = 0; i < nc; ++i) R->ctrl[i] = sctrl[i];
        counters_store(R, sK, L.ctl->err);
    }
}

}  // namespace
