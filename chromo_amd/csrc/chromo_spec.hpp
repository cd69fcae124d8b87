// chromo_spec.hpp -- device code of the speculative persistent kernel.
#pragma once

#include <cstddef>

#include "chromo_mc.hpp"

namespace {

// ===========================================================================
// Speculative evaluation: several proposals of a chain in flight at once.
//
// Inside a controller block the amplitudes are fixed, and a controller's amplitudes
// change only at the end of its own block, so the random draws of each proposal -- the
// proposal itself and its Metropolis draw -- do not depend on the accept/reject outcomes
// before it.  (The exception, a crank-shaft axis shorter than 1e-5 which draws a random
// axis, is detected and redone one at a time.)
//
// Proposals are numbered through the launch.  The drawing wavefront (Shape::GEN) draws
// them in order into a ring of slots.  Each of Shape::EV evaluating wavefronts takes the
// next number, evaluates that slot against the committed state with ev_eval in its own
// LDS block, and then waits for its turn: slots are resolved in order.  Meanwhile it
// looks each earlier slot that is resolved as accepted up in its own hash: a slot that
// reads a bead or a voxel written since its evaluation began is evaluated again at
// once.  At its turn it commits an accepted proposal and passes the turn on.  The
// chain therefore is the reference's sequential chain, whatever the schedule; and no
// wavefront waits for the slowest evaluation of a group, nor at the end of a block.
// What a slot cannot hold runs one at a time through mc_step_dev, when it is its turn
// and nothing else is in flight.
//
// Two shapes.  W = 2 (more replicas than compute units): wavefront 0 both draws and
// evaluates, two workgroups share a compute unit.  W = 4 (a compute unit per replica):
// three evaluators and one wavefront that only draws and keeps the books.
// ===========================================================================

template <int W>
struct Shape {
    static_assert(W == 2 || W == 4, "two or four wavefronts");
    static constexpr int EV = W == 2 ? 2 : 3;       // evaluating wavefronts
    static constexpr int GEN = W == 2 ? 0 : 3;      // the wavefront that draws and books
    static constexpr int RING = W == 2 ? 8 : 16;    // slots
    // Slots drawn past the first unresolved one, at most, and slots resolved but not yet
    // booked.  Slot d takes the place of slot d - RING, which has to be booked, and which a
    // slot in flight (numbers below first + EV) may still look at when it is among the
    // EV - 1 before that one.
    static constexpr int AHEAD = W == 2 ? 6 : 8;
    static_assert(AHEAD <= RING - EV + 1, "no slot is overwritten while it is looked at");
    // Voxel lists: slot a's is looked at by the next EV - 1 slots, which can be in flight
    // together with the EV - 1 after them.  Its own wavefront reads it up to its turn and
    // not after: from there on nothing keeps the others from a slot that has this list.
    static constexpr int LISTS = 2 * EV - 1;
    // Voxels of a block: two workgroups on a compute unit, or one.
    __host__ __device__ static constexpr int ucap(int Bp1)
    {
        return W == 2 ? (Bp1 <= 2 ? 640 : (Bp1 == 3 ? 528 : (Bp1 == 4 ? 432 : 368)))
                      : (Bp1 <= 4 ? 704 : 576);
    }
};

constexpr int SPEC_NMAX = SEG_MAX;    // tangent picks or binding beads of a slot
constexpr int SPEC_BEADS = 192;       // beads of a crank-shaft, end-pivot or slide slot
constexpr int SPEC_EVMAX = 3;
constexpr int CTL_WORDS = 16;
enum : int { SLOT_SMALL = 0, SLOT_EMPTY = 1, SLOT_SEQ = 2 };
constexpr int CK_WORDS = 40;
constexpr int GLIBC_BLOCKS = 4;                       // 31-word blocks of the additive generator drawn ahead, at most
constexpr int GLIBC_BUF = 31 * (GLIBC_BLOCKS + 1);    // its state, oldest word first, then the blocks
// a binding slot always fits a block: it is never given back (its MT19937 draws could
// not be)
static_assert(8 * SPEC_NMAX <= 368, "voxels of a binding slot");

struct SpecSlot {
    int32_t kind, move, binder, lhs;
    int32_t ud, s1, s2, list;                 // list: which voxel list is the slot's
    int64_t n, ind0, indf;
    double ang;                               // angle; slide: amplitude
    int32_t picks[SPEC_NMAX];                 // tangent rotation beads (31-bit draws)
    int32_t ps1[SPEC_NMAX], ps2[SPEC_NMAX];   // their unit-sphere draws
    int32_t newst[SPEC_NMAX];                 // binding: new states
    uint32_t ck[CK_WORDS];                    // RNG state before the proposal
};

struct SpecRes {
    double dEp, dEf, u, expdE;
    int32_t accepted, nbins, resample, overflow;
    int64_t rlo, rhi, wlo, whi;               // beads read [rlo, rhi], written [wlo, whi)
};

// The launch's state, slots by their number in it (numbers wrap: compared by difference).
struct SpecCtl {
    uint32_t next;                            // next slot to take
    uint32_t drawn;                           // slots before it are in the ring
    uint32_t resolved;                        // slots before it are committed or rejected
    int32_t back;                             // 1: slot back_at, then the first unresolved one, has to be
    uint32_t back_at;                         //    redone one at a time
    int32_t alone;                            // 1: the drawing wavefront runs a slot one at a time
    int32_t stop, err;
    int32_t idle[SPEC_EVMAX];                 // evaluating wavefront holds nothing in its block
    int32_t pad[CTL_WORDS - 8 - SPEC_EVMAX];
};
static_assert(sizeof(SpecCtl) == 4 * CTL_WORDS, "ctl_look reads it whole");

// LDS exchange area of the one-at-a-time path (seq_step).
struct SeqIO {
    uint32_t ck[CK_WORDS];
    int32_t mti, pad0;
    chromo_ctrl C;
    MoveOut out;
    uint32_t words[GLIBC_BUF + 1];   // gen_batch's
};

struct SpecLayout {
    size_t seg_bytes, lists, mt, slots, res, ctl, seq, total;
};

// LDS: one evaluator block per evaluating wavefront (together they serve as the
// one-at-a-time block), the voxel lists, the MT19937 block, the slot ring, per-slot
// results, the control words.
template <int W>
__host__ __device__ inline SpecLayout spec_layout(int Bp1)
{
    SpecLayout S;
    S.seg_bytes = ev_layout(Bp1, Shape<W>::ucap(Bp1)).total;
    size_t o = S.seg_bytes * (size_t)Shape<W>::EV;
    S.lists = o;
    o += sizeof(int2) * (size_t)(Shape<W>::LISTS * Shape<W>::ucap(Bp1));
    S.mt = o;
    o = align_up(o + MT_LDS_BYTES, 16);
    S.slots = o;
    o += sizeof(SpecSlot) * (size_t)Shape<W>::RING;
    S.res = o;
    o += sizeof(SpecRes) * (size_t)Shape<W>::RING;
    S.ctl = o;
    o = align_up(o + sizeof(SpecCtl), 16);
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
    int2 *lists;
    char *blocks;   // the evaluator blocks
};

// A stream checkpoint in LDS: the additive generator's words and indices, or the Philox
// position (words 33 and 34 the counter, 39 the index in its block: all rng_restore needs).
__device__ __forceinline__ void rng_save(const WaveRng &g, uint32_t *ck)
{
    const int lane = lane_id();
    if (g.mode == CHROMO_RNG_PHILOX) {
        uint64_t ctr = 0;
        int bi = 4;
        philox_pos(g, ctr, bi);
        if (lane == 0) {
            ck[33] = (uint32_t)ctr;
            ck[34] = (uint32_t)(ctr >> 32);
            ck[39] = (uint32_t)bi;
        }
    } else {
        if (lane < 31) ck[lane] = g.g;
        if (lane == 0) {
            ck[31] = (uint32_t)g.gf;
            ck[32] = (uint32_t)g.gr;
        }
    }
    wave_sync();
}

// Restores the stream (MT19937 is never rewound: no proposal that is redone consumed
// MT19937 draws).
__device__ __forceinline__ void rng_restore(WaveRng &g, const uint32_t *ck)
{
    wave_sync();
    const int lane = lane_id();
    if (g.mode == CHROMO_RNG_PHILOX) {
        philox_set(g, (uint64_t)ck[33] | ((uint64_t)ck[34] << 32), (int)ck[39]);
    } else {
        g.g = lane < 31 ? ck[lane] : 0u;
        g.gf = uni_i32((int)ck[31]);
        g.gr = uni_i32((int)ck[32]);
    }
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

// The next words of the stream in LDS, in order, as the draw functions would take them
// (a draw is a word >> 1): Philox words of the batch, or, computed ahead into buf, the
// reference's additive generator x[n] = x[n - 31] + x[n - 3].  Nothing is consumed.
struct RngWords {
    const uint32_t *w;
    int avail;
};

// `blocks`: 31-word blocks of the additive generator.  A block is three sums in steps of
// three: lanes 16 c + t hold word 3 t + c, and a scan over the 16 lanes of a row adds them
// up -- four adds for 31 words, which cost ~100 cycles each drawn one by one.
__device__ __forceinline__ RngWords rng_words(WaveRng &g, uint32_t *buf, int blocks)
{
    if (g.mode == CHROMO_RNG_PHILOX) {
        g.pidx = uni_i32(g.pidx);
        // near the batch's end: the batch again from the current block on
        if (g.pidx > 4 * WAVE - 128) {
            philox_fill(g, g.pbase + (uint64_t)(g.pidx >> 2));
            g.pidx &= 3;
        }
        return RngWords{g.mt + g.pidx, 4 * WAVE - g.pidx};
    }
    const int lane = lane_id();
    wave_sync();
    if (lane < 31) {
        const int i = lane - g.gf;
        buf[i < 0 ? i + 31 : i] = g.g;
    }
    wave_sync();
    const int c = lane >> 4, t = lane & 15, i = 3 * t + c;
    const bool in = c < 3 && i < 31;
    for (int b = 0; b < blocks; ++b) {
        const uint32_t *s = buf + 31 * b;
        int x = in ? (int)(s[i] + (t == 0 ? s[28 + c] : 0u)) : 0;
        x += dpp_i32<DPP_SHR1>(x);
        x += dpp_i32<DPP_SHR2>(x);
        x += dpp_i32<DPP_SHR4>(x);
        x += dpp_i32<DPP_SHR8>(x);
        if (in) buf[31 * (b + 1) + i] = (uint32_t)x;
        wave_sync();
    }
    return RngWords{buf + 31, 31 * blocks};
}

// The stream's checkpoint m words on (rng_save's form, of the words in v).
__device__ __forceinline__ void rng_mark(const WaveRng &g, const RngWords &v, int m, uint32_t *ck)
{
    const int lane = lane_id();
    if (g.mode == CHROMO_RNG_PHILOX) {
        WaveRng q = g;
        q.pidx = g.pidx + m;
        uint64_t ctr;
        int bi;
        philox_pos(q, ctr, bi);
        if (lane == 0) {
            ck[33] = (uint32_t)ctr;
            ck[34] = (uint32_t)(ctr >> 32);
            ck[39] = (uint32_t)bi;
        }
        return;
    }
    const int gf = (g.gf + m) % 31, i = lane - gf;
    if (lane < 31) ck[lane] = v.w[m - 31 + (i < 0 ? i + 31 : i)];
    if (lane == 0) {
        ck[31] = (uint32_t)gf;
        ck[32] = (uint32_t)((g.gr + m) % 31);
    }
}

// Consumes m of the words in v.
__device__ __forceinline__ void rng_take(WaveRng &g, const RngWords &v, int m)
{
    if (g.mode == CHROMO_RNG_PHILOX) {
        g.pidx += m;
        return;
    }
    const int lane = lane_id();
    g.gf = (g.gf + m) % 31;
    g.gr = (g.gr + m) % 31;
    const int i = lane - g.gf;
    if (lane < 31) g.g = v.w[m - 31 + (i < 0 ? i + 31 : i)];
}

// The usual proposals of controller C, drawn into the ring from slot number at on: up to
// `room` crank-shafts, end pivots or slides at once, one per lane, or one tangent rotation
// or binding move, its beads one per lane.  The same words, in the same order and with
// the same arithmetic, as gen_slot's draw-at-a-time code.  Returns the slots drawn; none,
// and nothing consumed, where the first proposal is not a usual one (a capped
// exponential drawn again, a bead picked twice, extra axis draws, a window that a slot
// does not hold, MT19937 to be regenerated): gen_slot then draws it one word at a time.
// Drawn one by one a slot cost the drawing wavefront about 5,000 cycles, most of them
// the latency of the exponential's logarithm and of one draw after the other.
template <int NB, int RING>
__device__ __forceinline__ int gen_batch(const chromo_replica *R, WaveRng &rng, const chromo_ctrl &C, SpecSlot *ring,
                                         uint32_t at, int room, uint32_t *buf)
{
    const int lane = lane_id();
    const int mv = uni_i32(C.move);
    const int64_t N = R->N;
    const double amp_move = C.amp_move;
    const int64_t amp_bead = C.amp_bead;
    const RngWords v = rng_words(rng, buf, mv == CHROMO_TANGENT_ROTATION ? GLIBC_BLOCKS : 1);
    if (mv == CHROMO_CRANK_SHAFT || mv == CHROMO_END_PIVOT || mv == CHROMO_SLIDE) {
        const int used = mv == CHROMO_CRANK_SHAFT ? 5 : (mv == CHROMO_END_PIVOT ? 6 : 7);
        const int most = v.avail / used < room ? v.avail / used : room;
        const bool in = lane < most;
        int32_t d[7];
#pragma unroll
        for (int t = 0; t < 7; ++t) d[t] = (int32_t)(v.w[in && t < used ? used * lane + t : 0] >> 1);
        bool ok = in;
        int64_t ind0 = 0, indf = 0;
        double ang = 0;
        int32_t s1 = 0, s2 = 0, lhs = 0, ud = 0;
        if (mv == CHROMO_CRANK_SHAFT) {
            ang = amp_move * (((double)d[0] / RMAX) - 0.5);
            const int64_t b0 = (int64_t)(int32_t)(((double)d[1] / RMAX) * (double)N);
            const int64_t b1 = imax64(from_point_once(d[2], d[3], amp_bead, N, b0, ok), 1);
            check_bead_bounds(b0, b1, N, ind0, indf);
            ud = d[4];
        } else if (mv == CHROMO_END_PIVOT) {
            ang = amp_move * (((double)d[0] / RMAX) - 0.5);
            lhs = (int32_t)(d[1] & 1);
            if (amp_bead > N) ok = false;
            const int64_t r = cexp_once(d[2], amp_bead, amp_bead, ok);
            ind0 = lhs == 1 ? 0 : N - r;
            indf = lhs == 1 ? r + 1 : N;
            if (indf > N) ok = false;
            s1 = d[3];
            s2 = d[4];
            ud = d[5];
        } else {
            ang = amp_move * ((double)d[0] / RMAX);
            s1 = d[1];
            s2 = d[2];
            const int64_t b0 = draw_mod(d[3], N);
            const int64_t b1 = from_point_once(d[4], d[5], amp_bead, N, b0, ok);
            check_bead_bounds(b0, b1, N, ind0, indf);
            ud = d[6];
        }
        const int64_t n = indf - ind0;
        ok = ok && n >= 1 && slot_holds(R, n);
        const int cnt = (int)__builtin_ctzll(~__ballot(ok));   // the leading usual ones
        if (lane < cnt) {
            SpecSlot &S = ring[(at + (uint32_t)lane) & (RING - 1)];
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
        for (int j = 0; j < cnt; ++j) rng_mark(rng, v, used * j, ring[(at + (uint32_t)j) & (RING - 1)].ck);
        rng_take(rng, v, used * cnt);
        wave_sync();
        return cnt;
    }
    SpecSlot &S = ring[at & (RING - 1)];
    int64_t n = 0, ind0 = 0, indf = 0;
    double ang = 0;
    int binder = 0, used = 0;
    int32_t ud = 0;
    if (mv == CHROMO_TANGENT_ROTATION) {
        ang = amp_move * (((double)(int32_t)(uni_u32(v.w[0]) >> 1) / RMAX) - 0.5);
        n = draw_mod((int32_t)(uni_u32(v.w[1]) >> 1), amp_bead) + 1;
        if (n > N || n > SPEC_NMAX || 3 + 3 * n > v.avail) return 0;
        const int k = uni_i32((int)n);
        const bool act = lane < k;
        const int c = (int)draw_mod((int32_t)(v.w[2 + (act ? lane : 0)] >> 1), N);
        bool twice = false;
        for (int j = 0; j + 1 < k; ++j) twice |= act && lane > j && c == (int)readlane_u32((uint32_t)c, j);
        if (wave_any(twice)) return 0;
        if (act) {
            S.picks[lane] = c;
            S.ps1[lane] = (int32_t)(v.w[2 + k + 2 * lane] >> 1);
            S.ps2[lane] = (int32_t)(v.w[3 + k + 2 * lane] >> 1);
        }
        ud = (int32_t)(uni_u32(v.w[2 + 3 * k]) >> 1);
        used = 3 + 3 * k;
    } else {
        binder = (int)((uni_u32(v.w[0]) >> 1) % (uint32_t)NB);
        const uint32_t top = (uint32_t)R->sites[binder];
        const int64_t b0 = draw_mod((int32_t)(uni_u32(v.w[1]) >> 1), N);
        bool ok = true;
        const int64_t b1 = from_point_once((int32_t)(uni_u32(v.w[2]) >> 1), (int32_t)(uni_u32(v.w[3]) >> 1), amp_bead,
                                           N, b0, ok);
        check_bead_bounds(b0, b1, N, ind0, indf);
        n = indf - ind0;
        if (!wave_any(ok) || n < 1 || n > SPEC_NMAX) return 0;
        // the new states: masked rejection (rnd_randint), 64 words looked at at once
        used = 4;
        if (top == 0) {
            if (lane < n) S.newst[lane] = 0;
        } else {
            uint32_t mask = top;
            mask |= mask >> 1;
            mask |= mask >> 2;
            mask |= mask >> 4;
            mask |= mask >> 8;
            mask |= mask >> 16;
            const bool mt = rng.mode == CHROMO_RNG_GLIBC;
            const int have = mt ? 624 - uni_i32(rng.mti) : v.avail - 4;
            uint32_t y = 0;
            if (lane < have) y = mt ? mt_temper(rng.mt[rng.mti + lane]) : v.w[4 + lane];
            y &= mask;
            const uint64_t m = __ballot(lane < have && y <= top);
            const int rank = __popcll(m & ((1ull << lane) - 1));
            const bool mine = (m >> lane & 1) && rank < n;
            const uint64_t last = __ballot(mine && rank == n - 1);
            if (last == 0) return 0;
            const int words = (int)__builtin_ctzll(last) + 1;
            if (!mt) {
                used += words;
                if (used >= v.avail) return 0;
            }
            if (mine) S.newst[rank] = (int32_t)y;
            if (mt) rng.mti = uni_i32(rng.mti) + words;
        }
        ud = (int32_t)(uni_u32(v.w[used]) >> 1);
        used += 1;
    }
    rng_mark(rng, v, 0, S.ck);
    if (lane == 0) {
        S.kind = SLOT_SMALL;
        S.move = mv;
        S.binder = binder;
        S.lhs = 0;
        S.ud = ud;
        S.s1 = 0;
        S.s2 = 0;
        S.n = n;
        S.ind0 = ind0;
        S.indf = indf;
        S.ang = ang;
    }
    rng_take(rng, v, used);
    wave_sync();
    return 1;
}

// Draws one proposal into slot S (the drawing wavefront), in the draw order of
// mc_step_dev.  A proposal that is too large for one wavefront, or that fails,
// is marked SLOT_SEQ with its draws given back: mc_step_dev redoes it.
template <int NB>
__device__ __forceinline__ int gen_slot(const chromo_replica *R, WaveRng &rng, const chromo_ctrl &C, SpecSlot &S)
{
    const int lane = lane_id();
    const int64_t N = R->N;
    rng_save(rng, S.ck);
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
                S.picks[lane] = (int32_t)fpick;
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
            if (lane < k) S.picks[lane] = (int32_t)mine;
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
    rng.g = 0;
    rng.gf = rng.gr = 0;
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
    const EvLds S = ev_lds(blocks, NB + 1, 0);
    ev_clear(S);
    EvBeads<NB> B;
    if (go) mc_evaluate<NB, TW>(R, EC, C, o, P, u, S, B, false);
    constexpr int U = Shape<W>::ucap(NB + 1);
    const size_t bytes = ev_layout(NB + 1, U).total;
    for (int b = 0; b < Shape<W>::EV; ++b) ev_clear(ev_lds(blocks + bytes * b, NB + 1, U));
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

// mc_step_dev with the usual proposals drawn at once into slot S (gen_batch), so that the
// loads of the window's beads go out before the proposal's arithmetic and the axis and
// fulcrum beads come with them; the others as mc_step_dev draws them.  buf: GLIBC_BUF
// words of LDS.  One launch per proposal, 161 in a row on
// 100,000 beads: 2.24 ms without it, 2.12 with it.
template <int NB, bool TW>
__device__ __forceinline__ void mc_step_slot(const chromo_replica *R, const EvConst &EC, WaveRng &rng, chromo_ctrl &C,
                                             MoveOut &out, const EvLds &L, SpecSlot &S, uint32_t *buf)
{
    const int lane = lane_id();
    Proposal P;
    EvBeads<NB> B;
    double u = 0;
    bool go = false;
    if (gen_batch<NB, 1>(R, rng, C, &S, 0, 1, buf) == 1) {
        const bool tangent = S.move == CHROMO_TANGENT_ROTATION;
        ev_load<NB, TW>(R, S.move, S.n, S.ind0, S.indf, 0, tangent && (lane & 31) < S.n ? S.picks[lane & 31] : 0, B);
        go = slot_proposal<NB>(R, S, P, B);
        if (go) {
            u = (double)S.ud / RMAX;
            out.err = 0;
            out.n = S.n;
            out.ind0 = tangent ? S.picks[0] : S.ind0;
            out.indf = tangent ? S.picks[0] + 1 : S.indf;
            C.num_attempt += 1;
        } else {
            rng_restore(rng, S.ck);
        }
    }
    const bool loaded = go;
    if (!go) go = mc_propose<NB>(R, rng, C, out, P, u);
    if (go) mc_evaluate<NB, TW>(R, EC, C, out, P, u, L, B, loaded);
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

// Whether slot S (result s, its voxels in the hash of block G) reads what the accepted
// slot Q (result a, its voxels in list) wrote.  Beads: a window reads its beads and one
// on either side, a tangent rotation its picks and their neighbours; a window writes its
// beads, a tangent rotation its picks (tangents only, which binding moves do not read).
// Voxels: Q's are looked up in S's hash.
__device__ __forceinline__ bool spec_conflict(const SpecSlot &S, const SpecRes &s, const EvLds &G, const SpecSlot &Q,
                                              const SpecRes &a, const int2 *list)
{
    const int lane = lane_id();
    const bool st = S.move == CHROMO_TANGENT_ROTATION, qt = Q.move == CHROMO_TANGENT_ROTATION;
    bool hit = false;
    if (st) {
        if (lane < S.n) {
            const int64_t mine = S.picks[lane];
            if (qt) {
                for (int q = 0; q < (int)Q.n; ++q) {
                    const int64_t d = Q.picks[q] - mine;
                    hit |= d >= -1 && d <= 1;
                }
            } else {
                hit = mine >= a.wlo - 1 && mine <= a.whi;
            }
        }
    } else if (qt) {
        if (lane < Q.n) hit = Q.picks[lane] >= s.rlo && Q.picks[lane] <= s.rhi;
    } else {
        hit = a.wlo <= s.rhi && s.rlo < a.whi;
        if (s.nbins > 0)
            for (int q = lane; q < a.nbins; q += WAVE) {
                const int2 v = list[q];
                int h = (int)((uint32_t)v.y >> 16);
                for (int probes = 0; probes < G.hsize; ++probes) {
                    const int key = G.hkey[h];
                    hit |= key == v.x;
                    if (key == v.x || key == HKEY_EMPTY) break;
                    h = (h + 1) & (G.hsize - 1);
                }
            }
    }
    return wave_any(hit);
}

// One wavefront: AcceptanceTracker updates (mc_stat.py:190-208), controller counts,
// replica counters and log records of the F resolved slots from number s0 on, one slot
// per lane; the same totals as record() called once per slot in order.
template <int RING>
__device__ __forceinline__ void spec_book(const chromo_replica *R, chromo_ctrl &C, Counters &K,
                                          const SpecSlot *ring, const SpecRes *res, uint32_t s0, int F)
{
    const int lane = lane_id();
    const int at_ring = (int)((s0 + (uint32_t)(lane < F ? lane : 0)) & (RING - 1));
    const SpecSlot &S = ring[at_ring];
    const SpecRes &q = res[at_ring];
    const bool live = lane < F && S.kind != SLOT_EMPTY;
    int64_t n = 0, nb = 0, bytes = 0;
    int acc = 0, tie = 0;
    if (live) {
        n = S.n;
        nb = q.nbins;
        acc = q.accepted;
        tie = fabs(q.u - q.expdE) < 1E-12;
        bytes = move_bytes(S.move, n, nb, R->B, acc);
    }
    const uint64_t live_m = __ballot(live);
    const uint64_t acc_m = __ballot(live && acc);
    const uint64_t tie_m = __ballot(live && tie);
    // sums over the first eight lanes
    const int64_t sn = sum_lanes8_i64(n), sb = sum_lanes8_i64(nb), sy = sum_lanes8_i64(bytes);
    const int64_t logged = K.logged;
    const int nlive = __popcll(live_m);
    if (R->log != nullptr && live) {
        const int64_t at = logged + __popcll(live_m & ((1ull << lane) - 1));
        if (at < R->log_cap) {
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

// Words of SpecCtl: what a wavefront wrote before it sets one is visible to who reads
// it there.
template <typename T>
__device__ __forceinline__ void ctl_set(T *f, T v)
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    if (lane_id() == 0) __hip_atomic_store(f, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

template <typename T>
__device__ __forceinline__ T ctl_get(const T *f)
{
    const T v = (T)uni_i32((int)__hip_atomic_load(f, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP));
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    return v;
}

// All of SpecCtl in one LDS read (its words share a read of 16 lanes, so they are of one
// moment), as scalars.
struct CtlNow {
    uint32_t drawn, resolved;
    int back, alone, over;    // over: stop or err
};
__device__ __forceinline__ CtlNow ctl_look(const SpecCtl *ctl)
{
    const uint32_t w = __hip_atomic_load((const uint32_t *)ctl + (lane_id() & (CTL_WORDS - 1)), __ATOMIC_RELAXED,
                                         __HIP_MEMORY_SCOPE_WORKGROUP);
    CtlNow c;
    c.drawn = readlane_u32(w, (int)offsetof(SpecCtl, drawn) / 4);
    c.resolved = readlane_u32(w, (int)offsetof(SpecCtl, resolved) / 4);
    c.back = (int)readlane_u32(w, (int)offsetof(SpecCtl, back) / 4);
    c.alone = (int)readlane_u32(w, (int)offsetof(SpecCtl, alone) / 4);
    c.over = (int)(readlane_u32(w, (int)offsetof(SpecCtl, stop) / 4) | readlane_u32(w, (int)offsetof(SpecCtl, err) / 4));
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    return c;
}

// A wait's next look: false (and the replica's error) once it passed its bound.
__device__ __forceinline__ bool spin_on(SpecCtl *ctl, int &spins)
{
    __builtin_amdgcn_s_sleep(1);
    if (++spins < SPIN_LIMIT) return true;
    ctl_set(&ctl->err, (int32_t)ERR_SPIN);
    return false;
}

// A controller block of the launch: controller ci in step `step`, slots start .. start + n - 1.
struct SpecBlock {
    int64_t step;
    int ci;
    uint32_t start;
    int n;
};

// What the drawing wavefront keeps.
struct SpecGen {
    WaveRng rng;
    SpecBlock book, draw;       // the block being booked; the one being drawn: that one or the next
    uint32_t drawn, booked;
    int list;                   // voxel list of the last slot drawn
    int64_t steps;
    int nc;
};

// Moves b to the next controller that makes proposals; step = steps when there is none.
__device__ __forceinline__ void block_next(SpecBlock &b, const chromo_ctrl *sctrl, int nc, int64_t steps)
{
    const uint32_t start = b.start + (uint32_t)b.n;
    b.start = start;
    b.n = 0;
    while (b.step < steps) {
        if (++b.ci >= nc) {
            b.ci = 0;
            if (++b.step >= steps) break;
        }
        if (sctrl[b.ci].on == 1 && sctrl[b.ci].num_per_cycle > 0) {
            b.n = uni_i32(sctrl[b.ci].num_per_cycle);
            break;
        }
    }
}

// The booked slots end a block: the amplitudes of its controller, and of the controllers
// without proposals that follow, are updated.
__device__ __forceinline__ void block_done(SpecGen &g, chromo_ctrl *sctrl)
{
    const int c0 = g.book.ci;
    const int64_t s0 = g.book.step;
    const bool same = g.draw.step == s0 && g.draw.ci == c0;
    block_next(g.book, sctrl, g.nc, g.steps);
    wave_sync();
    if (lane_id() == 0) {
        int64_t s = s0;
        int c = c0;
        while (s < g.book.step || (s == g.book.step && c < g.book.ci)) {
            if (s >= g.steps) break;
            update_amplitudes_dev(sctrl[c]);
            if (++c >= g.nc) {
                c = 0;
                ++s;
            }
        }
    }
    wave_sync();
    if (same) g.draw = g.book;
}

// Books the slots before number r.
template <int RING>
__device__ __forceinline__ void book_to(const chromo_replica *R, SpecGen &g, chromo_ctrl *sctrl, Counters &K,
                                        const SpecLds &L, uint32_t r)
{
    while (g.booked != r) {
        const int left = g.book.n - (int)(g.booked - g.book.start), have = (int)(r - g.booked);
        const int n = have < left ? have : left, F = n < 8 ? n : 8;
        spec_book<RING>(R, sctrl[g.book.ci], K, L.ring, L.res, g.booked, F);
        g.booked += (uint32_t)F;
        if (F == left) block_done(g, sctrl);
    }
}

// The drawing wavefront's work that is at hand: draws further slots, books the resolved
// ones, runs the first unresolved slot one at a time where that is needed (alone: only
// while this wavefront holds nothing in a block).  True when there was something to do.
template <int NB, int W, bool TW>
__device__ __forceinline__ bool spec_serve(const chromo_replica *R, const EvConst &EC, SpecGen &g, chromo_ctrl *sctrl,
                                           Counters &K, const SpecLds &L, bool alone)
{
    using SH = Shape<W>;
    constexpr int RING = SH::RING;
    SpecCtl *ctl = L.ctl;
    const int lane = lane_id();
    bool did = false;
    if (g.book.step >= g.steps) {
        ctl_set(&ctl->stop, 1);
        return true;
    }
    const uint32_t r = ctl_get(&ctl->resolved);
    // (a slot given back after r was read is a later one: left to the next call)
    if (r != g.drawn &&
        (L.ring[r & (RING - 1)].kind == SLOT_SEQ || (ctl_get(&ctl->back) && ctl_get(&ctl->back_at) == r))) {
        if (!alone) return false;
        book_to<RING>(R, g, sctrl, K, L, r);
        // what was drawn after slot r is dropped, and drawn again after it: the wavefronts
        // that evaluate it fall back to waiting for it
        if (g.drawn != r + 1) {
            g.drawn = r + 1;
            g.draw = g.book;
            g.list = uni_i32(L.ring[r & (RING - 1)].list);
            ctl_set(&ctl->drawn, g.drawn);
        }
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
        for (int w = 0; w < SH::EV; ++w)
            if (!ctl_get(&ctl->idle[w])) return false;
        SeqIO *io = L.seq;
        const SpecSlot &S0 = L.ring[r & (RING - 1)];
        chromo_ctrl &C = sctrl[g.book.ci];
        for (int i = lane; i < CK_WORDS; i += WAVE) io->ck[i] = S0.ck[i];
        if (lane == 0) {
            io->mti = g.rng.mti;
            io->C = C;
        }
        wave_sync();
        ctl_set(&ctl->alone, 1);
        seq_step<NB, W, TW>(R, EC, io, L.mt, L.blocks);
        rng_restore(g.rng, io->ck);
        g.rng.mti = uni_i32(io->mti);
        if (lane == 0) C = io->C;
        wave_sync();
        const MoveOut o = io->out;
        if (o.err) {
            ctl_set(&ctl->err, (int32_t)o.err);
            return true;
        }
        if (o.n > 0) record(R, C, o, K);
        wave_sync_global();
        g.booked = r + 1;
        // in this order: who holds number r goes on before anything may start again
        ctl_set(&ctl->resolved, r + 1);
        ctl_set(&ctl->back, 0);
        ctl_set(&ctl->alone, 0);
        if (g.booked - g.book.start == (uint32_t)g.book.n) block_done(g, sctrl);
        return true;
    }
    // nothing is drawn past a SLOT_SEQ slot
    bool more = g.drawn == r || L.ring[(g.drawn - 1) & (RING - 1)].kind != SLOT_SEQ;
    const uint32_t room_to = (int)(g.booked + RING - (r + SH::AHEAD)) < 0 ? g.booked + RING : r + SH::AHEAD;
    while (more && (int)(room_to - g.drawn) > 0) {
        if (g.drawn - g.draw.start == (uint32_t)g.draw.n) {
            // the next block, one ahead of the booked one, unless its controller's
            // amplitudes still depend on that one
            if (g.draw.start != g.book.start) break;
            SpecBlock b = g.draw;
            block_next(b, sctrl, g.nc, g.steps);
            if (b.step >= g.steps || b.ci == g.book.ci) break;
            g.draw = b;
        }
        const chromo_ctrl &C = sctrl[g.draw.ci];
        // MT19937 is not rewound: no binding slot is drawn behind one that may be given back
        if (g.rng.mode == CHROMO_RNG_GLIBC && C.move == CHROMO_CHANGE_BINDING_STATE && (int)(r - g.draw.start) < 0) break;
        const int left = g.draw.n - (int)(g.drawn - g.draw.start), room = (int)(room_to - g.drawn);
        int cnt = gen_batch<NB, RING>(R, g.rng, C, L.ring, g.drawn, left < room ? left : room, L.seq->words);
        if (cnt == 0) {
            more = gen_slot<NB>(R, g.rng, C, L.ring[g.drawn & (RING - 1)]) != SLOT_SEQ;
            cnt = 1;
        }
        for (int j = 0; j < cnt; ++j) {
            g.list = g.list + 1 == SH::LISTS ? 0 : g.list + 1;
            if (lane == 0) L.ring[(g.drawn + (uint32_t)j) & (RING - 1)].list = g.list;
        }
        g.drawn += (uint32_t)cnt;
        ctl_set(&ctl->drawn, g.drawn);
        did = true;
    }
    // several at a time, the last ones of a block at once: the block after the next waits
    // for them
    const int waiting = (int)(r - g.booked);
    if (waiting > 0 && (!did || waiting >= RING / 4 || (int)(r - (g.book.start + (uint32_t)g.book.n)) >= 0)) {
        book_to<RING>(R, g, sctrl, K, L, r);
        did = true;
    }
    return did;
}

template <int NB, int W, bool TW>
__device__ __forceinline__ void spec_run(const chromo_replica *R, const EvConst &EC, int64_t steps)
{
    using SH = Shape<W>;
    constexpr int Bp1 = NB + 1, RING = SH::RING, EV = SH::EV, U = SH::ucap(Bp1);
    static_assert((RING & (RING - 1)) == 0 && RING > SH::AHEAD, "ring positions wrap by mask");
    static_assert(U * Bp1 * 8 < 65536, "byte offsets of the deltas fit 16 bits");
    const SpecLayout SL = spec_layout<W>(Bp1);
    const int wv = wave_id(), lane = lane_id();
    SpecLds L;
    L.blocks = lds_dyn;
    L.lists = (int2 *)(lds_dyn + SL.lists);
    L.ring = (SpecSlot *)(lds_dyn + SL.slots);
    L.res = (SpecRes *)(lds_dyn + SL.res);
    L.ctl = (SpecCtl *)(lds_dyn + SL.ctl);
    L.seq = (SeqIO *)(lds_dyn + SL.seq);
    L.mt = (uint32_t *)(lds_dyn + SL.mt);
    EvLds G = ev_lds(L.blocks + SL.seg_bytes * (wv < EV ? wv : 0), Bp1, U);
    if (wv < EV) ev_clear(G);
    __shared__ chromo_ctrl sctrl[MAX_CTRL];
    __shared__ Counters sK;
    SpecCtl *ctl = L.ctl;
    const bool gen = wv == SH::GEN;
    constexpr bool DRAWS = SH::GEN < EV;   // an evaluating wavefront draws
    bool need_mt = false;
    SpecGen g;
    g.rng.mode = uni_i32(R->rng_mode);
    g.nc = R->n_ctrl < MAX_CTRL ? R->n_ctrl : MAX_CTRL;
    g.steps = steps;
    g.drawn = g.booked = 0;
    g.list = SH::LISTS - 1;
    if (gen) {
        need_mt = any_binding(R);
        rng_load(R, g.rng, L.mt, need_mt);
        if (lane == 0) {
            counters_load(R, sK);
            for (int i = 0; i < g.nc; ++i) sctrl[i] = R->ctrl[i];
            ctl->next = ctl->drawn = ctl->resolved = 0;
            ctl->back = ctl->alone = ctl->stop = ctl->err = 0;
            for (int w = 0; w < SPEC_EVMAX; ++w) ctl->idle[w] = 1;
        }
        wave_sync();
        // the controllers before the first with proposals are updated like the others
        g.book = SpecBlock{0, 0, 0, 0};
        if (g.nc < 1 || steps < 1) g.book.step = steps;
        else if (sctrl[0].on == 1 && sctrl[0].num_per_cycle > 0) g.book.n = uni_i32(sctrl[0].num_per_cycle);
        g.draw = g.book;
        if (g.book.step < steps && g.book.n == 0) block_done(g, sctrl);
    }
    __syncthreads();
    if (wv >= EV) {
        // draws and books only
        int spins = 0;
        while (!ctl_look(ctl).over) {
            if (spec_serve<NB, W, TW>(R, EC, g, sctrl, sK, L, true)) spins = 0;
            else if (!spin_on(ctl, spins)) break;
        }
    } else {
        uint32_t t = 0;
        bool have = false;   // holds number t
        for (;;) {
            // take a number, wait for its slot
            if (!have) {
                uint32_t v = 0;
                if (lane == 0) v = atomicAdd(&ctl->next, 1u);
                t = uni_u32(v);
                have = true;
            }
            SpecSlot &S = L.ring[t & (RING - 1)];
            bool go = false;
            uint32_t seen = 0;   // earlier slots up to here are committed or rejected
            for (int spins = 0;;) {
                const CtlNow c = ctl_look(ctl);
                if (c.over) break;
                if ((int)(c.resolved - t) > 0) {
                    have = false;   // it was run one at a time
                    break;
                }
                if ((int)(c.drawn - t) > 0 && !c.back && S.kind != SLOT_SEQ) {
                    // no longer idle, unless the slot was dropped meanwhile, or run one at
                    // a time between the looks (`back` falls after `resolved` rises)
                    ctl_set(&ctl->idle[wv], 0);
                    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
                    const CtlNow d = ctl_look(ctl);
                    if ((int)(d.drawn - t) > 0 && !d.back && (int)(d.resolved - t) <= 0) {
                        seen = d.resolved;
                        go = true;
                        break;
                    }
                    ctl_set(&ctl->idle[wv], 1);
                }
                if (DRAWS && gen) {
                    if (spec_serve<NB, W, TW>(R, EC, g, sctrl, sK, L, true)) {
                        spins = 0;
                        continue;
                    }
                }
                // a slot run one at a time may be of any length
                if (c.alone) spins = 0;
                if (!spin_on(ctl, spins)) break;
            }
            if (!have) continue;
            if (!go) break;
            SpecRes &res = L.res[t & (RING - 1)];
            G.uv = L.lists + U * uni_i32(S.list);
            EvKeep keep;
            Proposal P;
            int held = 0;
            bool turn = false, again = true;
            while (again) {
                again = false;
                ev_release(G, held);
                held = 0;
                if (S.kind == SLOT_SMALL) held = eval_slot<NB, TW>(R, EC, S, res, P, keep, G);
                for (int spins = 0;;) {
                    const CtlNow c = ctl_look(ctl);
                    if (c.over) break;
                    const uint32_t r = c.resolved;
                    bool hit = false;
                    for (; seen != r; ++seen) {
                        const SpecSlot &Q = L.ring[seen & (RING - 1)];
                        const SpecRes &q = L.res[seen & (RING - 1)];
                        if (!hit && S.kind == SLOT_SMALL && Q.kind == SLOT_SMALL && q.accepted)
                            hit = spec_conflict(S, res, G, Q, q, L.lists + U * uni_i32(Q.list));
                        spins = 0;
                    }
                    if (hit) {
                        again = true;
                        break;
                    }
                    if (r == t) {
                        turn = true;
                        break;
                    }
                    if ((int)(c.drawn - t) <= 0) break;   // dropped
                    if (DRAWS && gen) {
                        if (c.back) break;                // to be dropped, by this wavefront
                        if (spec_serve<NB, W, TW>(R, EC, g, sctrl, sK, L, false)) continue;
                    }
                    if (!spin_on(ctl, spins)) break;
                }
            }
            if (turn && S.kind == SLOT_SMALL && (res.resample || res.overflow)) {
                // an axis to be drawn again, or more voxels than the block holds
                if (lane == 0) ctl->back_at = t;
                ctl_set(&ctl->back, 1);
                turn = false;
            }
            if (turn) {
                if (S.kind == SLOT_SMALL && res.accepted) ev_commit<NB>(R, P, keep, G, held);
                ctl_set(&ctl->resolved, t + 1);
                have = false;
            }
            // whole, not by the slot's list: another slot may have that by now
            if (held) ev_clear(G);
            ctl_set(&ctl->idle[wv], 1);
        }
    }
    __syncthreads();
    if (gen) {
        // after a wait that passed its bound there may be committed slots left to book
        book_to<RING>(R, g, sctrl, sK, L, ctl->resolved);
        rng_store(R, g.rng, need_mt);
        if (lane == 0)
            for (int i = 0; i < g.nc; ++i) R->ctrl[i] = sctrl[i];
        counters_store(R, sK, ctl->err);
    }
}

}  // namespace
