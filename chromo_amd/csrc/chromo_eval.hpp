// chromo_eval.hpp -- evaluation of one proposal by one wavefront.
//
// The beads of a move go through in chunks of 32.  In a chunk lane i and lane
// 32 + i hold bead i: the lower half its current position, the upper half its trial
// one (chromo/fields.pyx:1434-1520 walks them as positions p = 2i + k), so every
// position has a lane of its own.  A position touches the 8 corners of its voxel
// cell: contribution e = 8p + l.
//
//  1. Each lane enters its 8 corner voxels into an LDS hash (all 8 compare-and-swaps
//     in flight at once).  The slot is a few low bits of the voxel's coordinates: the
//     voxels of one window lie together, so nearly all of them get a slot of their
//     own and probing is rare.
//  2. The contribution with the smallest e of each new voxel numbers it; numbers are
//     handed out corner by corner, lane by lane.
//  3. Fold: delta[voxel][species] lives in LDS.  One LDS floating-point add per
//     position, its lanes the position's corners times the species, issued in position
//     order: the LDS executes a wavefront's operations in order, so every voxel's
//     delta is the reference's left fold (fields.pyx:1491-1520, its 1e-18 rules
//     included) bit for bit, with no per-voxel lists, sorting or divergent loops.
//     (On a grid with a one-voxel axis corners of one position share a voxel: there
//     the corners are issued one after the other.)
//  4. Energy terms, one voxel per lane, in number order; one wave reduction in a fixed
//     order; Metropolis.
//
// The hash and the deltas last over the chunks of a move, so a move of any length is
// one evaluation as long as its voxels fit (EvLds::ucap); beyond that it overflows and
// the caller takes the global arena.  The evaluation's numbers do not depend on the
// block's capacity.
//
// What bounds it: one wavefront's chain of dependent LDS and HBM round trips.  Against
// per-voxel fold lists (hash, position masks, numbering, dealing by length, list
// building, divergent folds; moves above 32 beads one at a time): 512 replicas of
// 2,000-20,000 beads at steady-state windows, 20 sweeps, two wavefronts each,
// 50.4 -> 33.1 ms when it came in (30.2 to 30.9 ms now, with the slots of chromo_spec.hpp);
// 16 replicas with one wavefront each, 10 sweeps, 25.1 -> 20.2 ms.
#pragma once

#include "chromo_device.hpp"

namespace {

using namespace chromo;

constexpr int SEG_MAX = 32;       // beads of one chunk
constexpr int EV_LANES = 64;      // tangent picks or binding beads of one evaluation (one per lane)
constexpr int EV_POS = 2 * SEG_MAX;
constexpr int EV_WAVES = 4;       // wavefronts of a workgroup, at most
constexpr int EV_FREE = 0x7fffffff;             // hash value: no contribution yet
constexpr int EV_NUM = (int)0x80000000;         // hash value of voxel number q: EV_NUM + q

// Voxels a block holds.  The one-at-a-time block (hash of 2048): three workgroups on a
// compute unit.  A speculative evaluator's block (hash of 1024, the voxel list kept
// apart from it) takes what its workgroup's shape leaves it.
__host__ __device__ inline int ev_wide_ucap(int Bp1) { return Bp1 <= 2 ? 1024 : (Bp1 == 3 ? 896 : (Bp1 == 4 ? 704 : 576)); }
static_assert(1024 * 2 * 8 < 65536 && 896 * 3 * 8 < 65536 && 704 * 4 * 8 < 65536 && 576 * 5 * 8 < 65536,
              "byte offsets of the deltas fit 16 bits");

struct EvLayout {
    size_t c0, eq, pst, ends, tmat, hkey, hval, uv, acc, total;
};

// slot_ucap: voxels of a speculative evaluator's block, 0 for the one-at-a-time block.
__host__ __device__ inline EvLayout ev_layout(int Bp1, int slot_ucap)
{
    const bool wide = slot_ucap == 0;
    const size_t H = wide ? 2048 : 1024, U = (size_t)(wide ? ev_wide_ucap(Bp1) : slot_ucap);
    EvLayout L;
    size_t o = 0;
    L.c0 = o;   o += sizeof(double) * 8 * EV_POS;      // corner weight / volume per contribution
    L.eq = o;   o += sizeof(uint16_t) * 8 * EV_POS;    // byte offset of its voxel's deltas
    L.ends = o; o += sizeof(double) * 2 * 2 * 9;       // end beads: [first / last][current / trial][r, t3, t2]
    L.tmat = o; o += sizeof(double) * 12;              // the proposal's transform, for the commit
    L.pst = o;  o += sizeof(uint64_t) * EV_POS;        // weight factors per position: 1, then the binder states
    L.uv = o;   o += wide ? sizeof(int2) * U : 0;      // voxel, its hash slot | its first probe << 16
    L.acc = o;  o += sizeof(double) * U * Bp1;         // delta densities, then new densities
    L.hkey = o; o += sizeof(int32_t) * H;              // voxel
    L.hval = o; o += sizeof(int32_t) * H;              // smallest contribution, then number
    L.total = (o + 255) / 256 * 256;
    return L;
}

struct EvLds {
    double *c0, *ends, *tmat, *acc;
    uint16_t *eq;
    uint8_t *pst;       // factor m of position p at 8 p + m
    int32_t *hkey, *hval;
    int2 *uv;
    int hsize, ymask, zshift, ucap;
};

// A speculative evaluator sets uv to the list of the slot it evaluates.
__device__ __forceinline__ EvLds ev_lds(char *base, int Bp1, int slot_ucap)
{
    const bool wide = slot_ucap == 0;
    const EvLayout L = ev_layout(Bp1, slot_ucap);
    EvLds S;
    S.c0 = (double *)(base + L.c0);
    S.eq = (uint16_t *)(base + L.eq);
    S.ends = (double *)(base + L.ends);
    S.tmat = (double *)(base + L.tmat);
    S.pst = (uint8_t *)(base + L.pst);
    S.uv = (int2 *)(base + L.uv);
    S.acc = (double *)(base + L.acc);
    S.hkey = (int32_t *)(base + L.hkey);
    S.hval = (int32_t *)(base + L.hval);
    S.hsize = wide ? 2048 : 1024;
    S.ymask = wide ? 15 : 7;
    S.zshift = wide ? 8 : 7;
    S.ucap = wide ? ev_wide_ucap(Bp1) : slot_ucap;
    return S;
}

// Empties the hash.  One wavefront.
__device__ __forceinline__ void ev_clear(const EvLds &S)
{
    for (int i = 4 * lane_id(); i < S.hsize; i += 4 * WAVE) {
        *(int4 *)&S.hkey[i] = make_int4(HKEY_EMPTY, HKEY_EMPTY, HKEY_EMPTY, HKEY_EMPTY);
        *(int4 *)&S.hval[i] = make_int4(EV_FREE, EV_FREE, EV_FREE, EV_FREE);
    }
    wave_sync();
}

// Empties the hash slots of an evaluation's U voxels.
__device__ __forceinline__ void ev_release(const EvLds &S, int U)
{
    for (int q = lane_id(); q < U; q += WAVE) {
        const int h = S.uv[q].y & 0xffff;
        S.hkey[h] = HKEY_EMPTY;
        S.hval[h] = EV_FREE;
    }
    wave_sync();
}

// ---- per-launch constants -----------------------------------------------------

// Grid constants with the reciprocals the exact divisions below use, worked out once
// per launch and kept in LDS.
enum : int { EC_WIDTH = 0, EC_D = 3, EC_SUB = 6, EC_NSUB = 9, EC_LEN = 12 };
struct EvConst {
    double len[EC_LEN], rec[EC_LEN];  // per axis: box width, voxel size, sub-bin width, sub-bins; their reciprocals
    double hw[3], hs[3], half_points;
    double vol, rvol, vbV, cphi;      // vol_bin, its reciprocal, vol_bin / bead_vol, chi (vol_bin / bead_vol)
    int32_t n[3], fast, recip, cross;
};

// Fills the constants; the first wavefront of the workgroup, the caller synchronises.
// One division per lane, so the launch waits for one: in three lanes of four divisions
// each they took 0.4 us of a launch that evaluates one proposal.
__device__ __forceinline__ void ev_const(EvConst *C, const chromo_replica *R)
{
    const int t = (int)threadIdx.x;
    if (t >= WAVE) return;
    const bool axis = t < EC_LEN;
    const int j = t % 3;
    const double *const row = t < EC_D ? R->width : (t < EC_SUB ? R->dxyz : R->sub_width);
    double den = R->vol_bin;
    if (axis) den = t < EC_NSUB ? row[j] : (double)R->n_sub[j];
    if (t == EC_LEN + 1) den = R->bead_vol;
    const double q = (t == EC_LEN + 1 ? R->vol_bin : 1.0) / den;
    if (axis) {
        C->len[t] = den;
        C->rec[t] = q;
    } else if (t == EC_LEN) {
        C->vol = den;
        C->rvol = q;
        C->half_points = R->half_points;
        C->fast = R->fast_field;
    } else if (t == EC_LEN + 1) {
        C->vbV = q;
        C->cphi = R->chi * q;
    }
    if (t < 3) {
        C->hw[t] = R->half_width[t];
        C->hs[t] = R->half_step[t];
        C->n[t] = (int32_t)(t == 0 ? R->nx : (t == 1 ? R->ny : R->nz));
    }
    const bool used = t < EC_SUB || (t < EC_NSUB && R->fast_field) || t == EC_LEN;
    const bool out = wave_any(used && !recip_range(den));
    const bool x = wave_any(t < R->B * R->B && R->cross[t] != 0);
    if (t == 0) {
        C->recip = !out;
        C->cross = x;
    }
}

// Lower voxel indices and lower-corner weights of one position: voxel_lower's values
// (chromo_device.hpp), the three axes as independent straight-line chains.
__device__ __forceinline__ void ev_lower(const chromo_replica *R, const EvConst &C, const double *pos, int ix[3],
                                         double w[3], int &ties)
{
    bool far = C.recip == 0;
    double a[3];
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        a[j] = pos[j] + C.hw[j];
        far = far || !(fabs(a[j]) < 0x1p40 * C.len[(C.fast ? EC_SUB : EC_WIDTH) + j]);
    }
    if (wave_any(far)) {
        // a coordinate far outside the box, or a grid of extreme size: the general path
        int64_t i64[3];
        voxel_lower(R, pos, i64, w, ties);
#pragma unroll
        for (int j = 0; j < 3; ++j) ix[j] = (int)i64[j];
        return;
    }
    if (C.fast) {
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            const double qs = div_by(a[j], C.len[EC_SUB + j], C.rec[EC_SUB + j]);
            const double sb = floor(qs);
            ties += fabs(qs - rint(qs)) < TIE_VOXEL_EPS;
            // sb mod n_sub, whole numbers below 2^41: exact
            double i = fma(-floor(sb * C.rec[EC_NSUB + j]), C.len[EC_NSUB + j], sb);
            if (i < 0) i += C.len[EC_NSUB + j];
            if (i >= C.len[EC_NSUB + j]) i -= C.len[EC_NSUB + j];
            const double u = div_by((i - C.half_points) * C.len[EC_SUB + j], C.len[EC_D + j], C.rec[EC_D + j]);
            const double ind = floor(u);
            ix[j] = (ind == -1.0) ? C.n[j] - 1 : (int)ind;
            w[j] = 1 - (u - ind);
        }
        return;
    }
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        // Python's a % W: the quotient from the reciprocal is off by at most one, which
        // the first remainder's sign and range show; the second is exact (fmod_exact)
        const double W = C.len[EC_WIDTH + j];
        double q = trunc(a[j] * C.rec[EC_WIDTH + j]);
        double r = fma(-q, W, a[j]);
        q += (a[j] >= 0) ? ((r < 0) ? -1.0 : (r >= W ? 1.0 : 0.0)) : ((r > 0) ? 1.0 : (r <= -W ? -1.0 : 0.0));
        r = fma(-q, W, a[j]);
        r = (r == 0) ? copysign(0.0, a[j]) : r;
        r += (r < 0) ? W : 0.0;
        double x = div_by(r - C.hs[j], C.len[EC_D + j], C.rec[EC_D + j]);
        if (!(x >= -1.0 && x < (double)C.n[j])) x = 0.0;
        const double f = floor(x);
        ix[j] = (f == -1.0) ? C.n[j] - 1 : (int)f;
        w[j] = 1 - (x - f);
        ties += fabs(x - rint(x)) < TIE_VOXEL_EPS;
    }
}

// ---- loads --------------------------------------------------------------------

// Neighbour block of a crank-shaft, end-pivot or slide move, one per wavefront,
// filled straight from HBM into LDS.  Doubles 16 s + q, s = 0 for bead ind0 - 1 and
// bond (ind0 - 1, ind0), s = 1 for bead indf and bond (indf - 1, indf): q = 0-2 r,
// 3-5 t3, 6-10 bond; on a twisting chain 11-13 t2, 14-15 the bond's twist rows.
__device__ __forceinline__ double *ev_nbr()
{
    __shared__ double nbr[EV_WAVES][32];
    return nbr[wave_id()];
}

// The neighbour block once its direct-to-LDS loads have landed.  The compiler's
// wait insertion does not tie these loads to later LDS reads of the block (it
// places its vmcnt wait after them), so the wait is explicit, and the asm's
// memory clobber keeps the reads below it.
__device__ __forceinline__ const double *ev_nbr_ready()
{
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    return ev_nbr();
}

// What one chunk of an evaluation reads of the chain, loaded in one batch: the lane's
// bead (window bead 32 c + i, or tangent pick), its coordinates, binder states and
// (binding moves) modifications; for a tangent rotation the r, t3 and bond of the
// neighbour on the half's side (lower half b - 1, upper half b + 1).
template <int NB>
struct EvBeads {
    int64_t b;
    double o[9];
    int8_t so[NB], mods[NB];
    double nr[6];
    Bond nbond;
    bool has;
};

template <int NB, bool TW>
__device__ __forceinline__ void ev_load(const chromo_replica *R, int mv, int64_t n, int64_t ind0, int64_t indf, int c,
                                        int64_t pick, EvBeads<NB> &B)
{
    const int lane = lane_id(), side = lane >> 5;
    const int64_t N = R->N, i = (int64_t)SEG_MAX * c + (lane & 31);
    const GLOBAL_AS double *Pp = gmem(R->pos);
    const bool tangent = mv == CHROMO_TANGENT_ROTATION, binding = mv == CHROMO_CHANGE_BINDING_STATE;
    const bool act = i < n;
    const int64_t b = tangent ? (act ? pick : 0) : (act ? ind0 + i : ind0);
    B.b = b;
#pragma unroll
    for (int q = 0; q < 9; ++q) B.o[q] = 0;
#pragma unroll
    for (int m = 0; m < NB; ++m) B.so[m] = B.mods[m] = 0;
    if (act) {
#pragma unroll
        for (int q = 0; q < 9; ++q) B.o[q] = Pp[q * N + b];
#pragma unroll
        for (int m = 0; m < NB; ++m) B.so[m] = gmem(R->states)[(int64_t)m * N + b];
        if (binding) {
#pragma unroll
            for (int m = 0; m < NB; ++m) B.mods[m] = gmem(R->marks)[(int64_t)m * N + b];
        }
    }
    if (tangent) {
        B.has = act && (side == 0 ? b != 0 : b + 1 != N);
#pragma unroll
        for (int q = 0; q < 6; ++q) B.nr[q] = 0;
        B.nbond = Bond{0, 0, 0, 0, 0};
        if (B.has) {
            const int64_t a = side == 0 ? b - 1 : b + 1;
#pragma unroll
            for (int q = 0; q < 6; ++q) B.nr[q] = Pp[q * N + a];
            B.nbond = load_bond(R->bonds, N, side == 0 ? b - 1 : b);
        }
    } else if (!binding && c == 0 && N >= 2) {
        // dword j of the neighbour block on lane j; every lane loads (the places a move
        // has no neighbour or a chain no twist for repeat a valid address)
        const int d = lane >> 1, s = d >> 4;
        int q = d & 15;
        if (!TW && q > 10) q = 0;
        int64_t bead = s == 0 ? ind0 - 1 : indf, bond = s == 0 ? ind0 - 1 : indf - 1;
        bead = bead < 0 ? 0 : (bead > N - 1 ? N - 1 : bead);
        bond = bond < 0 ? 0 : (bond > N - 2 ? N - 2 : bond);
        const bool is_bond = (q >= 6 && q < 11) || q >= 14;
        const int64_t row = q < 6 ? q : (q < 11 ? q - 6 : (q < 14 ? q - 5 : q - 9));
        const double *src = is_bond ? R->bonds + row * (N - 1) + bond : R->pos + row * N + bead;
        __builtin_amdgcn_global_load_lds((const void *)((const uint32_t *)src + (lane & 1)),
                                         (void __attribute__((address_space(3))) *)ev_nbr(), 4, 0, 0);
    }
}

// r of bead x (wave-uniform, ind0 - 1 <= x <= indf) of a crank-shaft, end-pivot or slide.
template <int NB>
__device__ __forceinline__ void ev_r3(const chromo_replica *R, const EvBeads<NB> &B, int64_t x, int64_t ind0,
                                      int64_t indf, double v[3])
{
    if (x == ind0 - 1 || x == indf) {
        const double *nb = ev_nbr_ready() + (x == indf ? 16 : 0);
        for (int j = 0; j < 3; ++j) v[j] = nb[j];
    } else if (x - ind0 < SEG_MAX) {
        for (int j = 0; j < 3; ++j) v[j] = readlane_f64(B.o[j], (int)(x - ind0));
    } else {
        for (int j = 0; j < 3; ++j) v[j] = gmem(R->pos)[j * R->N + x];
    }
}

// ---- evaluation ----------------------------------------------------------------

// Wave-uniform results of one evaluation.
struct EvRes {
    double dEp, dEf, expdE;
    int U, accepted, overflow;
};

// The trial coordinates of the lane's bead, kept for the commit of a move of at most
// SEG_MAX beads.
struct EvKeep {
    double w[9];
    int64_t b;
};

// Trial coordinates of bead (o) under proposal P, lane-local (move_funcs.pyx:139-154).
__device__ __forceinline__ void ev_transform(const Proposal &P, const double o[9], double w[9])
{
    const int mv = P.move;
    if (mv == CHROMO_CRANK_SHAFT || mv == CHROMO_END_PIVOT) {
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            w[j] = rowdot(&P.T[4 * j], o[0], o[1], o[2]) + P.T[4 * j + 3];
            w[3 + j] = rowdot(&P.T[4 * j], o[3], o[4], o[5]);
            w[6 + j] = rowdot(&P.T[4 * j], o[6], o[7], o[8]);
        }
    } else if (mv == CHROMO_SLIDE) {
#pragma unroll
        for (int j = 0; j < 3; ++j) w[j] = o[j] + P.T[4 * j + 3];
#pragma unroll
        for (int c = 3; c < 9; ++c) w[c] = o[c];
    } else {
#pragma unroll
        for (int c = 0; c < 9; ++c) w[c] = o[c];
    }
}

// E_pair of the bond from (r0, t30) to (r1, t31), polymers.pyx:1148-1175,1177-1346.
__device__ __forceinline__ double bond_E(const Bond &bd, const double *r0, const double *r1, const double *t30,
                                         const double *t31)
{
    double dr[3], drp[3], be[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) dr[i] = r1[i] - r0[i];
    const double par = dot3(t30, dr);
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        drp[i] = dr[i] - t30[i] * par;
        be[i] = t31[i] - t30[i] - drp[i] * bd.eta;
    }
    return E_pair(bd, be, par, drp);
}

// The fold of one chunk's npos positions into S.acc (fields.pyx:1491-1520): lanes
// 8 m + l of a position's group hold species m of corner l; PB positions share the
// arithmetic of one step, and their adds are issued one position after the other.  Every
// row of the chunk's arrays is written (a position past npos with weights of zero), so
// the steps need no bounds.  THR: the 1e-18 rule; without it a zero weight alone is
// passed over.
template <int NB, bool THR>
__device__ __forceinline__ void ev_fold(const EvLds &S, int npos, bool degen)
{
    constexpr int Bp1 = NB + 1, LP = 8 * Bp1, PB = WAVE / LP, UN = PB == 1 ? 8 : 4;
    static_assert(EV_POS % (PB * UN) == 0, "whole steps");
    const int lane = lane_id(), l = lane & 7;
    const bool in = lane < PB * LP;
    const int pj = in ? lane / LP : 0, m = in ? (lane % LP) >> 3 : 0;
    char *acc = (char *)(S.acc + m);
    for (int p0 = 0; p0 < npos; p0 += PB * UN) {
        double t[UN];
        char *to[UN];
        bool go[UN];
#pragma unroll
        for (int k = 0; k < UN; ++k) {
            const int p = p0 + k * PB + pj;
            // species 0 has the factor 1: no branch, so the steps' loads go out together
            t[k] = S.c0[8 * p + l] * (double)S.pst[8 * p + m];
            to[k] = acc + S.eq[8 * p + l];
            go[k] = in && (THR ? fabs(t[k]) > 1E-18 : !(fabs(t[k]) <= 0));
        }
        if (!degen) {
#pragma unroll
            for (int k = 0; k < UN; ++k) {
#pragma unroll
                for (int j = 0; j < PB; ++j) {
                    if (go[k] && pj == j) lds_add((double *)to[k], t[k]);
                    __builtin_amdgcn_wave_barrier();
                }
            }
        } else {
#pragma unroll
            for (int k = 0; k < UN; ++k) {
                for (int s = 0; s < 8 * PB; ++s) {
                    if (go[k] && pj == (s >> 3) && l == (s & 7)) lds_add((double *)to[k], t[k]);
                    __builtin_amdgcn_wave_barrier();
                }
            }
        }
    }
    wave_sync();
}

// One voxel's share of get_dE_binders_and_beads (fields.pyx:1723-1750) and of
// nonspecific_interact_dE (fields.pyx:1792-1842), as voxel_dE_terms, with the chi
// prefactor from the launch's constants and the cross-talk sums only where a
// coefficient is not zero.
template <int NB>
__device__ __forceinline__ void ev_terms(const chromo_replica *R, const EvConst &C, int v, const double *r,
                                         const double *a, double *S2, double *SX, double &NS)
{
    double aj[NB];
#pragma unroll
    for (int j = 0; j < NB; ++j) {
        aj[j] = r[j + 1] + a[j + 1];
        double d2 = aj[j] * aj[j] - r[j + 1] * r[j + 1];
        if (fabs(d2) < 1E-18) d2 = 0;
        S2[j] += d2;
    }
    if (C.cross) {
#pragma unroll
        for (int j = 0; j < NB; ++j)
#pragma unroll
            for (int k = 0; k < NB; ++k) {
                double dx = (aj[j] * (r[k + 1] + a[k + 1])) - (r[j + 1] * r[k + 1]);
                if (fabs(dx) < 1E-18) dx = 0;
                SX[j * NB + k] += dx;
            }
    }
    const double V = R->bead_vol, vf = R->vf_limit;
    const double cphi = R->access_vol ? R->chi * (R->access_vol[v] / V) : C.cphi;
    const double vf0 = r[0] * V, vf1 = vf0 + (a[0] * V);
    if (vf0 > vf && vf1 > vf) atomicAdd((unsigned long long *)&R->counters[CHROMO_CNT_TIE_HUGE], 1ull);
    NS += vf1 > vf ? E_HUGE_FIELD * vf1 : cphi * (vf1 * vf1);
    NS -= vf0 > vf ? E_HUGE_FIELD * vf0 : cphi * (vf0 * vf0);
}

// Metropolis on dEp and dEf (mc_sim.pyx:152-182).
__device__ __forceinline__ void ev_metropolis(double dEp, double dEf, bool field, double u, int U, EvRes &res)
{
    double dE = 0;
    dE += dEp;
    if (field) dE += dEf;
    res.dEp = dEp;
    res.dEf = dEf;
    res.expdE = exp(-dE);
    res.accepted = u < res.expdE;
    res.U = U;
}

// A tangent rotation of n <= EV_LANES picks (pick i and its rotation on lane i of P):
// elastic dE only.  The lower half of the wavefront takes the bond below each picked
// bead, the upper half the bond above.  B: ev_load's data of the first chunk.
template <int NB, bool TW>
__device__ __forceinline__ void ev_tangent(const chromo_replica *R, const Proposal &P, double u, EvRes &res, EvKeep &K,
                                           EvBeads<NB> &B)
{
    const int lane = lane_id(), side = lane >> 5;
    const int64_t N = R->N;
    const int n = (int)P.n;
    double dEp = 0;
    for (int c = 0; SEG_MAX * c < n; ++c) {
        const int i = SEG_MAX * c + (lane & 31), nb = n - SEG_MAX * c < SEG_MAX ? n - SEG_MAX * c : SEG_MAX;
        if (c > 0) ev_load<NB, TW>(R, P.move, n, 0, 0, c, __shfl(P.mypick, i & 63), B);
        double T[9];
#pragma unroll
        for (int q = 0; q < 9; ++q) T[q] = __shfl(P.myT[q], i & 63);
        double w[9];
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            w[j] = B.o[j];
            w[3 + j] = rowdot(&T[3 * j], B.o[3], B.o[4], B.o[5]);
            w[6 + j] = rowdot(&T[3 * j], B.o[6], B.o[7], B.o[8]);
        }
        double e = 0;
        if (B.has) {
            double twt = 0, twc = 0;
            if constexpr (TW) {
                if (side == 0) twist_forward(R->bonds, R->pos, N, B.b - 1, B.o, w, twt, twc);
                else twist_reverse(R->bonds, R->pos, N, B.b + 1, B.o, w, twt, twc);
            }
            // the bond's lower and upper bead, current and trial
            const bool lo = side == 0;
            double r0[3], r1[3], t0c[3], t1c[3], t0t[3], t1t[3];
#pragma unroll
            for (int j = 0; j < 3; ++j) {
                r0[j] = lo ? B.nr[j] : B.o[j];
                r1[j] = lo ? B.o[j] : B.nr[j];
                t0c[j] = lo ? B.nr[3 + j] : B.o[3 + j];
                t1c[j] = lo ? B.o[3 + j] : B.nr[3 + j];
                t0t[j] = lo ? B.nr[3 + j] : w[3 + j];
                t1t[j] = lo ? w[3 + j] : B.nr[3 + j];
            }
            e = (bond_E(B.nbond, r0, r1, t0t, t1t) + twt) - (bond_E(B.nbond, r0, r1, t0c, t1c) + twc);
        }
        // per bead 0 + lower + upper, then bead by bead
        const double up = __shfl(e, (lane & 31) + 32);
        double eb = 0;
        eb += e;
        eb += up;
        for (int j = 0; j < nb; ++j) dEp += readlane_f64(eb, j);
        if (c == 0) {
#pragma unroll
            for (int q = 0; q < 9; ++q) K.w[q] = w[q];
            K.b = B.b;
        }
    }
    ev_metropolis(dEp, 0, false, u, 0, res);
}

// Evaluates proposal P against the committed state: polymer dE (SSWLC.compute_dE,
// polymers.pyx:1024-1082), field dE (UniformDensityField.compute_dE,
// fields.pyx:1149-1233) and the Metropolis test with the uniform draw u
// (mc_sim.pyx:152-182).  Crank-shaft, end-pivot and slide moves of any length,
// tangent rotations and binding moves of at most EV_LANES beads.  Writes nothing
// outside S and K.  One whole wavefront; S's hash is empty on entry and holds the
// move's res.U voxels on return (ev_release empties it; after an overflow it is
// empty).  B holds what ev_load fetched for chunk 0.
template <int NB, bool TW>
__device__ __forceinline__ void ev_eval(const chromo_replica *R, const EvConst &C, const Proposal &P, double u,
                                        const EvLds &S, EvRes &res, EvKeep &K, EvBeads<NB> &B)
{
    constexpr int Bp1 = NB + 1;
    const int lane = lane_id(), i32 = lane & 31, k = lane >> 5;
    const int64_t N = R->N;
    const int mv = P.move;
    const int64_t n = P.n, ind0 = P.ind0, indf = P.indf;
    res.overflow = 0;
    if (mv == CHROMO_TANGENT_ROTATION) {
        ev_tangent<NB, TW>(R, P, u, res, K, B);
        return;
    }
    const bool state_change = mv == CHROMO_CHANGE_BINDING_STATE;
    const bool field = R->field_on != 0;
    const bool thr = C.fast == 0;
    const int nx = C.n[0], ny = C.n[1], nz = C.n[2], nxy = nx * ny;
    const bool degen = nx == 1 || ny == 1 || nz == 1;
    const double *avol = R->access_vol;
    const int ct = state_change ? 0 : R->confine_type;
    const double cl = R->confine_length;
    const GLOBAL_AS double *rho_g = gmem(R->density);

    double dEp = 0;
    int dbl[NB], dbl_t[NB], out_t = 0, out_c = 0, U = 0;
#pragma unroll
    for (int j = 0; j < NB; ++j) dbl[j] = dbl_t[j] = 0;
    double rho[2][Bp1];
    const int nchunks = (int)((n + SEG_MAX - 1) / SEG_MAX);
    for (int c = 0; c < nchunks; ++c) {
        const int64_t i = (int64_t)SEG_MAX * c + i32;
        const bool act = i < n;
        const int nb = (int)(n - (int64_t)SEG_MAX * c < SEG_MAX ? n - (int64_t)SEG_MAX * c : SEG_MAX);
        if (c > 0) ev_load<NB, TW>(R, mv, n, ind0, indf, c, 0, B);
        double w[9];
        ev_transform(P, B.o, w);
        if (c == 0) {
#pragma unroll
            for (int q = 0; q < 9; ++q) K.w[q] = w[q];
            K.b = B.b;
        }
        int8_t sn[NB];
#pragma unroll
        for (int m = 0; m < NB; ++m) sn[m] = B.so[m];
        if (state_change) {
            const int nw = __shfl(P.mynew, (int)(i & 63));
#pragma unroll
            for (int m = 0; m < NB; ++m)
                if (m == P.binder && act) sn[m] = (int8_t)nw;
            double e = 0;
            if (act) e = bead_binding_dE<NB>(R, B.mods, B.so, sn);
            for (int j = 0; j < nb; ++j) dEp += readlane_f64(e, j);
        } else if (act) {
            // the end beads of the window, both configurations
            constexpr int Q = TW ? 9 : 6;
            if (i == 0) {
#pragma unroll
                for (int q = 0; q < Q; ++q) S.ends[9 * k + q] = k ? w[q] : B.o[q];
            }
            if (i == n - 1) {
#pragma unroll
                for (int q = 0; q < Q; ++q) S.ends[18 + 9 * k + q] = k ? w[q] : B.o[q];
            }
        }
        if (!field) {
            // only the end beads matter
            if (c == 0 && nchunks > 2) c = nchunks - 2;
            continue;
        }
        double pt[3];
#pragma unroll
        for (int j = 0; j < 3; ++j) pt[j] = (k == 0 || state_change) ? B.o[j] : w[j];

        // count_doubly_bound (fields.pyx:1877-1937) and confinement (:121-202)
#pragma unroll
        for (int j = 0; j < NB; ++j) {
            dbl[j] += __popcll(__ballot(act && k == 0 && B.so[j] == 2));
            dbl_t[j] += __popcll(__ballot(act && k == 0 && sn[j] == 2));
        }
        if (ct == 1) {
            const uint64_t m = __ballot(act && sqrt(dot3(pt, pt)) > cl);
            out_c += __popc((uint32_t)m);
            out_t += __popc((uint32_t)(m >> 32));
        } else if (ct != 0) {
#pragma unroll
            for (int j = 0; j < 3; ++j) out_t += __popcll(__ballot(act && k == 1 && fabs(pt[j]) > cl / 2));
        }

        // the position's corner voxels and weight / volume (fields.pyx:1472-1488)
        const int p = 2 * i32 + k;
        int v8[8], h8[8];
        double c8[8];
        uint64_t sp = 1;
        int ties = 0;
#pragma unroll
        for (int m = 0; m < NB; ++m) sp |= (uint64_t)(uint8_t)(k == 0 ? B.so[m] : sn[m]) << (8 * (m + 1));
        uint32_t bad = 0;
        int hb[8];
        if (act) {
            int ix[3];
            double wt[3];
            ev_lower(R, C, pt, ix, wt, ties);
            const int x1 = ix[0] + 1 == nx ? 0 : ix[0] + 1, y1 = ix[1] + 1 == ny ? 0 : ix[1] + 1,
                      z1 = ix[2] + 1 == nz ? 0 : ix[2] + 1;
            const double ux = 1 - wt[0], uy = 1 - wt[1], uz = 1 - wt[2];
            const double xy[4] = {wt[0] * wt[1], ux * wt[1], wt[0] * uy, ux * uy};
            const int yz[4] = {nx * ix[1] + nxy * ix[2], nx * y1 + nxy * ix[2], nx * ix[1] + nxy * z1,
                               nx * y1 + nxy * z1};
            const int hx[2] = {ix[0] & 15, x1 & 15}, hy[2] = {(ix[1] & S.ymask) << 4, (y1 & S.ymask) << 4},
                      hz[2] = {(ix[2] & 7) << S.zshift, (z1 & 7) << S.zshift};
#pragma unroll
            for (int l = 0; l < 8; ++l) {
                v8[l] = ((l & 1) ? x1 : ix[0]) + yz[l >> 1];
                h8[l] = hb[l] = hx[l & 1] | hy[(l >> 1) & 1] | hz[l >> 2];
                c8[l] = xy[l & 3] * ((l & 4) ? uz : wt[2]);
            }
            int old[8];
#pragma unroll
            for (int l = 0; l < 8; ++l) old[l] = atomicCAS(&S.hkey[h8[l]], HKEY_EMPTY, v8[l]);
            if (avol) {
#pragma unroll
                for (int l = 0; l < 8; ++l) c8[l] = c8[l] / avol[v8[l]];
            } else if (C.recip) {
                const double vol = C.vol, rvol = C.rvol;
#pragma unroll
                for (int l = 0; l < 8; ++l) c8[l] = div_by(c8[l], vol, rvol);
            } else {
#pragma unroll
                for (int l = 0; l < 8; ++l) c8[l] = c8[l] / C.vol;
            }
#pragma unroll
            for (int l = 0; l < 8; ++l) bad |= (old[l] != HKEY_EMPTY && old[l] != v8[l]) ? 1u << l : 0u;
        }
        // linear probing of the few whose slot another voxel holds
        int probes = 0;
        while (wave_any(bad != 0) && probes < S.hsize) {
            ++probes;
#pragma unroll
            for (int l = 0; l < 8; ++l) {
                if (bad >> l & 1) {
                    h8[l] = (h8[l] + 1) & (S.hsize - 1);
                    const int old = atomicCAS(&S.hkey[h8[l]], HKEY_EMPTY, v8[l]);
                    if (old == HKEY_EMPTY || old == v8[l]) bad &= ~(1u << l);
                }
            }
        }
        count_ties(R, ties);
        const bool full = wave_any(bad != 0);
        if (act && !full) {
#pragma unroll
            for (int l = 0; l < 8; ++l) atomicMin(&S.hval[h8[l]], 8 * p + l);
        }
        wave_sync();
        // number the voxels this chunk is the first to touch
        const int U0 = U;
        int hv[8];
#pragma unroll
        for (int l = 0; l < 8; ++l) hv[l] = (act && !full) ? S.hval[h8[l]] : 0;
#pragma unroll
        for (int l = 0; l < 8; ++l) {
            const bool first = act && !full && hv[l] == 8 * p + l;
            int cnt;
            const int q = U + wave_excl_count(first, cnt);
            if (first && q < S.ucap) {
                S.hval[h8[l]] = EV_NUM + q;
                S.uv[q] = make_int2(v8[l], h8[l] | (hb[l] << 16));
            }
            U += cnt;
        }
        if (full || U > S.ucap) {
            ev_clear(S);
            res.overflow = 1;
            res.U = U;
            return;
        }
        for (int t = U0 * Bp1 + lane; t < U * Bp1; t += WAVE) S.acc[t] = 0;
        wave_sync();
        {
            // the position's rows; the current position takes its weights away
            uint32_t qq[8];
#pragma unroll
            for (int l = 0; l < 8; ++l)
                qq[l] = act ? (uint32_t)(S.hval[h8[l]] - EV_NUM) * (uint32_t)(sizeof(double) * Bp1) : 0u;
            *(uint4 *)&S.eq[8 * p] = make_uint4(qq[0] | qq[1] << 16, qq[2] | qq[3] << 16, qq[4] | qq[5] << 16,
                                                qq[6] | qq[7] << 16);
#pragma unroll
            for (int l = 0; l < 8; l += 2)
                *(double2 *)&S.c0[8 * p + l] = act ? make_double2(k ? c8[l] : -c8[l], k ? c8[l + 1] : -c8[l + 1])
                                                   : make_double2(0, 0);
            *(uint64_t *)&S.pst[8 * p] = sp;
        }
        wave_sync();
        if (c == nchunks - 1) {
            // every voxel is known: the first densities travel during the fold
#pragma unroll
            for (int a = 0; a < 2; ++a) {
                const int q = a * WAVE + lane;
                const int v = q < U ? S.uv[q].x : 0;
#pragma unroll
                for (int m = 0; m < Bp1; ++m) rho[a][m] = q < U ? rho_g[(int64_t)v * Bp1 + m] : 0.0;
            }
        }
        if (thr) ev_fold<NB, true>(S, 2 * nb, degen);
        else ev_fold<NB, false>(S, 2 * nb, degen);
    }

    if (!state_change) {
        // the two bonds that leave the window, trial and current, one lane each:
        // lane 2 s + k, s = 0 bond (ind0 - 1, ind0), s = 1 bond (indf - 1, indf)
        wave_sync();
        const double *nb = ev_nbr_ready();
        double e = 0;
        if (lane < 4) {
            const int s = lane >> 1;
            const double *x = nb + 16 * s, *y = &S.ends[18 * s + 9 * (lane & 1)];
            const Bond bd{x[6], x[7], x[8], x[9], x[10]};
            double r0[3], r1[3], t0[3], t1[3];
#pragma unroll
            for (int j = 0; j < 3; ++j) {
                r0[j] = s == 0 ? x[j] : y[j];
                r1[j] = s == 0 ? y[j] : x[j];
                t0[j] = s == 0 ? x[3 + j] : y[3 + j];
                t1[j] = s == 0 ? y[3 + j] : x[3 + j];
            }
            double tw = 0;
            if constexpr (TW) {
                double a0[3], a1[3];
#pragma unroll
                for (int j = 0; j < 3; ++j) {
                    a0[j] = s == 0 ? x[11 + j] : y[6 + j];
                    a1[j] = s == 0 ? y[6 + j] : x[11 + j];
                }
                tw = twist_energy(x[14], x[15], twist_omega(a0, t0, a1, t1));
            }
            e = bond_E(bd, r0, r1, t0, t1) + tw;
        }
        const double ef = readlane_f64(e, 1) - readlane_f64(e, 0), er = readlane_f64(e, 3) - readlane_f64(e, 2);
        if (ind0 != 0) dEp += ef;
        if (indf != N) dEp += er;
    }

    double dEf = 0;
    if (field) {
        double S2[NB], SX[NB * NB], NS = 0;
#pragma unroll
        for (int j = 0; j < NB; ++j) S2[j] = 0;
#pragma unroll
        for (int j = 0; j < NB * NB; ++j) SX[j] = 0;
        for (int q0 = 0; q0 < U; q0 += 2 * WAVE) {
#pragma unroll
            for (int a = 0; a < 2; ++a) {
                const int q = q0 + a * WAVE + lane;
                double r[Bp1];
#pragma unroll
                for (int m = 0; m < Bp1; ++m) r[m] = rho[a][m];
                // the next densities travel during this round's terms
                const int qn = q + 2 * WAVE;
                if (qn < U) {
                    const int vn = S.uv[qn].x;
#pragma unroll
                    for (int m = 0; m < Bp1; ++m) rho[a][m] = rho_g[(int64_t)vn * Bp1 + m];
                }
                if (q < U) {
                    double d[Bp1];
#pragma unroll
                    for (int m = 0; m < Bp1; ++m) d[m] = S.acc[q * Bp1 + m];
                    ev_terms<NB>(R, C, S.uv[q].x, r, d, S2, SX, NS);
#pragma unroll
                    for (int m = 0; m < Bp1; ++m) S.acc[q * Bp1 + m] = r[m] + d[m];
                }
            }
        }
        const double share = wave_sum(lane_field_share<NB>(R, S2, SX, NS));
        dEf = field_dE_total<NB>(R, share, dbl_t, dbl, out_t, out_c, state_change);
    }
    if (!state_change && n > SEG_MAX && lane < 12) {
        // the commit works the trial coordinates out again
        double t = 0;
#pragma unroll
        for (int q = 0; q < 12; ++q) t = lane == q ? P.T[q] : t;
        S.tmat[lane] = t;
    }
    ev_metropolis(dEp, dEf, field, u, U, res);
}

// Writes an accepted proposal: bead coordinates or states (MCAdapter.accept,
// moves.pyx:190-226) and the touched voxels' densities (update_affected_densities,
// fields.pyx:1968-1975).  P as evaluated, of which moves of more than SEG_MAX beads
// take the transform from S.tmat (P.T is not read).
template <int NB>
__device__ __forceinline__ void ev_commit(const chromo_replica *R, const Proposal &P, const EvKeep &K, const EvLds &S,
                                          int U)
{
    constexpr int Bp1 = NB + 1;
    const int lane = lane_id(), mv = P.move;
    const int64_t N = R->N, n = P.n;
    GLOBAL_AS double *Pp = gmem(R->pos);
    if (mv == CHROMO_CHANGE_BINDING_STATE) {
        if (lane < n) gmem(R->states)[(int64_t)P.binder * N + P.ind0 + lane] = (int8_t)P.mynew;
    } else if (n <= SEG_MAX) {
        const int c0 = (mv == CHROMO_TANGENT_ROTATION) ? 3 : 0;
        const int c1 = (mv == CHROMO_SLIDE) ? 3 : 9;
        if (lane < n) {
#pragma unroll
            for (int c = 0; c < 9; ++c)
                if (c >= c0 && c < c1) Pp[c * N + K.b] = K.w[c];
        }
    } else if (mv == CHROMO_TANGENT_ROTATION) {
        if (lane < n) {
            double o[9];
#pragma unroll
            for (int c = 3; c < 9; ++c) o[c] = Pp[c * N + P.mypick];
#pragma unroll
            for (int j = 0; j < 3; ++j) {
                Pp[(3 + j) * N + P.mypick] = rowdot(&P.myT[3 * j], o[3], o[4], o[5]);
                Pp[(6 + j) * N + P.mypick] = rowdot(&P.myT[3 * j], o[6], o[7], o[8]);
            }
        }
    } else {
        Proposal Q;
        Q.move = mv;
#pragma unroll
        for (int q = 0; q < 12; ++q) Q.T[q] = S.tmat[q];
        const int c1 = mv == CHROMO_SLIDE ? 3 : 9;
        for (int64_t i = lane; i < n; i += WAVE) {
            const int64_t b = P.ind0 + i;
            double o[9], w[9];
#pragma unroll
            for (int c = 0; c < 9; ++c) o[c] = c < c1 ? Pp[c * N + b] : 0.0;
            ev_transform(Q, o, w);
#pragma unroll
            for (int c = 0; c < 9; ++c)
                if (c < c1) Pp[c * N + b] = w[c];
        }
    }
    GLOBAL_AS double *rho = gmem(R->density);
    for (int q = lane; q < U; q += WAVE) {
        const int64_t v = S.uv[q].x;
#pragma unroll
        for (int m = 0; m < Bp1; ++m) rho[v * Bp1 + m] = S.acc[q * Bp1 + m];
    }
}

}  // namespace
