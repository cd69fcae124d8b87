// chromo_density.hpp -- deterministic voxel-density scatter shared by the MC
// initialisation and the reference energies.
//
// UniformDensityField.update_all_densities_for_all_polymers
// (chromo/fields.pyx:2041-2106) adds every bead's eight trilinear weights to
// the grid in bead order.  To reproduce those per-voxel sums bit for bit in
// parallel, beads are listed per tile of voxels, and one wavefront per tile folds its
// list in bead order into LDS.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <string>
#include <type_traits>

#include "chromo_device.hpp"

namespace chromo {
namespace {

// Grid of a UniformDensityField (fields.pyx:536-575).
struct GridGeom {
    int64_t nx, ny, nz;
    double width[3], dxyz[3], half_width[3], half_step[3];
    double vol_bin;
    const double *access_vol = nullptr;   // per-voxel accessible volumes, or nullptr: vol_bin
};

// Bead coordinate c of bead b is p[c * sc + b * sb].
struct PosView {
    const double *p;
    int64_t sc, sb;
};

__device__ __forceinline__ void grid_lower(const GridGeom &G, double x0, double x1, double x2,
                                           int64_t ix[3], double w[3])
{
    const int64_t nn[3] = {G.nx, G.ny, G.nz};
    const double xs[3] = {x0, x1, x2};
    for (int j = 0; j < 3; ++j) {
        double x = pymod(xs[j] + G.half_width[j], G.width[j]) - G.half_step[j];
        double q = x / G.dxyz[j];
        if (!(q >= -1.0 && q < (double)nn[j])) q = 0.0;
        int64_t ind = (int64_t)floor(q);
        ix[j] = (ind == -1) ? nn[j] - 1 : ind;
        w[j] = 1 - (q - (double)ind);
    }
}

constexpr size_t SCRATCH_ALIGN = 256;

inline size_t align_scratch(size_t o) { return (o + SCRATCH_ALIGN - 1) / SCRATCH_ALIGN * SCRATCH_ALIGN; }

}  // namespace
}  // namespace chromo

#include "chromo_tiles.hpp"

namespace chromo {
namespace {

// One scatter: a chain's beads into its density grid.
struct ScatterJob {
    GridGeom G;
    TileGeom T;
    int64_t N;
    PosView P;
    const int8_t *states;
    double *density;                // n_bins x Bp1
    int32_t *cell, *list;           // per bead; the tiles' bead lists
    int32_t *cnt, *fill;            // per tile
    ListPlace *base, *cursor;
    int32_t Bp1, cleanup;
};

// A job's scratch carved from base (nullptr: sizes only); returns the bytes used, a
// multiple of SCRATCH_ALIGN.  cnt, fill and cursor lie in a row, the first of them.
inline size_t scatter_carve(ScatterJob &J, char *base)
{
    size_t o = 0;
    auto take = [&](auto *&p, size_t n) {
        p = base ? (std::remove_reference_t<decltype(p)>)(base + o) : nullptr;
        o = align_scratch(o + sizeof(*p) * n);
    };
    take(J.cnt, (size_t)J.T.ntiles);
    take(J.fill, (size_t)J.T.ntiles);
    take(J.cursor, 1);
    take(J.base, (size_t)J.T.ntiles);
    take(J.cell, (size_t)J.N);
    take(J.list, (size_t)J.N * tile_images(J.T));
    return o;
}

inline ScatterJob scatter_job(const GridGeom &G, int64_t N, int Bp1, PosView P, const int8_t *states, double *density,
                              int cleanup)
{
    ScatterJob J{};
    J.G = G;
    J.T = fold_geom(G);
    J.N = N;
    J.P = P;
    J.states = states;
    J.density = density;
    J.Bp1 = Bp1;
    J.cleanup = cleanup;
    return J;
}

// The kernels take job blockIdx.y of a table in device memory, or (TABLE false) the one
// in `one`: both are read with scalar loads.
template <bool TABLE>
__global__ void k_scatter_clear(const ScatterJob *__restrict__ jobs, const ScatterJob one)
{
    const ScatterJob &J = TABLE ? jobs[blockIdx.y] : one;
    const int i = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    if (i < J.T.ntiles) J.cnt[i] = J.fill[i] = 0;
    if (i == 0) *J.cursor = 0;
}

template <bool TABLE>
__global__ void k_scatter_base(const ScatterJob *__restrict__ jobs, const ScatterJob one)
{
    const ScatterJob &J = TABLE ? jobs[blockIdx.y] : one;
    if ((int)(blockIdx.x * blockDim.x) >= J.T.ntiles) return;
    tile_bases(J.cnt, J.base, J.cursor, J.T.ntiles);
}

template <bool TABLE, bool PLACE>
__global__ void __launch_bounds__(BIN_THREADS) k_scatter_bin(const ScatterJob *__restrict__ jobs, const ScatterJob one)
{
    const ScatterJob &J = TABLE ? jobs[blockIdx.y] : one;
    if ((int64_t)blockIdx.x * BIN_THREADS >= J.N) return;
    tile_bin<PLACE, false, true>(J.G, J.T, J.N, J.P, J.cell, PLACE ? J.fill : J.cnt, J.base, J.list);
}

// Ascending sort of a[0 .. n) in global memory by one wavefront: a bitonic network whose
// comparators all point the same way (each merge starts with a mirrored step), so that
// the places past n, which would hold the largest keys, need not exist.
__device__ __forceinline__ void wave_sort(int32_t *a, int n)
{
    const uint32_t lane = (uint32_t)lane_id(), un = (uint32_t)n;
    for (int kb = 1; kb <= 31 && (1u << (kb - 1)) < un; ++kb) {
        for (int db = kb - 1; db >= 0; --db) {
            // pair t: groups of 2^db pairs over 2^(db + 1) places
            for (uint32_t t = lane; ((t >> db) << (db + 1)) < un; t += WAVE) {
                const uint32_t g = (t >> db) << (db + 1), o = t & ((1u << db) - 1);
                const uint32_t i = g + o, j = db == kb - 1 ? g + (2u << db) - 1 - o : i + (1u << db);
                if (j < un) {
                    const int32_t x = a[i], y = a[j];
                    if (x > y) {
                        a[i] = y;
                        a[j] = x;
                    }
                }
            }
            wave_sync_global();
        }
    }
}

// A tile's list in bead order, without sorting it: the placement leaves it as runs in
// bead order (what one block placed), so only the runs are ordered, by their first bead.
// Run k of that order starts at list place from[k] and at position off[k] of the order;
// off[runs] = len.  When there are more than RUNS_MAX runs, or runs that overlap (entries
// a block had to place one by one), the list itself is sorted and is one run.  One
// wavefront; returns the number of runs.
constexpr int RUNS_MAX = 128;

__device__ __forceinline__ int list_runs(int32_t *list, int len, int32_t *from, int32_t *off, int32_t *key)
{
    const int lane = lane_id();
    int runs = 0;
    for (int i0 = 0; i0 < len && runs <= RUNS_MAX; i0 += WAVE) {
        const int i = i0 + lane;
        const int x = i < len ? list[i] : 0, y = i > 0 && i < len ? list[i - 1] : 0;
        const bool head = i < len && (i == 0 || x < y || (x ^ y) >> 8 != 0);
        static_assert(BIN_THREADS == 256, "a run's beads share their upper bits");
        int cnt;
        const int k = runs + wave_excl_count(head, cnt);
        if (head && k < RUNS_MAX) {
            from[k] = i;
            key[k] = x;
        }
        runs += cnt;
    }
    wave_sync();
    bool bad = runs > RUNS_MAX;
    if (!bad) {
        // ranks by counting; a run's length from the next run's start
        int lens[RUNS_MAX / WAVE], rank[RUNS_MAX / WAVE], keep[RUNS_MAX / WAVE];
#pragma unroll
        for (int q = 0; q < RUNS_MAX / WAVE; ++q) {
            lens[q] = rank[q] = keep[q] = 0;
            const int k = q * WAVE + lane;
            if (q * WAVE >= runs) continue;
            if (k < runs) {
                const int mine = key[k], end = k + 1 < runs ? from[k + 1] : len;
                keep[q] = from[k];
                lens[q] = end - keep[q];
                for (int j = 0; j < runs; ++j) rank[q] += key[j] < mine;
                // no other run starts between this one's first and last bead
                const int last = list[end - 1];
                for (int j = 0; j < runs; ++j) bad = bad || (key[j] > mine && key[j] <= last);
            }
        }
        bad = wave_any(bad);
        wave_sync();
        if (!bad) {
#pragma unroll
            for (int q = 0; q < RUNS_MAX / WAVE; ++q) {
                const int k = q * WAVE + lane;
                if (q * WAVE < runs && k < runs) {
                    from[rank[q]] = keep[q];
                    off[rank[q]] = lens[q];
                }
            }
            wave_sync();
            int at = 0;
            for (int k0 = 0; k0 < runs; k0 += WAVE) {
                const int k = k0 + lane, n = k < runs ? off[k] : 0;
                int tot;
                const int o = wave_excl_scan(n, tot);
                if (k < runs) off[k] = at + o;
                at += tot;
            }
            if (lane == 0) off[runs] = len;
            wave_sync();
            return runs;
        }
    }
    wave_sort(list, len);
    if (lane == 0) {
        from[0] = 0;
        off[0] = 0;
        off[1] = len;
    }
    wave_sync();
    return 1;
}

// The density of one tile's voxels: the reference's bead-order fold
// (fields.pyx:2063-2106) by one wavefront.  The tile's beads go through 64 at a time in
// bead order, each lane working out its bead's weights / volume and voxel places; then
// one LDS floating-point add per bead, its lanes the corners times the species, issued
// in bead order: the LDS executes a wavefront's operations in order, so each voxel's sum
// is the reference's left fold bit for bit.  (On a grid with a one-voxel axis corners of
// a bead share a voxel and are issued one after the other.)
// What bounds it: each wavefront's chain of loads and LDS round trips (27,000 cycles for
// a tile of 60 listed beads) at three to four wavefronts per SIMD.  10^6 beads, B = 4,
// 128^3: 171 us, of 262 us a scatter; the merge of eight sorted buckets per voxel it
// replaces took 311 us, of 700.  With 8 x 8 x 4 tiles the longest list decides (241 us).
template <bool TABLE, int NB>
__global__ void __launch_bounds__(WAVE) k_scatter_fold(const ScatterJob *__restrict__ jobs, const ScatterJob one)
{
    constexpr int Bp1 = NB + 1, LP = 8 * Bp1, PB = WAVE / LP, UN = PB == 1 ? 8 : 4;
    constexpr int VOX = FOLD_MAX[0] * FOLD_MAX[1] * FOLD_MAX[2];
    // the sums of the tile's voxels, then a row per corner that nobody reads for corners
    // outside the tile (one row for all would make their adds wait for each other)
    __shared__ double sum[(VOX + 8) * Bp1], c0[8 * WAVE];
    __shared__ uint16_t vox[8 * WAVE];      // byte offset of a corner's sums
    __shared__ uint8_t fac[8 * WAVE];       // factor m of bead p at 8 p + m: 1, then the binder states
    __shared__ int32_t from[RUNS_MAX], off[RUNS_MAX + 1];
    static_assert(sizeof(c0) >= sizeof(int32_t) * RUNS_MAX, "the runs' keys use c0 before its first use");
    constexpr uint32_t ROW = sizeof(double) * Bp1;
    static_assert((VOX + 8) * ROW < 65536, "byte offsets fit 16 bits");
    const ScatterJob &J = TABLE ? jobs[blockIdx.y] : one;
    const int tile = (int)blockIdx.x;
    if (tile >= J.T.ntiles || J.Bp1 != Bp1) return;
    const TileGeom &T = J.T;
    const int lane = lane_id();
    const int tt[3] = {tile % T.nt[0], (tile / T.nt[0]) % T.nt[1], tile / (T.nt[0] * T.nt[1])};
    int start[3], size[3];
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        start[j] = tile_start(T.n[j], T.nt[j], tt[j]);
        size[j] = tile_start(T.n[j], T.nt[j], tt[j] + 1) - start[j];
    }
    const bool degen = T.n[0] == 1 || T.n[1] == 1 || T.n[2] == 1;
    const int stride[3] = {1, FOLD_MAX[0], FOLD_MAX[0] * FOLD_MAX[1]};
    for (int i = lane; i < VOX * Bp1; i += WAVE) sum[i] = 0;
    const uint32_t len = (uint32_t)J.cnt[tile];     // its places and the step past the last in 32 bits
    int32_t *list = J.list + J.base[tile];
    const int runs = len > 0 ? list_runs(list, (int)len, from, off, (int32_t *)c0) : 0;
    const bool in = lane < PB * LP;
    const int pj = in ? lane / LP : 0, m = in ? (lane % LP) >> 3 : 0, l8 = lane & 7;
    char *acc = (char *)(sum + m);
    const double *avol = J.G.access_vol;
    for (uint32_t i0 = 0; i0 < len; i0 += WAVE) {
        const int n = len - i0 < (uint32_t)WAVE ? (int)(len - i0) : WAVE;
        if (lane < n) {
            const int32_t i = (int32_t)(i0 + (uint32_t)lane);
            // the run that holds position i0 + lane of the order
            int lo = 0, hi = runs;
            while (hi - lo > 1) {
                const int mid = (lo + hi) >> 1;
                if (off[mid] <= i) lo = mid;
                else hi = mid;
            }
            const int64_t b = list[from[lo] + (i - off[lo])];
            double x[3], w[3];
            int ix[3];
#pragma unroll
            for (int j = 0; j < 3; ++j) x[j] = J.P.p[j * J.P.sc + b * J.P.sb];
            uint64_t st = 1;
#pragma unroll
            for (int j = 0; j < NB; ++j) st |= (uint64_t)(uint8_t)J.states[(int64_t)j * J.N + b] << (8 * (j + 1));
            tile_lower(J.G, T, x, ix, w);
            int at[3][2], ax[3][2];     // place of the lower and upper corner in the tile (-1: outside), on the grid
#pragma unroll
            for (int j = 0; j < 3; ++j) {
                ax[j][0] = ix[j];
                ax[j][1] = ix[j] + 1 == T.n[j] ? 0 : ix[j] + 1;
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    const int d = ax[j][e] - start[j];
                    at[j][e] = d >= 0 && d < size[j] ? d * stride[j] : -1;
                }
            }
            const double u[3] = {1 - w[0], 1 - w[1], 1 - w[2]};
            const double xy[4] = {w[0] * w[1], u[0] * w[1], w[0] * u[1], u[0] * u[1]};
            uint32_t q[8];
#pragma unroll
            for (int l = 0; l < 8; ++l) {
                const int vx = at[0][l & 1], vy = at[1][(l >> 1) & 1], vz = at[2][l >> 2];
                q[l] = ((vx | vy | vz) < 0 ? (uint32_t)(VOX + l) : (uint32_t)(vx + vy + vz)) * ROW;
                const double c = xy[l & 3] * ((l & 4) ? u[2] : w[2]);
                double d;
                if (avol)
                    d = c / avol[(int64_t)ax[0][l & 1] +
                                 (int64_t)T.n[0] * (ax[1][(l >> 1) & 1] + (int64_t)T.n[1] * ax[2][l >> 2])];
                else
                    d = T.recip ? div_by(c, J.G.vol_bin, T.rvol) : c / J.G.vol_bin;
                c0[8 * lane + l] = d;
            }
            *(uint4 *)&vox[8 * lane] = make_uint4(q[0] | q[1] << 16, q[2] | q[3] << 16, q[4] | q[5] << 16,
                                                  q[6] | q[7] << 16);
            *(uint64_t *)&fac[8 * lane] = st;
        } else {
            // the steps below run over whole groups: rows past the last bead add nothing
#pragma unroll
            for (int l = 0; l < 8; ++l) vox[8 * lane + l] = (uint16_t)((VOX + l) * ROW);
#pragma unroll
            for (int l = 0; l < 8; ++l) c0[8 * lane + l] = 0;
            *(uint64_t *)&fac[8 * lane] = 0;
        }
        wave_sync();
        for (int p0 = 0; p0 < n; p0 += PB * UN) {
            static_assert(WAVE % (PB * UN) == 0, "whole steps");
            double t[UN];
            char *to[UN];
#pragma unroll
            for (int k = 0; k < UN; ++k) {
                const int p = p0 + k * PB + pj;
                t[k] = c0[8 * p + l8] * (double)(int8_t)fac[8 * p + m];
                to[k] = acc + vox[8 * p + l8];
            }
            if (!degen) {
#pragma unroll
                for (int k = 0; k < UN; ++k) {
#pragma unroll
                    for (int j = 0; j < PB; ++j) {
                        if (in && pj == j) lds_add((double *)to[k], t[k]);
                        __builtin_amdgcn_wave_barrier();
                    }
                }
            } else {
#pragma unroll
                for (int k = 0; k < UN; ++k)
                    for (int s = 0; s < 8 * PB; ++s) {
                        if (in && pj == (s >> 3) && l8 == (s & 7)) lds_add((double *)to[k], t[k]);
                        __builtin_amdgcn_wave_barrier();
                    }
            }
        }
        wave_sync();
    }
    wave_sync();
    for (int i = lane; i < VOX * Bp1; i += WAVE) {
        const int v = i / Bp1, s = i % Bp1;
        const int x = v % FOLD_MAX[0], y = (v / FOLD_MAX[0]) % FOLD_MAX[1], z = v / (FOLD_MAX[0] * FOLD_MAX[1]);
        if (x >= size[0] || y >= size[1] || z >= size[2]) continue;
        const int64_t gv = (start[0] + x) + (int64_t)T.n[0] * ((start[1] + y) + (int64_t)T.n[1] * (start[2] + z));
        double a = sum[i];
        if (J.cleanup && fabs(a) < 1E-18) a = 0;
        J.density[gv * Bp1 + s] = a;
    }
}

// Largest sizes among the jobs of one launch, and the binder counts present (bit B).
struct ScatterSpan {
    int64_t N = 0;
    int32_t ntiles = 0;
    int binders = 0;
    void add(const ScatterJob &J)
    {
        N = J.N > N ? J.N : N;
        ntiles = J.T.ntiles > ntiles ? J.T.ntiles : ntiles;
        binders |= 1 << (J.Bp1 - 1);
    }
};

template <bool TABLE>
hipError_t scatter_launch(const ScatterJob *jobs, const ScatterJob &one, int njobs, const ScatterSpan &X, hipStream_t st)
{
    const unsigned y = (unsigned)njobs;
    const dim3 gt((unsigned)((X.ntiles + 255) / 256), y), gb((unsigned)((X.N + BIN_THREADS - 1) / BIN_THREADS), y);
    const dim3 gf((unsigned)X.ntiles, y), bin(BIN_THREADS), wave(WAVE);
    hipLaunchKernelGGL((k_scatter_clear<TABLE>), gt, dim3(256), 0, st, jobs, one);
    hipLaunchKernelGGL((k_scatter_bin<TABLE, false>), gb, bin, 0, st, jobs, one);
    hipLaunchKernelGGL((k_scatter_base<TABLE>), gt, dim3(256), 0, st, jobs, one);
    hipLaunchKernelGGL((k_scatter_bin<TABLE, true>), gb, bin, 0, st, jobs, one);
    if (X.binders & 1) hipLaunchKernelGGL((k_scatter_fold<TABLE, 0>), gf, wave, 0, st, jobs, one);
    if (X.binders & 2) hipLaunchKernelGGL((k_scatter_fold<TABLE, 1>), gf, wave, 0, st, jobs, one);
    if (X.binders & 4) hipLaunchKernelGGL((k_scatter_fold<TABLE, 2>), gf, wave, 0, st, jobs, one);
    if (X.binders & 8) hipLaunchKernelGGL((k_scatter_fold<TABLE, 3>), gf, wave, 0, st, jobs, one);
    if (X.binders & 16) hipLaunchKernelGGL((k_scatter_fold<TABLE, 4>), gf, wave, 0, st, jobs, one);
    return hipGetLastError();
}

// Runs the jobs (a table of njobs in device memory, or jobs == nullptr and `one`),
// their scratch carved: five launches and one per further binder count.  Cleared by a
// kernel rather than hipMemsetAsync: a caller may capture this sequence in a HIP graph.
inline hipError_t scatter_run(const ScatterJob *jobs, const ScatterJob &one, int njobs, const ScatterSpan &X,
                              hipStream_t st)
{
    return jobs ? scatter_launch<true>(jobs, one, njobs, X, st) : scatter_launch<false>(nullptr, one, 1, X, st);
}

}  // namespace
}  // namespace chromo
