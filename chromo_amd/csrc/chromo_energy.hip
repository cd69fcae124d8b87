// chromo_energy.hip -- absolute energies and their adjoint (gfx950).
//
// The Monte Carlo dE of chromo (chromo/polymers.pyx:1024-1538,
// chromo/fields.pyx:1149-1842) are differences of
//
//   E(r, theta) = E_elastic(r)                       sum over bonds of E_pair
//               + E_field(rho(r), theta)             voxel sums below
//               + E_bind(states, theta)              single-site free energies
//
//   E_field = sum_v [ sum_j pref_j rho_vj^2 + sum_jk X_jk rho_vj rho_vk + g(phi_v) ]
//             + sum_j intra_j D_j
//   pref_j = eps_jj v_j Vbin / 2,  X_jk = eps_jk v_j Vbin (cross-talk),
//   intra_j = eps_jj (1 - v_j / Vbin),  phi_v = rho_v0 V,
//   g(phi) = chi (Vbin / V) phi^2  (phi <= vf_limit)  else 1e99 phi,
//   E_bind = sum_b sum_j [ F_j(marks, s) - s mu_j f ]  (mu_j > 0: - s mu_j (2 - f)).
//
// (The reference's own compute_E uses chi phi (1 - phi) and omits cross-talk,
// so its differences are not the move dE; chromo_energy_reference reproduces
// that function separately.)  Gradients: with respect to bead positions
// through the trilinear weights (dw/dx = -+1/dx) and the SSWLC bond energy, and
// with respect to theta = (chi, eps_ij for i <= j, mu_j).  Densities are
// recomputed rather than stored; every sum is exact or in a fixed order.
#include <hip/hip_runtime.h>

#include <math.h>
#include <stdint.h>
#include <string.h>

#include <mutex>
#include <string>
#include <type_traits>

#include "chromo_density.hpp"
#include "chromo_device.hpp"
#include "chromo_fixed.hpp"
#include "chromo_index.hpp"

using namespace chromo;

namespace {

constexpr int EB = 256;   // block size of the energy kernels
constexpr int MAXT = 64;  // partial-sum slots per block

int eset(int code, const std::string &m) { return chromo::set_last_error(code, m); }

#define HIPE(x)                                                                            \
    do {                                                                                   \
        hipError_t e_ = (x);                                                               \
        if (e_ != hipSuccess) return eset(-2, std::string(#x) + ": " + hipGetErrorString(e_)); \
    } while (0)

struct EModel {
    int64_t N;
    int B;
    int twist;
    GridGeom G;
    const double *t3;
    const int8_t *states, *marks;
    const double *bonds;
    double bead_vol, vf_limit, mu_adjust;
    double v_int[CHROMO_MAX_BINDERS];
    int cross_mask[CHROMO_MAX_BINDERS * CHROMO_MAX_BINDERS];
    double F[CHROMO_MAX_BINDERS][CHROMO_MAX_MARK][CHROMO_MAX_SITES + 1];
};

// theta layout: [chi, eps_00, eps_01, .., eps_0B-1, eps_11, .., eps_B-1B-1, mu_0 .. mu_B-1]
__host__ __device__ inline int eps_index(int B, int i, int j)
{
    if (i > j) {
        int t = i;
        i = j;
        j = t;
    }
    // rows 0..i-1 hold B, B-1, .. entries
    return 1 + i * B - (i * (i - 1)) / 2 + (j - i);
}

__host__ __device__ inline int n_theta(int B) { return 1 + B * (B + 1) / 2 + B; }

struct Coef {
    double chi;
    double pref[CHROMO_MAX_BINDERS], intra[CHROMO_MAX_BINDERS];
    double X[CHROMO_MAX_BINDERS * CHROMO_MAX_BINDERS];
    double mu[CHROMO_MAX_BINDERS];
};

__device__ inline Coef coef_of(const EModel &M, const double *th)
{
    Coef c;
    const int B = M.B;
    const double vb = M.G.vol_bin;
    c.chi = th[0];
    for (int j = 0; j < B; ++j) {
        double e = th[eps_index(B, j, j)];
        c.pref[j] = 0.5 * e * M.v_int[j] * vb;
        c.intra[j] = e * (1 - M.v_int[j] / vb);
        c.mu[j] = th[1 + B * (B + 1) / 2 + j];
        for (int k = 0; k < B; ++k)
            c.X[j * B + k] = M.cross_mask[j * B + k] ? th[eps_index(B, j, k)] * M.v_int[j] * vb : 0.0;
    }
    return c;
}

// coef_of for a binder count known at compile time: the same arithmetic, with
// constant indices (registers instead of scratch in the per-voxel and per-bead loops)
template <int B>
__device__ inline Coef coef_of(const EModel &M, const double *th)
{
    Coef c;
    const double vb = M.G.vol_bin;
    c.chi = th[0];
#pragma unroll
    for (int j = 0; j < B; ++j) {
        double e = th[eps_index(B, j, j)];
        c.pref[j] = 0.5 * e * M.v_int[j] * vb;
        c.intra[j] = e * (1 - M.v_int[j] / vb);
        c.mu[j] = th[1 + B * (B + 1) / 2 + j];
#pragma unroll
        for (int k = 0; k < B; ++k)
            c.X[j * B + k] = M.cross_mask[j * B + k] ? th[eps_index(B, j, k)] * M.v_int[j] * vb : 0.0;
    }
    return c;
}

// Block partials are stored term-major: part[t * gridDim.x + block], so that the
// final sums read each term's partials contiguously.

// Fixed-order block sum of NT partial values per thread: a butterfly within each
// wavefront, then the wavefront sums in wavefront order.
// SHARED: for another block of the same launch, past the caches of this block's die.
template <int NT, int THREADS = EB, bool SHARED = false>
__device__ void block_reduce_store(const double (&vals)[NT], double *part)
{
    __shared__ double sh[THREADS / 64][NT];
    const int wv = threadIdx.x / 64, lane = threadIdx.x % 64;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        double s = vals[t];
        for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
        if (lane == 0) sh[wv][t] = s;
    }
    __syncthreads();
    if ((int)threadIdx.x < NT) {
        double s = sh[0][threadIdx.x];
        for (int w = 1; w < THREADS / 64; ++w) s += sh[w][threadIdx.x];
        double *to = &part[(int64_t)threadIdx.x * gridDim.x + blockIdx.x];
        if (SHARED) __hip_atomic_store(to, s, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        else *to = s;
    }
}

// fixed-order block sum of nt partial values per thread
__device__ void block_reduce_store(double *vals, int nt, double *part)
{
    __shared__ double sh[EB];
    for (int t = 0; t < nt; ++t) {
        sh[threadIdx.x] = vals[t];
        __syncthreads();
        for (int s = EB / 2; s > 0; s >>= 1) {
            if ((int)threadIdx.x < s) sh[threadIdx.x] += sh[threadIdx.x + s];
            __syncthreads();
        }
        if (threadIdx.x == 0) part[(int64_t)t * gridDim.x + blockIdx.x] = sh[0];
        __syncthreads();
    }
}

// ---- field terms: densities, voxel energies, gradient at the beads ---------------
//
// The adjoint needs a deterministic density, not the reference's bead-order fold.
// Each corner weight becomes an integer of two words (chromo_fixed.hpp), and the words are
// summed in 64 bits each, times the binder state for the binder rows: the sums are exact,
// so they do not depend on the order in which the LDS takes them.  A voxel's total is
// rounded to double once and divided by its volume.

// Coefficients of the voxel terms in scalar registers: held in vector registers through
// the tile loop they spill.
template <int B>
struct VoxelCoef {
    double pref2[B], XX[B * B], gphi, dphi;
    __device__ __forceinline__ VoxelCoef(const EModel &M, const TileGeom &T, const double *theta)
    {
        const Coef c = coef_of<B>(M, theta);
        gphi = uni_f64(c.chi * T.vbV);
        dphi = uni_f64(2 * c.chi * T.vbV);
#pragma unroll
        for (int j = 0; j < B; ++j) {
            pref2[j] = uni_f64(2 * c.pref[j]);
#pragma unroll
            for (int k = 0; k < B; ++k) XX[j * B + k] = uni_f64(c.X[j * B + k] + c.X[k * B + j]);
        }
    }
};

// The sums of a tile or part: [species][low, high][voxel]; a voxel's dE/drho overwrites
// its low words.
// SIDE: places per axis, the tile's or part's voxels and their upper neighbours.
template <int B, int SIDE>
using TileSums = unsigned long long[B + 1][2][SIDE * SIDE * SIDE];
constexpr int TILE_SIDE = 9, PART_SIDE = 5;
static_assert(TILE_MAX[0] < TILE_SIDE && TILE_MAX[1] < TILE_SIDE && TILE_MAX[2] < TILE_SIDE &&
              (TILE_SIDE - 1 + 1) / 2 < PART_SIDE, "places of a tile and of half of one");

// A tile's or part's first voxels and sizes.
struct TileBox {
    int start[3], size[3];
};

// Whether X is all of axis j, wrapping onto itself.  (For a tile the same either way; this
// one keeps the tile kernel's registers in bounds.)
template <int SIDE>
__device__ __forceinline__ bool whole_axis(const TileGeom &T, const TileBox &X, int j)
{
    return SIDE == TILE_SIDE ? T.nt[j] == 1 : X.size[j] == T.n[j];
}

// Adds bead b's corner weights to the sums of the box X (its upper neighbours included).
// b's cell is inside X or a neighbour; note(whether inside).
template <int B, int SIDE, class F>
__device__ __forceinline__ void tile_add(const EModel &M, const TileGeom &T, const double *r, int32_t b,
                                         const TileBox &X, TileSums<B, SIDE> &sums, F note)
{
    double x[3], w[3];
    int ix[3];
#pragma unroll
    for (int j = 0; j < 3; ++j) x[j] = r[row3(b, j)];
    int st[B];
#pragma unroll
    for (int j = 0; j < B; ++j) st[j] = M.states[(int64_t)j * M.N + b];
    tile_lower(M.G, T, x, ix, w);
    int at[3][2];       // voxel place of the lower and upper corner, -1: not among these voxels
    bool own = true;
    const int stride[3] = {1, SIDE, SIDE * SIDE};
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        if (whole_axis<SIDE>(T, X, j)) {
            at[j][0] = ix[j] * stride[j];
            at[j][1] = (ix[j] + 1 == T.n[j] ? 0 : ix[j] + 1) * stride[j];
        } else {
            const int l = tile_local(T.n[j], X.start[j], X.size[j], ix[j]);
            own = own && l >= 0 && l < X.size[j];
            at[j][0] = l >= 0 ? l * stride[j] : -1;
            at[j][1] = l < X.size[j] ? (l + 1) * stride[j] : -1;
        }
    }
    note(own);
    // corner_weight's products, the last factor scaled
    const double ux = 1 - w[0], uy = 1 - w[1], uz = (1 - w[2]) * FIXED60_SCALE, wz = w[2] * FIXED60_SCALE;
    const double xy[4] = {w[0] * w[1], ux * w[1], w[0] * uy, ux * uy};
#pragma unroll
    for (int l = 0; l < 8; ++l) {
        const int vx = at[0][l & 1], vy = at[1][(l >> 1) & 1], vz = at[2][l >> 2];
        if ((vx | vy | vz) < 0) continue;
        const int v = vx + vy + vz;
        const Fixed60 f = fixed60(xy[l & 3] * ((l & 4) ? uz : wz));
        atomicAdd(&sums[0][0][v], (unsigned long long)(long long)f.lo);
        atomicAdd(&sums[0][1][v], (unsigned long long)f.hi);
#pragma unroll
        for (int j = 0; j < B; ++j) {
            if (st[j] != 0) {
                atomicAdd(&sums[j + 1][0][v], (unsigned long long)(long long)(f.lo * st[j]));
                atomicAdd(&sums[j + 1][1][v], (unsigned long long)(f.hi * (uint32_t)st[j]));
            }
        }
    }
}

// Densities, energy terms of the voxels of the tile or part itself, dE/drho in place.
// acc: [0..B) S_jj, [B..B+B(B-1)/2) S_jk (j<k), then sum g, sum dg/dchi.
template <int B, bool GRAD, int THREADS, int SIDE, int NT>
__device__ __forceinline__ void tile_voxels(const EModel &M, const TileGeom &T, const VoxelCoef<B> &c,
                                            const TileBox &X, TileSums<B, SIDE> &sums, double (&acc)[NT])
{
    constexpr int Bp1 = B + 1;
    const double V = M.bead_vol, vb = M.G.vol_bin;
    for (int v = threadIdx.x; v < SIDE * SIDE * SIDE; v += THREADS) {
        const int vx = v % SIDE, vy = (v / SIDE) % SIDE, vz = v / (SIDE * SIDE);
        double rho[Bp1];
#pragma unroll
        for (int j = 0; j < Bp1; ++j) {
            const double f = from_fixed60(sums[j][1][v], sums[j][0][v]);
            rho[j] = T.recip ? div_by(f, vb, T.rvol) : f / vb;
        }
        const double phi = rho[0] * V;
        const bool huge = phi > M.vf_limit;
        if (vx < X.size[0] && vy < X.size[1] && vz < X.size[2]) {
            int s = B;
#pragma unroll
            for (int j = 0; j < B; ++j) {
                acc[j] += rho[j + 1] * rho[j + 1];
#pragma unroll
                for (int k = j + 1; k < B; ++k) acc[s++] += rho[j + 1] * rho[k + 1];
            }
            acc[s] += huge ? E_HUGE_FIELD * phi : c.gphi * (phi * phi);
            acc[s + 1] += huge ? 0.0 : T.vbV * (phi * phi);
        }
        if (GRAD) {
            double d[Bp1];
            d[0] = V * (huge ? E_HUGE_FIELD : c.dphi * phi);
#pragma unroll
            for (int j = 0; j < B; ++j) {
                double g = c.pref2[j] * rho[j + 1];
#pragma unroll
                for (int k = 0; k < B; ++k) g += c.XX[j * B + k] * rho[k + 1];
                d[j + 1] = g;
            }
#pragma unroll
            for (int j = 0; j < Bp1; ++j) sums[j][0][v] = (unsigned long long)__double_as_longlong(d[j]);
        }
    }
}

// The field's gradient at bead b into grad (ADD: added to it), by the trilinear chain rule,
// when its cell is inside.
template <int B, int SIDE, bool ADD>
__device__ __forceinline__ void tile_gather(const EModel &M, const TileGeom &T, const double *r, int32_t b,
                                            const TileBox &X, const TileSums<B, SIDE> &sums, double *grad)
{
    double x[3], w[3];
    int ix[3];
#pragma unroll
    for (int j = 0; j < 3; ++j) x[j] = r[row3(b, j)];
    tile_lower(M.G, T, x, ix, w);
    int at[3][2];
    bool own = true;
    const int stride[3] = {1, SIDE, SIDE * SIDE};
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        const int l = ix[j] - X.start[j];
        own = own && l >= 0 && l < X.size[j];
        at[j][0] = l * stride[j];
        at[j][1] = (whole_axis<SIDE>(T, X, j) && l + 1 == X.size[j] ? 0 : l + 1) * stride[j];
    }
    if (!own) return;
    double st[B];
#pragma unroll
    for (int j = 0; j < B; ++j) st[j] = (double)M.states[(int64_t)j * M.N + b];
    // along x first: A the interpolated value, D the difference, for each
    // (y, z); then along y and z
    const double ux = 1 - w[0], uy = 1 - w[1], uz = 1 - w[2], vb = M.G.vol_bin;
    double A[4], D[4], g[3];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        double h[2];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const int v = at[0][e] + at[1][q & 1] + at[2][q >> 1];
            h[e] = __longlong_as_double((long long)sums[0][0][v]);
#pragma unroll
            for (int j = 0; j < B; ++j) h[e] += st[j] * __longlong_as_double((long long)sums[j + 1][0][v]);
        }
        A[q] = w[0] * h[0] + ux * h[1];
        D[q] = h[1] - h[0];
    }
    g[0] = (w[2] * (w[1] * D[0] + uy * D[1]) + uz * (w[1] * D[2] + uy * D[3])) * T.rd[0];
    g[1] = (w[2] * (A[1] - A[0]) + uz * (A[3] - A[2])) * T.rd[1];
    g[2] = ((w[1] * A[2] + uy * A[3]) - (w[1] * A[0] + uy * A[1])) * T.rd[2];
#pragma unroll
    for (int j = 0; j < 3; ++j) g[j] = T.recip ? div_by(g[j], vb, T.rvol) : g[j] / vb;
#pragma unroll
    for (int j = 0; j < 3; ++j) grad[row3(b, j)] = ADD ? grad[row3(b, j)] + g[j] : g[j];
}

__device__ __forceinline__ TileBox tile_box(const TileGeom &T, int tile)
{
    const int tt[3] = {tile % T.nt[0], (tile / T.nt[0]) % T.nt[1], tile / (T.nt[0] * T.nt[1])};
    TileBox X;
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        X.start[j] = tile_start(T.n[j], T.nt[j], tt[j]);
        X.size[j] = tile_start(T.n[j], T.nt[j], tt[j] + 1) - X.start[j];
    }
    return X;
}

// Cell c of the grid, by axis.
__device__ __forceinline__ void cell_axes(const TileGeom &T, int32_t cell, int ix[3])
{
    const uint32_t c = (uint32_t)cell, q = c / (uint32_t)T.n[0];
    ix[0] = (int)(c - q * (uint32_t)T.n[0]);
    ix[1] = (int)(q % (uint32_t)T.n[1]);
    ix[2] = (int)(q / (uint32_t)T.n[1]);
}

// The tiles whose lists are not split.  Block partials: tile_voxels' acc.
template <int B, bool GRAD>
__global__ void __launch_bounds__(TILE_THREADS, 4)
k_e_tile(EModel M, TileGeom T, const double *theta, const double *r, TileCounters C, const ListPlace *base,
         const int32_t *list, LongTiles L, double *grad, double *part)
{
    constexpr int NT = B + B * (B - 1) / 2 + 2;
    __shared__ TileSums<B, TILE_SIDE> sums;
    __shared__ int32_t owned[TILE_OWN], nown;
    const int t = threadIdx.x;
    double acc[NT];
#pragma unroll
    for (int q = 0; q < NT; ++q) acc[q] = 0;
    const VoxelCoef<B> c(M, T, theta);
    const int32_t most = split_above(C, L);
    for (int tile = blockIdx.x; tile < T.ntiles; tile += gridDim.x) {
        const TileBox X = tile_box(T, tile);
        uint32_t len = (uint32_t)C.cnt[tile];
        if (len > (uint32_t)most) len = 0;      // as if it were empty: tile_parts does it
        const int32_t *mine = list + base[tile];
        for (int i = t; i < (int)(sizeof(sums) / 8); i += TILE_THREADS) (&sums[0][0][0])[i] = 0;
        if (t == 0) nown = 0;
        __syncthreads();
        // the beads' corner weights.  Lists hold runs of the chain, whose neighbours share
        // voxels: the lanes of a wavefront take entries far apart, so that their adds
        // meet different voxels
        const uint32_t per = (len + TILE_THREADS - 1) / TILE_THREADS;
        for (uint32_t k = 0; k < per; ++k) {
            const uint32_t i = (uint32_t)((t & 63) * (TILE_THREADS / 64) + (t >> 6)) * per + k;
            if (i >= len) continue;
            const int32_t b = mine[i];
            tile_add<B, TILE_SIDE>(M, T, r, b, X, sums, [&](bool own) {
                if (GRAD && own) {
                    const int o = atomicAdd(&nown, 1);
                    if (o < TILE_OWN) owned[o] = b;
                }
            });
        }
        __syncthreads();
        // densities, energy terms of the tile's own voxels, dE/drho in place
        tile_voxels<B, GRAD, TILE_THREADS, TILE_SIDE>(M, T, c, X, sums, acc);
        __syncthreads();
        if (GRAD) {
            // trilinear chain rule at the beads of the tile's own cells
            const uint32_t no = (uint32_t)nown;
            const bool noted = no <= (uint32_t)TILE_OWN;
            for (uint32_t i = (uint32_t)t; i < (noted ? no : len); i += TILE_THREADS) {
                const int32_t b = noted ? owned[i] : mine[i];
                tile_gather<B, TILE_SIDE, false>(M, T, r, b, X, sums, grad);
            }
            __syncthreads();
        }
    }
    block_reduce_store<NT, TILE_THREADS>(acc, part);
}

// LDS of tile_parts.
template <int B>
struct PartLds {
    TileSums<B, PART_SIDE> sums;
    int32_t picked[PART_NOTES], npicked;    // beads near the part
    int32_t owned[PART_NOTES], nowned;      // those in its cells
    int32_t longs[LONG_GROUPS], nlong;      // long lists before each group of tiles, in all
};

// The tiles with long lists, each in 8 parts (halves per axis), one block per part: a
// block picks its beads from the tile's list.  Adds the field's gradient to grad; writes
// tile_voxels' sums to part, past the caches of this block's die.
// A condensed chain fills few tiles, and one block per tile left most of the chip idle, the
// others bound by their compute unit's LDS adds.  10^6 beads at 25 per voxel, B = 4, 128^3:
// 744 -> 461 us an evaluation; 100,000 in 16^3 voxels of 64^3, B = 2: 237 -> 133 us.  What
// bounds it: the adds still (a part lists 3.4 beads per own bead), and picking.
template <int B, bool GRAD>
__device__ __forceinline__ void tile_parts(const EModel &M, const TileGeom &T, const double *theta, const double *r,
                                           const int32_t *cell, const int32_t *cnt, const ListPlace *base,
                                           const int32_t *list, const LongTiles &L, double *grad, double *part,
                                           PartLds<B> &S)
{
    constexpr int NT = B + B * (B - 1) / 2 + 2, SCAN = PART_SCAN;
    const int t = threadIdx.x;
    double acc[NT];
#pragma unroll
    for (int q = 0; q < NT; ++q) acc[q] = 0;
    const VoxelCoef<B> c(M, T, theta);
    const int groups = (T.ntiles + LONG_GROUP - 1) / LONG_GROUP;
    if (t < WAVE) {
        int sum = 0;
        for (int g0 = 0; g0 < groups; g0 += WAVE) {
            int all;
            const int g = g0 + t, below = wave_excl_scan(g < groups ? L.count[g] : 0, all);
            if (g < groups) S.longs[g] = sum + below;
            sum += all;
        }
        if (t == 0) S.nlong = sum;
    }
    __syncthreads();
    const int nlong = uni_i32(S.nlong);
    for (int item = blockIdx.x; item < nlong * TILE_PARTS; item += gridDim.x) {
        const int h = item / TILE_PARTS;
        int lo = 0, hi = groups;
        while (hi - lo > 1) {
            const int mid = (lo + hi) >> 1;
            if (uni_i32(S.longs[mid]) <= h) lo = mid;
            else hi = mid;
        }
        const int tile = uni_i32(L.tile[LONG_GROUP * lo + (h - uni_i32(S.longs[lo]))]);
        TileBox X = tile_box(T, tile);
#pragma unroll
        for (int j = 0; j < 3; ++j) tile_half((item >> j) & 1, X.start[j], X.size[j]);
        if (X.size[0] == 0 || X.size[1] == 0 || X.size[2] == 0) continue;
        const uint32_t len = (uint32_t)cnt[tile];
        const int32_t *mine = list + base[tile];
        for (int i = t; i < (int)(sizeof(S.sums) / 8); i += PART_THREADS) (&S.sums[0][0][0])[i] = 0;
        if (t == 0) S.npicked = S.nowned = 0;
        __syncthreads();
        // picks beads from entry `from` of the list on, as many as S.picked[] surely holds;
        // returns the entry after them.  near: those near the part, of which those in its
        // cells are noted in S.owned[] while there is room; else those in its cells.
        auto pick = [&](uint32_t from, bool near) {
            static_assert(PART_NOTES >= 2 * SCAN * PART_THREADS, "two steps fit");
            for (;;) {
                int32_t bead[SCAN], at[SCAN];
#pragma unroll
                for (int q = 0; q < SCAN; ++q) {
                    const uint32_t i = from + (uint32_t)(q * PART_THREADS + t);
                    bead[q] = i < len ? mine[i] : -1;
                }
#pragma unroll
                for (int q = 0; q < SCAN; ++q) at[q] = bead[q] >= 0 ? cell[bead[q]] : 0;
#pragma unroll
                for (int q = 0; q < SCAN; ++q) {
                    int ix[3];
                    cell_axes(T, at[q], ix);
                    bool is = bead[q] >= 0, own = is;
#pragma unroll
                    for (int j = 0; j < 3; ++j) {
                        is = is && tile_near(T.n[j], X.start[j], X.size[j], ix[j]);
                        own = own && ix[j] >= X.start[j] && ix[j] < X.start[j] + X.size[j];
                    }
                    if (near ? is : own) S.picked[atomicAdd(&S.npicked, 1)] = bead[q];
                    if (GRAD && near && own) {
                        const int o = atomicAdd(&S.nowned, 1);
                        if (o < PART_NOTES) S.owned[o] = bead[q];
                    }
                }
                from += SCAN * PART_THREADS;
                __syncthreads();
                const int n = uni_i32(S.npicked);
                // nobody adds to S.npicked before everybody has read it
                __syncthreads();
                if (from >= len || n > PART_NOTES - SCAN * PART_THREADS) return from;
            }
        };
        for (uint32_t from = 0; from < len;) {
            from = pick(from, true);
            const uint32_t n = (uint32_t)uni_i32(S.npicked), per = (n + PART_THREADS - 1) / PART_THREADS;
            for (uint32_t k = 0; k < per; ++k) {
                const uint32_t i = (uint32_t)((t & 63) * (PART_THREADS / 64) + (t >> 6)) * per + k;
                if (i < n) tile_add<B, PART_SIDE>(M, T, r, S.picked[i], X, S.sums, [](bool) {});
            }
            __syncthreads();
            if (t == 0) S.npicked = 0;
            __syncthreads();
        }
        tile_voxels<B, GRAD, PART_THREADS, PART_SIDE>(M, T, c, X, S.sums, acc);
        __syncthreads();
        if (!GRAD) continue;
        const uint32_t no = (uint32_t)uni_i32(S.nowned);
        if (no <= (uint32_t)PART_NOTES) {
            for (uint32_t i = (uint32_t)t; i < no; i += PART_THREADS)
                tile_gather<B, PART_SIDE, true>(M, T, r, S.owned[i], X, S.sums, grad);
        } else {
            for (uint32_t from = 0; from < len;) {
                from = pick(from, false);
                const uint32_t n = (uint32_t)uni_i32(S.npicked);
                for (uint32_t i = (uint32_t)t; i < n; i += PART_THREADS)
                    tile_gather<B, PART_SIDE, true>(M, T, r, S.picked[i], X, S.sums, grad);
                __syncthreads();
                if (t == 0) S.npicked = 0;
                __syncthreads();
            }
        }
        __syncthreads();
    }
    block_reduce_store<NT, PART_THREADS, true>(acc, part);
}

// ---- bead / bond terms -------------------------------------------------------
// Elastic energy of bond (r0, t30) -> (r1, t31), and (grad) its derivative with
// respect to r1 - r0 with the tangents fixed, from the same intermediates.
__device__ inline double E_pair_and_grad(const Bond &bd, const double *r0, const double *r1, const double *t30,
                                         const double *t31, bool grad, double g[3])
{
    double dr[3], drp[3], be[3];
    for (int i = 0; i < 3; ++i) dr[i] = r1[i] - r0[i];
    double par = dot3(t30, dr);
    for (int i = 0; i < 3; ++i) {
        drp[i] = dr[i] - t30[i] * par;
        be[i] = t31[i] - t30[i] - drp[i] * bd.eta;
    }
    if (grad) {
        // perp = P dr with P = I - t t^T; bend = t31 - t30 - eta perp
        double a[3];
        for (int i = 0; i < 3; ++i) a[i] = bd.eperp * drp[i] - bd.eta * bd.eb * be[i];
        double ta = dot3(t30, a);
        for (int i = 0; i < 3; ++i) g[i] = (a[i] - t30[i] * ta) + bd.ep * (par - bd.gam) * t30[i];
    }
    return E_pair(bd, be, par, drp);
}

// slots: [0] E_elastic, [1] E_bind, [2..2+B) D_j, [2+B..2+2B) sum s_j
// grad: the field's gradient on entry (k_e_tile), with the bonds' on return.
template <int B>
__global__ void __launch_bounds__(EB) k_e_bead(EModel M, const double *theta, const double *r, double *grad,
                                               double *part)
{
    constexpr int NT = 2 + 2 * B;
    const int64_t N = M.N;
    const Coef c = coef_of<B>(M, theta);
    double acc[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[t] = 0;
    const double f = M.mu_adjust;
    // bond i = (i, i + 1): each is evaluated once, by thread i - b0 of the block
    // that holds bead i (the block's first bond (b0 - 1, b0) by its last thread);
    // the derivatives meet in LDS, where beads b and b + 1 read them
    __shared__ double gbond[EB + 1][3];
    const int t = threadIdx.x;
    for (int64_t b0 = (int64_t)blockIdx.x * EB; b0 < N; b0 += (int64_t)gridDim.x * EB) {
        const int64_t b = b0 + t;
        const double *rb = r + 3 * b;
        const double *tb = M.t3 + 3 * b;
        double g[3] = {0, 0, 0};
        if (grad && b < N)
            for (int j = 0; j < 3; ++j) g[j] = grad[3 * b + j];
        if (b + 1 < N) {
            Bond bd = load_bond(M.bonds, N, b);
            double gd[3];
            acc[0] += E_pair_and_grad(bd, rb, r + 3 * (b + 1), tb, M.t3 + 3 * (b + 1), grad != nullptr, gd);
            if (grad)
                for (int j = 0; j < 3; ++j) gbond[t + 1][j] = gd[j];
        }
        if (grad && t == EB - 1 && b0 > 0) {
            Bond bd = load_bond(M.bonds, N, b0 - 1);
            double gd[3];
            E_pair_and_grad(bd, r + 3 * (b0 - 1), r + 3 * b0, M.t3 + 3 * (b0 - 1), M.t3 + 3 * b0, true, gd);
            for (int j = 0; j < 3; ++j) gbond[0][j] = gd[j];
        }
        if (b < N) {
#pragma unroll
            for (int j = 0; j < B; ++j) {
                const int s = M.states[(int64_t)j * N + b];
                int m = M.marks[(int64_t)j * N + b];
                double mu = c.mu[j];
                double e = M.F[j][m][s];
                e += (mu > 0) ? -(double)s * (mu * (2 - f)) : -(double)s * mu * f;
                acc[1] += e;
                acc[2 + j] += (s == 2);
                acc[2 + B + j] += (double)s * ((mu > 0) ? (2 - f) : f);
            }
        }
        if (grad) {
            // every thread of the block reaches both barriers
            __syncthreads();
            if (b < N) {
                if (b + 1 < N)   // bond (b, b+1): r0 = r_b
                    for (int j = 0; j < 3; ++j) g[j] -= gbond[t + 1][j];
                if (b > 0)       // bond (b-1, b): r1 = r_b
                    for (int j = 0; j < 3; ++j) g[j] += gbond[t][j];
                for (int j = 0; j < 3; ++j) grad[3 * b + j] = g[j];
            }
            __syncthreads();
        }
    }
    block_reduce_store<NT>(acc, part);
}

// Sums of the block partials of ntv voxel terms and ntb bead terms, by one block of W
// wavefronts: wavefront w takes terms w, w + W, ...; lane i adds partials i,
// i + 64, ... in increasing order (loaded 16 at a time, so that one round trip
// covers 16 of them), then a butterfly over the 64 lanes.  The order depends on
// the sizes only, so the sums are the same on every run.
// SHARED: partials that other blocks of the same launch wrote.
constexpr int FINAL_THREADS = 1024;
constexpr int FINAL_READ = 1024;    // partials of a term that one round trip covers

template <int THREADS = FINAL_THREADS, bool SHARED = false>
__device__ void final_sums(const double *vpart, int nbv, int ntv, const double *bpart, int nbb, int ntb,
                           double *sv, double *sb)
{
    const int wv = threadIdx.x / 64, lane = threadIdx.x % 64;
    for (int q = wv; q < ntv + ntb; q += THREADS / 64) {
        const bool vox = q < ntv;
        const double *p = vox ? vpart : bpart;
        const int nbk = vox ? nbv : nbb, t = vox ? q : q - ntv;
        double s = 0;
        for (int i0 = lane; i0 < nbk; i0 += 64 * 16) {
            double x[16];
#pragma unroll
            for (int j = 0; j < 16; ++j) {
                const int i = i0 + 64 * j;
                const double *at = p + ((int64_t)t * nbk + i);
                if (SHARED) x[j] = i < nbk ? __hip_atomic_load(at, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0.0;
                else x[j] = i < nbk ? *at : 0.0;
            }
#pragma unroll
            for (int j = 0; j < 16; ++j)
                if (i0 + 64 * j < nbk) s += x[j];
        }
        for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
        if (lane == 0) (vox ? sv : sb)[t] = s;
    }
    __syncthreads();
}

// The energies and dE/dtheta from the sums, for B binders (compile-time, so the
// coefficients and sums stay in registers), by one thread.
template <int B>
__device__ __forceinline__ void assemble(const EModel &M, const double *theta, const double *sv, const double *sb,
                                         double *E_out, double *gtheta)
{
    const Coef c = coef_of<B>(M, theta);
    const double vb = M.G.vol_bin;
    double S[CHROMO_MAX_BINDERS * CHROMO_MAX_BINDERS];
    int s = B;
#pragma unroll
    for (int j = 0; j < B; ++j) {
        S[j * B + j] = sv[j];
#pragma unroll
        for (int k = j + 1; k < B; ++k) {
            S[j * B + k] = sv[s];
            S[k * B + j] = sv[s];
            ++s;
        }
    }
    const double Eg = sv[s], dchi = sv[s + 1];
    double Ef = 0;
#pragma unroll
    for (int j = 0; j < B; ++j) {
        Ef += c.pref[j] * S[j * B + j];
        Ef += c.intra[j] * sb[2 + j];
#pragma unroll
        for (int k = 0; k < B; ++k) Ef += c.X[j * B + k] * S[j * B + k];
    }
    Ef += Eg;
    const double Eel = sb[0], Ebd = sb[1];
    E_out[0] = Eel + Ef + Ebd;
    E_out[1] = Eel;
    E_out[2] = Ef;
    E_out[3] = Ebd;
    if (gtheta) {
        gtheta[0] = dchi;
#pragma unroll
        for (int j = 0; j < B; ++j)
#pragma unroll
            for (int k = j; k < B; ++k) {
                double g;
                if (j == k) {
                    g = 0.5 * M.v_int[j] * vb * S[j * B + j] + (1 - M.v_int[j] / vb) * sb[2 + j];
                    if (M.cross_mask[j * B + j]) g += M.v_int[j] * vb * S[j * B + j];
                } else {
                    g = ((M.cross_mask[j * B + k] ? M.v_int[j] : 0.0) +
                         (M.cross_mask[k * B + j] ? M.v_int[k] : 0.0)) * vb * S[j * B + k];
                }
                gtheta[eps_index(B, j, k)] = g;
            }
#pragma unroll
        for (int j = 0; j < B; ++j) gtheta[1 + B * (B + 1) / 2 + j] = -sb[2 + B + j];
    }
}

// Final reduction over block partials (fixed order) and assembly.
template <int B>
__global__ void __launch_bounds__(FINAL_THREADS)
k_e_final(EModel M, const double *theta, const double *vpart, int nbv, int ntv, const double *bpart, int nbb,
          int ntb, double *E_out, double *gtheta)
{
    __shared__ double sv[MAXT], sb[MAXT];
    final_sums(vpart, nbv, ntv, bpart, nbb, ntb, sv, sb);
    if (threadIdx.x == 0) assemble<B>(M, theta, sv, sb, E_out, gtheta);
}

// The same where lists may have to be split.  If they are, all blocks of the launch work on
// those tiles first, and the last one done goes on; otherwise all but the first have
// nothing to do.  (A launch of their own would cost every evaluation 4 us.  This costs 1.5
// of 55 us at 100,000 beads, nothing measurable at 10^6.)
template <int B, bool GRAD>
__global__ void __launch_bounds__(PART_THREADS, 4)
k_e_split(EModel M, TileGeom T, const double *theta, const double *r, const int32_t *cell, TileCounters C,
          const ListPlace *base, const int32_t *list, LongTiles L, double *grad, double *lpart, const double *vpart,
          int nbv, int ntv, const double *bpart, int nbb, int ntb, double *E_out, double *gtheta)
{
    __shared__ double sv[MAXT], sb[MAXT], sl[MAXT];
    __shared__ PartLds<B> lds;
    __shared__ int32_t ticket;
    const bool split = uni_i32(*C.split) != 0;
    if (split) {
        tile_parts<B, GRAD>(M, T, theta, r, cell, C.cnt, base, list, L, grad, lpart, lds);
        // this block's partials have arrived before its ticket is drawn
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (threadIdx.x == 0)
            ticket = __hip_atomic_fetch_add(C.ticket, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();
        if (ticket != (int)gridDim.x - 1) return;
        final_sums<PART_THREADS, true>(lpart, (int)gridDim.x, ntv, nullptr, 0, 0, sl, nullptr);
    } else if (blockIdx.x != 0) {
        return;
    }
    final_sums<PART_THREADS>(vpart, nbv, ntv, bpart, nbb, ntb, sv, sb);
    if (threadIdx.x != 0) return;
    if (split)
        for (int q = 0; q < ntv; ++q) sv[q] += sl[q];
    assemble<B>(M, theta, sv, sb, E_out, gtheta);
}

// ---- the reference's compute_E (fields.pyx:1939-2286, polymers.pyx:1348-1381) ----

// Python round(x, 2) > lim, evaluated on the exact binary value of x.
__device__ inline double py_round2(double x)
{
    double p = x * 100.0;
    double e = fma(x, 100.0, -p);   // exact residual: x * 100 = p + e
    double k = rint(p);
    double d = p - k;
    if (d == 0.5 && e > 0) k += 1.0;
    else if (d == -0.5 && e < 0) k -= 1.0;
    return k / 100.0;
}

// slots: [0..B) sum rho_j^2, [B] nonspecific E
__global__ void k_ref_voxel(EModel M, const double *pref, double chi, const double *rho, double *part,
                            int nt)
{
    const int B = M.B, Bp1 = B + 1;
    const int64_t nb = M.G.nx * M.G.ny * M.G.nz;
    double acc[MAXT];
    for (int t = 0; t < nt; ++t) acc[t] = 0;
    const double V = M.bead_vol, vb = M.G.vol_bin;
    for (int64_t v = (int64_t)blockIdx.x * EB + threadIdx.x; v < nb; v += (int64_t)gridDim.x * EB) {
        const double *r = rho + v * Bp1;
        for (int j = 0; j < B; ++j) acc[j] += r[j + 1] * r[j + 1];
        double vf = r[0] * V;
        if (py_round2(vf) > M.vf_limit) acc[B] += E_HUGE_FIELD * vf;
        else acc[B] += chi * (vb / V) * vf * (1 - vf);
    }
    block_reduce_store(acc, nt, part);
}

// slots: [0] SSWLC.compute_E bonds (SSTWLC.compute_E with the twist term), [1..1+B)
// doubly bound counts
__global__ void k_ref_bead(EModel M, const double *pos, int64_t sc, int64_t sb, double *part, int nt)
{
    const int B = M.B;
    const int64_t N = M.N;
    double acc[MAXT];
    for (int t = 0; t < nt; ++t) acc[t] = 0;
    for (int64_t b = (int64_t)blockIdx.x * EB + threadIdx.x; b < N; b += (int64_t)gridDim.x * EB) {
        if (b + 1 < N) {
            double r0[3], r1[3], t30[3], t31[3];
            for (int j = 0; j < 3; ++j) {
                r0[j] = pos[j * sc + b * sb];
                r1[j] = pos[j * sc + (b + 1) * sb];
                t30[j] = pos[(3 + j) * sc + b * sb];
                t31[j] = pos[(3 + j) * sc + (b + 1) * sb];
            }
            Bond bd = load_bond(M.bonds, N, b);
            double dr[3], drp[3], be[3];
            for (int j = 0; j < 3; ++j) dr[j] = r1[j] - r0[j];
            double par = dot3(t30, dr);
            for (int j = 0; j < 3; ++j) drp[j] = dr[j] - t30[j] * par;
            for (int j = 0; j < 3; ++j) {   // bend = t3_1; bend += -t3_0 - eta dr_perp
                be[j] = t31[j];
                be[j] += -t30[j] - bd.eta * drp[j];
            }
            double tw = 0;
            if (M.twist) {
                double t20[3], t21[3], et, tw0;
                for (int j = 0; j < 3; ++j) {
                    t20[j] = pos[(6 + j) * sc + b * sb];
                    t21[j] = pos[(6 + j) * sc + (b + 1) * sb];
                }
                load_twist(M.bonds, N, b, et, tw0);
                tw = twist_energy(et, tw0, twist_omega(t20, t30, t21, t31));
            }
            acc[0] += E_pair(bd, be, par, drp) + tw;
        }
        for (int j = 0; j < B; ++j) acc[1 + j] += (M.states[(int64_t)j * N + b] == 2);
    }
    block_reduce_store(acc, nt, part);
}

__global__ void __launch_bounds__(FINAL_THREADS)
k_ref_final(EModel M, const double *pref, const double *intra, const double *vpart, int nbv,
            const double *bpart, int nbb, double *out)
{
    __shared__ double sv[MAXT], sb[MAXT];
    const int B = M.B;
    final_sums(vpart, nbv, B + 1, bpart, nbb, B + 1, sv, sb);
    if (threadIdx.x != 0) return;
    double E = 0;
    for (int i = 0; i < B; ++i) {
        E += pref[i] * sv[i];
        E += intra[i] * sb[1 + i];
    }
    E += sv[B];
    out[0] = sb[0];
    out[1] = E;
}

// Blocks of a voxel or bead kernel: at most 2048 (eight waves per SIMD of the
// device), so that the final sums read few partials per term.
int grid_blocks(int64_t n)
{
    int64_t g = (n + EB - 1) / EB;
    if (g > 2048) g = 2048;
    if (g < 1) g = 1;
    return (int)g;
}

int make_model(const chromo_energy_model *m, EModel &M)
{
    if (m == nullptr) return eset(-1, "model is NULL");
    if (m->B < 1 || m->B > CHROMO_MAX_BINDERS) return eset(-1, "B outside 1..4");
    if (m->N < 2) return eset(-1, "N < 2");
    // the scatter stores bead indices as int32 and uses 0x7fffffff as its empty marker
    if (m->N >= 0x7fffffffLL) return eset(-1, "N must be below 2^31 - 1");
    if (n_theta(m->B) > MAXT || 2 + 2 * m->B > MAXT) return eset(-1, "too many terms");
    M.N = m->N;
    M.B = m->B;
    M.twist = m->twist != 0;
    M.G.nx = m->nx;
    M.G.ny = m->ny;
    M.G.nz = m->nz;
    const double W[3] = {m->x_width, m->y_width, m->z_width};
    const int64_t n[3] = {m->nx, m->ny, m->nz};
    for (int j = 0; j < 3; ++j) {
        M.G.width[j] = W[j];
        M.G.dxyz[j] = W[j] / (double)n[j];
        M.G.half_width[j] = 0.5 * W[j];
        M.G.half_step[j] = 0.5 * M.G.dxyz[j];
    }
    M.G.vol_bin = m->x_width * m->y_width * m->z_width / (double)(m->nx * m->ny * m->nz);
    M.t3 = m->t3;
    M.states = m->states;
    M.marks = m->marks;
    M.bonds = m->bonds;
    M.bead_vol = m->bead_vol;
    M.vf_limit = m->vf_limit;
    M.mu_adjust = m->mu_adjust;
    for (int j = 0; j < CHROMO_MAX_BINDERS; ++j) M.v_int[j] = m->v_int[j];
    for (int j = 0; j < CHROMO_MAX_BINDERS * CHROMO_MAX_BINDERS; ++j) M.cross_mask[j] = 0;
    for (int j = 0; j < m->B; ++j)
        for (int k = 0; k < m->B; ++k) M.cross_mask[j * m->B + k] = m->cross_mask[j * CHROMO_MAX_BINDERS + k];
    memcpy(M.F, m->F, sizeof(M.F));
    int64_t nb = m->nx * m->ny * m->nz;
    if (nb < 1 || nb > 2048LL * 2048LL) return eset(-1, "grid size outside 1..2^22 voxels");
    return 0;
}

// make_model and the argument checks of the energy adjoint's entry points.
int make_adjoint_model(const chromo_energy_model *m, const double *d_r, const double *d_theta, const double *d_E,
                       EModel &M)
{
    const int rc = make_model(m, M);
    if (rc) return rc;
    if (M.twist) return eset(-1, "the energy adjoint has no twist term (SSTWLC)");
    if (!d_r || !d_theta || !d_E) return eset(-1, "NULL argument");
    return 0;
}

// Device buffers of one evaluation of the reference energies, carved from one
// allocation.
struct EnergyBufs {
    ScatterJob J;
    double *vpart = nullptr, *bpart = nullptr;
    int gv = 0, gb = 0;
};

// Carves the buffers of an evaluation of M from base (nullptr: sizes only) and
// returns the bytes used.  rho: the caller's density array, or nullptr: one of its own.
size_t energy_carve(const EModel &M, const PosView &P, double *rho, char *base, EnergyBufs &Bf)
{
    const int64_t nb = M.G.nx * M.G.ny * M.G.nz;
    const int Bp1 = M.B + 1;
    // UniformDensityField.update_all_densities: no 1e-18 clean-up
    Bf.J = scatter_job(M.G, M.N, Bp1, P, M.states, rho, 0);
    size_t o = scatter_carve(Bf.J, base);
    auto take = [&](size_t bytes) {
        double *p = base ? (double *)(base + o) : nullptr;
        o = align_scratch(o + bytes);
        return p;
    };
    Bf.gv = grid_blocks(nb);
    Bf.gb = grid_blocks(M.N);
    if (!rho) Bf.J.density = take(sizeof(double) * nb * Bp1);
    Bf.vpart = take(sizeof(double) * MAXT * Bf.gv);
    Bf.bpart = take(sizeof(double) * MAXT * Bf.gb);
    return o;
}

// Where lists are split (tile_parts), the long ones: more than 1/512 of all entries (about
// two per bead), so that one block would be at it when the others are done; and, where
// there are tiles for every block, more than two and a half times the mean, so that a grid
// that is full everywhere is not split.  They are where one list holds `huge` beads:
// splitting costs 30 to 60 us beside the tile kernel's time for the lists below that
// (20,000 beads in 9^3 voxels: 92 us with or without, 150 us split from 4,096 on).
// Short chains' never are: looking for long lists costs 1.5 us of 49.
void long_list(int64_t N, int64_t ntiles, LongTiles &L)
{
    constexpr int64_t NONE = 0x7fffffff;
    int64_t most = LONG_LIST;
    if (most < N / 256) most = N / 256;
    if (ntiles >= PART_BLOCKS && most < 5 * N / ntiles) most = 5 * N / ntiles;
    int64_t huge = 2 * most > HUGE_LIST ? 2 * most : HUGE_LIST;
    if (N <= SPLIT_MIN) most = huge = NONE;
    L.most = (int32_t)(most < NONE ? most : NONE);
    L.huge = (int32_t)(huge < NONE ? huge : NONE);
}

// The same for the energy and its adjoint: the tiles' lists and the block partials.
struct AdjointBufs {
    TileCounters C{};
    int32_t *cell = nullptr, *list = nullptr;
    ListPlace *base = nullptr;
    LongTiles longs{};
    double *vpart = nullptr, *bpart = nullptr, *lpart = nullptr;
    int gt = 0, gb = 0, gl = 0;     // blocks of k_e_tile, k_e_bead, k_e_split (0: not used)
};

size_t adjoint_carve(const EModel &M, const TileGeom &T, char *base, AdjointBufs &Bf)
{
    size_t o = 0;
    auto take = [&](size_t bytes) {
        char *p = base ? base + o : nullptr;
        o = align_scratch(o + bytes);
        return p;
    };
    Bf.gt = T.ntiles < TILE_BLOCKS ? T.ntiles : TILE_BLOCKS;
    Bf.gb = grid_blocks(M.N) < FINAL_READ ? grid_blocks(M.N) : FINAL_READ;
    Bf.C.n = T.ntiles;
    Bf.C.cnt = (int32_t *)take(sizeof(int32_t) * T.ntiles);
    Bf.C.fill = (int32_t *)take(sizeof(int32_t) * T.ntiles);
    Bf.base = (ListPlace *)take(sizeof(ListPlace) * T.ntiles);
    Bf.C.cursor = (ListPlace *)take(sizeof(ListPlace));
    Bf.cell = (int32_t *)take(sizeof(int32_t) * M.N);
    Bf.list = (int32_t *)take(sizeof(int32_t) * M.N * tile_images(T));
    Bf.vpart = (double *)take(sizeof(double) * MAXT * Bf.gt);
    Bf.bpart = (double *)take(sizeof(double) * MAXT * Bf.gb);
    const size_t groups = (size_t)((T.ntiles + LONG_GROUP - 1) / LONG_GROUP);
    Bf.longs.tile = (int32_t *)take(sizeof(int32_t) * LONG_GROUP * groups);
    Bf.longs.count = (int32_t *)take(sizeof(int32_t) * groups);
    Bf.C.split = (int32_t *)take(sizeof(int32_t));
    Bf.C.ticket = (int32_t *)take(sizeof(int32_t));
    long_list(M.N, T.ntiles, Bf.longs);
    // (all lists hold about two entries per bead)
    const int64_t parts = TILE_PARTS * (2 * M.N / Bf.longs.most + 1);
    Bf.gl = M.N <= SPLIT_MIN ? 0 : (parts < PART_BLOCKS ? (int)parts : PART_BLOCKS);
    Bf.lpart = (double *)take(sizeof(double) * MAXT * Bf.gl);
    return o;
}

// One allocation (stream-ordered) freed on every return path.
struct StreamBuffer {
    char *p = nullptr;
    hipStream_t st = nullptr;
    ~StreamBuffer()
    {
        if (p) (void)hipFreeAsync(p, st);
    }
};

template <int B>
void launch_adjoint(const EModel &M, const TileGeom &T, const double *r, const double *theta, double *E, double *grad,
                    double *gtheta, const AdjointBufs &Bf, hipStream_t st)
{
    const auto go = [&](auto GRAD) {
        constexpr bool G = decltype(GRAD)::value;
        hipLaunchKernelGGL((k_e_tile<B, G>), dim3(Bf.gt), dim3(TILE_THREADS), 0, st, M, T, theta, r, Bf.C, Bf.base,
                           Bf.list, Bf.longs, grad, Bf.vpart);
        hipLaunchKernelGGL(k_e_bead<B>, dim3(Bf.gb), dim3(EB), 0, st, M, theta, r, grad, Bf.bpart);
        constexpr int NV = B + B * (B - 1) / 2 + 2, NB = 2 + 2 * B;
        if (Bf.gl == 0)
            hipLaunchKernelGGL(k_e_final<B>, dim3(1), dim3(FINAL_THREADS), 0, st, M, theta, Bf.vpart, Bf.gt, NV, Bf.bpart,
                               Bf.gb, NB, E, gtheta);
        else
            hipLaunchKernelGGL((k_e_split<B, G>), dim3(Bf.gl), dim3(PART_THREADS), 0, st, M, T, theta, r, Bf.cell, Bf.C,
                               Bf.base, Bf.list, Bf.longs, grad, Bf.lpart, Bf.vpart, Bf.gt, NV, Bf.bpart, Bf.gb, NB, E,
                               gtheta);
    };
    if (grad) go(std::true_type{});
    else go(std::false_type{});
}

// E, dE/dr and dE/dtheta of M at (r, theta) with the buffers Bf.
int energy_adjoint_run(const EModel &M, const TileGeom &T, const double *d_r, const double *d_theta, double *d_E,
                       double *d_grad_r, double *d_grad_theta, const AdjointBufs &Bf, hipStream_t st)
{
    const PosView P{d_r, 1, 3};
    const unsigned gb = (unsigned)((M.N + BIN_THREADS - 1) / BIN_THREADS), gt = (unsigned)((T.ntiles + 255) / 256);
    // cleared by a kernel rather than hipMemsetAsync: a caller may capture this
    // sequence in a HIP graph
    hipLaunchKernelGGL(k_tile_clear, dim3(gt), dim3(256), 0, st, Bf.C);
    hipLaunchKernelGGL(k_tile_bin<false>, dim3(gb), dim3(BIN_THREADS), 0, st, M.G, T, M.N, P, Bf.cell, Bf.C.cnt,
                       (const ListPlace *)nullptr, (int32_t *)nullptr, SplitBeads{});
    static_assert(LONG_GROUP == 256, "the grid gt");
    hipLaunchKernelGGL(k_tile_base, dim3(gt), dim3(LONG_GROUP), 0, st, Bf.C, Bf.base, Bf.longs);
    hipLaunchKernelGGL(k_tile_bin<true>, dim3(gb), dim3(BIN_THREADS), 0, st, M.G, T, M.N, P, Bf.cell, Bf.C.fill, Bf.base,
                       Bf.list, SplitBeads{Bf.C, Bf.longs, d_grad_r});
    switch (M.B) {
    case 1: launch_adjoint<1>(M, T, d_r, d_theta, d_E, d_grad_r, d_grad_theta, Bf, st); break;
    case 2: launch_adjoint<2>(M, T, d_r, d_theta, d_E, d_grad_r, d_grad_theta, Bf, st); break;
    case 3: launch_adjoint<3>(M, T, d_r, d_theta, d_E, d_grad_r, d_grad_theta, Bf, st); break;
    default: launch_adjoint<4>(M, T, d_r, d_theta, d_E, d_grad_r, d_grad_theta, Bf, st); break;
    }
    HIPE(hipGetLastError());
    return 0;
}

// The scratch chromo_energy_adjoint_noalloc documents and checks: a limit on sizes
// that does not move with the kernels.
size_t noalloc_bytes(const EModel &M, bool grad)
{
    const size_t nb = (size_t)(M.G.nx * M.G.ny * M.G.nz), Bp1 = (size_t)M.B + 1, N = (size_t)M.N;
    size_t o = 0;
    for (size_t x : {4 * N, 4 * N, 32 * N, 32 * N, 4 * nb, 4 * nb, 4 * nb, (size_t)8192, (size_t)8192, (size_t)8,
                     8 * nb * Bp1, grad ? 8 * nb * Bp1 : (size_t)0, 8 * MAXT * (size_t)grid_blocks((int64_t)nb),
                     8 * MAXT * (size_t)grid_blocks(M.N)})
        o = align_scratch(o + x);
    return o;
}

// ---- the allocation-free evaluation -----------------------------------------

// Device memory of chromo_energy_adjoint_noalloc: one array per GPU, held until
// the process ends.  Host code reaches it only through the address that
// hipGetSymbolAddress returns for the current device (the array's name is a
// host-side stand-in, not a device address).
constexpr size_t NOALLOC_BYTES = size_t(32) << 20;
__device__ __align__(256) char scratch[NOALLOC_BYTES];

constexpr int NOALLOC_MAX_DEVICES = 64;
std::mutex g_noalloc_mu;
char *g_noalloc_ptr[NOALLOC_MAX_DEVICES] = {};

// The scratch array of the current device, looked up once per device.
int noalloc_scratch(char **out)
{
    int dev = 0;
    HIPE(hipGetDevice(&dev));
    if (dev < 0 || dev >= NOALLOC_MAX_DEVICES) return eset(-1, "device index outside 0..63");
    std::lock_guard<std::mutex> lock(g_noalloc_mu);
    if (!g_noalloc_ptr[dev]) {
        void *p = nullptr;
        HIPE(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        if (!p) return eset(-2, "hipGetSymbolAddress gave no address for the scratch array");
        g_noalloc_ptr[dev] = (char *)p;
    }
    *out = g_noalloc_ptr[dev];
    return 0;
}

}  // namespace

extern "C" {

int chromo_energy_adjoint(const chromo_energy_model *model, const double *d_r, const double *d_theta,
                          double *d_E, double *d_grad_r, double *d_grad_theta, void *stream)
{
    EModel M;
    int rc = make_adjoint_model(model, d_r, d_theta, d_E, M);
    if (rc) return rc;
    hipStream_t st = (hipStream_t)stream;
    const TileGeom T = tile_geom(M.G, TILE_MAX, M.bead_vol);
    AdjointBufs Bf;
    StreamBuffer buf;
    buf.st = st;
    HIPE(hipMallocAsync((void **)&buf.p, adjoint_carve(M, T, nullptr, Bf), st));
    adjoint_carve(M, T, buf.p, Bf);
    return energy_adjoint_run(M, T, d_r, d_theta, d_E, d_grad_r, d_grad_theta, Bf, st);
}

int64_t chromo_energy_adjoint_bytes(const chromo_energy_model *model)
{
    EModel M;
    const int rc = make_model(model, M);
    if (rc) return rc;
    AdjointBufs Bf;
    return (int64_t)adjoint_carve(M, tile_geom(M.G, TILE_MAX, M.bead_vol), nullptr, Bf);
}

int chromo_energy_adjoint_ws(const chromo_energy_model *model, const double *d_r, const double *d_theta,
                             double *d_E, double *d_grad_r, double *d_grad_theta, void *d_ws, int64_t ws_bytes,
                             void *stream)
{
    EModel M;
    int rc = make_adjoint_model(model, d_r, d_theta, d_E, M);
    if (rc) return rc;
    const TileGeom T = tile_geom(M.G, TILE_MAX, M.bead_vol);
    AdjointBufs Bf;
    const size_t bytes = adjoint_carve(M, T, nullptr, Bf);
    if (!d_ws || ws_bytes < 0 || (size_t)ws_bytes < bytes)
        return eset(-1, "the workspace holds fewer bytes than chromo_energy_adjoint_bytes");
    if ((uintptr_t)d_ws % 16) return eset(-1, "the workspace must be 16-byte aligned");
    adjoint_carve(M, T, (char *)d_ws, Bf);
    return energy_adjoint_run(M, T, d_r, d_theta, d_E, d_grad_r, d_grad_theta, Bf, (hipStream_t)stream);
}

int chromo_energy_adjoint_noalloc(const chromo_energy_model *model, const double *d_r, const double *d_theta,
                                  double *d_E, double *d_grad_r, double *d_grad_theta, void *stream)
{
    EModel M;
    int rc = make_adjoint_model(model, d_r, d_theta, d_E, M);
    if (rc) return rc;
    const TileGeom T = tile_geom(M.G, TILE_MAX, M.bead_vol);
    AdjointBufs Bf;
    const size_t doc = noalloc_bytes(M, d_grad_r != nullptr), own = adjoint_carve(M, T, nullptr, Bf);
    const size_t bytes = doc > own ? doc : own;
    if (bytes > NOALLOC_BYTES)
        return eset(-1, "the evaluation needs " + std::to_string(bytes) + " bytes of scratch; the allocation-free "
                        "entry point holds " + std::to_string(NOALLOC_BYTES) + " (use chromo_energy_adjoint)");
    char *base = nullptr;
    rc = noalloc_scratch(&base);
    if (rc) return rc;
    adjoint_carve(M, T, base, Bf);
    return energy_adjoint_run(M, T, d_r, d_theta, d_E, d_grad_r, d_grad_theta, Bf, (hipStream_t)stream);
}

int chromo_energy_reference(const chromo_energy_model *model, const double *d_pos, int32_t soa,
                            const double *d_pref, const double *d_intra, double chi,
                            double *d_density_out, double *d_out, void *stream)
{
    EModel M;
    int rc = make_model(model, M);
    if (rc) return rc;
    if (!d_pos || !d_pref || !d_intra || !d_out) return eset(-1, "NULL argument");
    hipStream_t st = (hipStream_t)stream;
    const int B = M.B;
    const int64_t sc = soa ? M.N : 1, sbd = soa ? 1 : 9;
    const PosView P{d_pos, sc, sbd};
    EnergyBufs Bf;
    StreamBuffer buf;
    buf.st = st;
    HIPE(hipMallocAsync((void **)&buf.p, energy_carve(M, P, d_density_out, nullptr, Bf), st));
    energy_carve(M, P, d_density_out, buf.p, Bf);
    const double *rho = Bf.J.density;
    const int gv = Bf.gv, gb = Bf.gb;
    ScatterSpan X;
    X.add(Bf.J);
    hipError_t e = scatter_run(nullptr, Bf.J, 1, X, st);
    if (e != hipSuccess) return eset(-2, std::string("density scatter: ") + hipGetErrorString(e));
    hipLaunchKernelGGL(k_ref_voxel, dim3(gv), dim3(EB), 0, st, M, d_pref, chi, rho, Bf.vpart, B + 1);
    hipLaunchKernelGGL(k_ref_bead, dim3(gb), dim3(EB), 0, st, M, d_pos, sc, sbd, Bf.bpart, B + 1);
    hipLaunchKernelGGL(k_ref_final, dim3(1), dim3(FINAL_THREADS), 0, st, M, d_pref, d_intra, Bf.vpart, gv, Bf.bpart,
                       gb, d_out);
    HIPE(hipGetLastError());
    return 0;
}

}  // extern "C"
