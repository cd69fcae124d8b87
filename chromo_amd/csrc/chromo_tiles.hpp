// chromo_tiles.hpp -- a density grid in tiles and the bead lists of the tiles, for the
// scatter (chromo_density.hpp, which includes this file) and the energy adjoint's tile
// kernel (chromo_energy.hip): voxel densities, field energy and gradient in LDS.
//
// For the adjoint the grid is cut into tiles of at most 8 x 8 x 8 voxels.  Every bead is listed in
// the tile of its lower-corner cell and in the tiles that cell is a neighbour of
// (at most one per axis), so a tile's list holds every bead that reaches its voxels
// and their upper neighbours.  One block per tile then does what took four passes over
// memory: it adds the beads' corner weights into LDS, turns each voxel's density into
// its energy terms and dE/drho in place, and gathers dE/drho back at the beads of its
// own cells.  Neither the densities nor dE/drho ever reach HBM.  Where a condensed chain
// crowds a few tiles, those are worked on in parts, a block per part.
//
// What bounds it: at 10^6 beads, B = 4, 128^3 voxels a third of the time is the adds (8
// corners x species x 2 words per bead and tile, a third of them conflicting), a quarter
// turning sums into dE/drho, a sixth the gather at the beads, the rest loads, weights and
// the barriers between; two blocks of eight wavefronts share a compute unit's LDS.
// Tiles of 8 x 8 x 4 with four smaller blocks take the same time (less waiting, more
// halo).  One evaluation there: 417 us as bucketed records, a gather of every record by
// its eight voxels and passes for the voxel and bead terms; 259 us so.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "chromo_device.hpp"
#include "chromo_index.hpp"

namespace chromo {
namespace {

// The adjoint's tiles have at most 8 x 8 x 8 voxels (TILE_MAX).  Tile t of an axis of n
// voxels cut into nt tiles starts at t n / nt: tiles of at least half the size when there
// are several, so a cell touches at most one face per axis and the lists hold at most twice
// the beads per axis.  An axis that fits one tile is one tile that wraps onto itself.
// The scatter (FOLD_MAX and smaller) needs no upper neighbours, and smaller tiles keep more
// wavefronts on a compute unit; a cell of its one-voxel tiles touches both faces, and only
// the upper one counts.
constexpr int TILE_MAX[3] = {8, 8, 8};
static_assert((TILE_MAX[0] + 1) / 2 >= 2 && (TILE_MAX[1] + 1) / 2 >= 2 && (TILE_MAX[2] + 1) / 2 >= 2,
              "a cell of a tile that also lists its upper neighbours lies on one face");
constexpr int FOLD_MAX[3] = {4, 4, 4};
constexpr int TILE_THREADS = 512;
constexpr int TILE_OWN = 1024;              // beads of its own cells a tile notes down in LDS
constexpr int TILE_BLOCKS = 1024;           // blocks of the tile kernel, at most
constexpr int LONG_LIST = 2048, HUGE_LIST = 8192;       // beads of a list (long_list)
constexpr int SPLIT_MIN = 4 * HUGE_LIST;    // beads of a chain whose lists are never split
constexpr int TILE_PARTS = 8;               // of a tile with a long list
constexpr int PART_THREADS = 512, PART_SCAN = 4, PART_NOTES = 4096;
constexpr int PART_BLOCKS = 512;            // two per compute unit

struct TileGeom {
    int32_t n[3], nt[3], ntiles;
    int32_t recip;                          // the divisors below suit div_by
    double rw[3], rd[3], rvol;              // 1 / width, 1 / voxel side, 1 / vol_bin
    double vbV;                             // vol_bin / bead_vol
};

inline TileGeom tile_geom(const GridGeom &G, const int (&most)[3], double bead_vol)
{
    TileGeom T;
    const int64_t n[3] = {G.nx, G.ny, G.nz};
    T.ntiles = 1;
    T.recip = recip_range(G.vol_bin);
    T.rvol = 1.0 / G.vol_bin;
    T.vbV = G.vol_bin / bead_vol;
    for (int j = 0; j < 3; ++j) {
        T.n[j] = (int32_t)n[j];
        T.nt[j] = (int32_t)((n[j] + most[j] - 1) / most[j]);
        T.ntiles *= T.nt[j];
        T.recip = T.recip && recip_range(G.width[j]) && recip_range(G.dxyz[j]);
        T.rw[j] = 1.0 / G.width[j];
        T.rd[j] = 1.0 / G.dxyz[j];
    }
    return T;
}

// The scatter's tiles: the largest of these shapes that still gives every compute unit
// several wavefronts, one per tile.  A tile's beads are folded one after the other, so a
// small grid with many beads wants small tiles, and a large one large tiles (fewer beads
// listed twice).
constexpr int FOLD_TILES = 2048;

inline TileGeom fold_geom(const GridGeom &G)
{
    constexpr int shapes[4][3] = {{FOLD_MAX[0], FOLD_MAX[1], FOLD_MAX[2]}, {4, 4, 2}, {2, 2, 2}, {1, 1, 1}};
    TileGeom T;
    for (const auto &most : shapes) {
        T = tile_geom(G, most, 1.0);
        if (T.ntiles >= FOLD_TILES) break;
    }
    return T;
}

// Tiles that list one bead, at most.
inline int tile_images(const TileGeom &T)
{
    int k = 1;
    for (int j = 0; j < 3; ++j) k *= T.nt[j] > 1 ? 2 : 1;
    return k;
}

// grid_lower's cell and weights (chromo_density.hpp), bit for bit, with the exact
// divisions from reciprocals where the grid allows.
__device__ __forceinline__ void tile_lower(const GridGeom &G, const TileGeom &T, const double *x, int ix[3],
                                           double w[3])
{
    double a[3];
    bool far = !T.recip;
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        a[j] = x[j] + G.half_width[j];
        far = far || !(fabs(a[j]) < 0x1p40 * G.width[j]);
    }
    if (far) {
        int64_t i64[3];
        grid_lower(G, x[0], x[1], x[2], i64, w);
#pragma unroll
        for (int j = 0; j < 3; ++j) ix[j] = (int)i64[j];
        return;
    }
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        const double W = G.width[j];
        double q = trunc(a[j] * T.rw[j]);
        double r = fma(-q, W, a[j]);
        q += (a[j] >= 0) ? ((r < 0) ? -1.0 : (r >= W ? 1.0 : 0.0)) : ((r > 0) ? 1.0 : (r <= -W ? -1.0 : 0.0));
        r = fma(-q, W, a[j]);
        r += (r < 0) ? W : 0.0;
        double u = div_by(r - G.half_step[j], G.dxyz[j], T.rd[j]);
        if (!(u >= -1.0 && u < (double)T.n[j])) u = 0.0;
        const double f = floor(u);
        ix[j] = (f == -1.0) ? T.n[j] - 1 : (int)f;
        w[j] = 1 - (u - f);
    }
}

// Where a list begins in the array of all lists, which hold a bead up to eight times: 64
// bits (268,435,456 beads in one-voxel tiles pass 2^31 entries).
using ListPlace = unsigned long long;

// What a count of the lists starts from: their lengths, the entries placed, the end of the
// last list, whether long lists are split, and a ticket.
struct TileCounters {
    int32_t *cnt, *fill, *split, *ticket;
    ListPlace *cursor;
    int32_t n;
};

__global__ void k_tile_clear(TileCounters C)
{
    const int i = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    if (i < C.n) C.cnt[i] = C.fill[i] = 0;
    if (i == 0) {
        *C.cursor = 0;
        *C.split = 0;
        *C.ticket = 0;
    }
}

// The long lists, of more than `most` beads, in tile order per block of k_tile_base: tiles
// tile[LONG_GROUP g + k] for k < count[g].  They are split where one holds more than `huge`.
constexpr int LONG_GROUP = 256, LONG_GROUPS = 2048;     // 2^22 voxels make 2^19 tiles at most
struct LongTiles {
    int32_t *tile, *count;
    int32_t most, huge;
};

// Beads of a list from which on it is split; known once k_tile_base is done.
__device__ __forceinline__ int32_t split_above(const TileCounters &C, const LongTiles &L)
{
    return uni_i32(*C.split) ? L.most : 0x7fffffff;
}

// Room for every list: a wavefront's lists in a row, the wavefronts in the order they
// arrive (nothing depends on where a list lies).
__device__ __forceinline__ void tile_bases(const int32_t *cnt, ListPlace *base, ListPlace *cursor, int n)
{
    const int i = (int)(blockIdx.x * blockDim.x + threadIdx.x), lane = lane_id();
    const int64_t k = i < n ? cnt[i] : 0;
    int64_t sum = k;    // of the lanes up to this one
    for (int o = 1; o < WAVE; o <<= 1) {
        const int64_t below = __shfl_up(sum, o);
        if (lane >= o) sum += below;
    }
    ListPlace at = 0;
    if (lane == WAVE - 1) at = atomicAdd(cursor, (ListPlace)sum);
    at = (ListPlace)readlane_i64((int64_t)at, WAVE - 1);
    if (i < n) base[i] = at + (ListPlace)(sum - k);
}

__global__ void __launch_bounds__(LONG_GROUP)
k_tile_base(TileCounters C, ListPlace *base, LongTiles L)
{
    tile_bases(C.cnt, base, C.cursor, C.n);
    __shared__ int32_t waves[LONG_GROUP / WAVE];
    const int i = (int)(blockIdx.x * LONG_GROUP + threadIdx.x), w = (int)threadIdx.x / WAVE;
    const int len = i < C.n ? C.cnt[i] : 0;
    int mine;
    int at = wave_excl_count(len > L.most, mine);
    if (lane_id() == 0) waves[w] = mine;
    if (len > L.huge) atomicOr(C.split, 1);
    __syncthreads();
    int all = 0;
    for (int k = 0; k < LONG_GROUP / WAVE; ++k) {
        at += k < w ? waves[k] : 0;
        all += waves[k];
    }
    if (len > L.most) L.tile[(int)blockIdx.x * LONG_GROUP + at] = i;
    if (threadIdx.x == 0) L.count[blockIdx.x] = all;
}

// PLACE false: each bead's cell into cell[], and the lists' lengths into num.  PLACE
// true: the beads into their lists, num counting the entries placed.  A block counts its beads per
// list in LDS first (consecutive beads lie in a few tiles), so that a list costs it one
// global atomic; a list that finds no room in the block's table takes its entries from
// the global counter one by one.  STABLE: what a block places in a list through its
// table is in bead order (a bit per bead and list in LDS, the rank the bits below).
// Otherwise the order within a list is any.  UPPER: a bead whose own tile's list is split
// gets a zero field gradient.
constexpr int TILE_TABLE = 512, TILE_PROBES = 16, BIN_THREADS = 256;

struct SplitBeads {
    TileCounters C;
    LongTiles L;
    double *grad;           // N x 3, or nullptr
};

template <bool PLACE, bool UPPER, bool STABLE>
__device__ __forceinline__ void tile_bin(const GridGeom &G, const TileGeom &T, int64_t N, const PosView &P,
                                         int32_t *cell, int32_t *num, const ListPlace *base, int32_t *list,
                                         const SplitBeads &X = SplitBeads{})
{
    constexpr int W = BIN_THREADS / WAVE;
    __shared__ int32_t key[TILE_TABLE], cntl[TILE_TABLE], from[TILE_TABLE];
    __shared__ unsigned long long bits[STABLE && PLACE ? TILE_TABLE * W : 1];
    const int t = (int)threadIdx.x, wv = t / WAVE, lane = t % WAVE;
    const int32_t most = PLACE && UPPER ? split_above(X.C, X.L) : 0;
    for (int i = t; i < TILE_TABLE; i += BIN_THREADS) {
        key[i] = -1;
        cntl[i] = 0;
    }
    if (STABLE && PLACE)
        for (int i = t; i < TILE_TABLE * W; i += BIN_THREADS) bits[i] = 0;
    __syncthreads();
    const int64_t b = (int64_t)blockIdx.x * BIN_THREADS + t;
    int slot[8], rank[8], tile[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) {
        tile[q] = -1;
        slot[q] = -1;
        rank[q] = 0;
    }
    if (b < N) {
        int ix[3];
        if (PLACE) {
            const uint32_t c = (uint32_t)cell[b], q = c / (uint32_t)T.n[0];
            ix[0] = (int)(c - q * (uint32_t)T.n[0]);
            ix[1] = (int)(q % (uint32_t)T.n[1]);
            ix[2] = (int)(q / (uint32_t)T.n[1]);
        } else {
            double x[3], w[3];
            for (int j = 0; j < 3; ++j) x[j] = P.p[j * P.sc + b * P.sb];
            tile_lower(G, T, x, ix, w);
            cell[b] = ix[0] + T.n[0] * (ix[1] + T.n[1] * ix[2]);
        }
        int s[3][2], k[3];
#pragma unroll
        for (int j = 0; j < 3; ++j) k[j] = axis_tiles<UPPER>(T.n[j], T.nt[j], ix[j], s[j]);
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            if ((q & 1) >= k[0] || ((q >> 1) & 1) >= k[1] || (q >> 2) >= k[2]) continue;
            tile[q] = s[0][q & 1] + T.nt[0] * (s[1][(q >> 1) & 1] + T.nt[1] * s[2][q >> 2]);
            int h = tile[q] & (TILE_TABLE - 1);
            for (int p = 0; p < TILE_PROBES; ++p) {
                const int old = atomicCAS(&key[h], -1, tile[q]);
                if (old == -1 || old == tile[q]) {
                    slot[q] = h;
                    break;
                }
                h = (h + 1) & (TILE_TABLE - 1);
            }
            if (slot[q] < 0) rank[q] = atomicAdd(&num[tile[q]], 1);
            else if (STABLE && PLACE) atomicOr(&bits[slot[q] * W + wv], 1ull << lane);
            else rank[q] = atomicAdd(&cntl[slot[q]], 1);
        }
    }
    __syncthreads();
    for (int i = t; i < TILE_TABLE; i += BIN_THREADS)
        if (key[i] >= 0) {
            int n = cntl[i];
            if (STABLE && PLACE)
                for (int w = 0; w < W; ++w) n += __popcll(bits[i * W + w]);
            from[i] = atomicAdd(&num[key[i]], n);
            if (PLACE && UPPER) cntl[i] = X.C.cnt[key[i]] > most;
        }
    if (!PLACE) return;
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 8; ++q) {
        if (tile[q] < 0) continue;
        ListPlace at = base[tile[q]] + (ListPlace)rank[q];
        if (slot[q] >= 0) {
            at += (ListPlace)from[slot[q]];
            if (STABLE) {
                for (int w = 0; w < wv; ++w) at += (ListPlace)__popcll(bits[slot[q] * W + w]);
                at += (ListPlace)__popcll(bits[slot[q] * W + wv] & ((1ull << lane) - 1));
            }
        }
        list[at] = (int32_t)b;
    }
    // entry 0 is the bead's own tile
    if (UPPER && X.grad && tile[0] >= 0 && (slot[0] >= 0 ? cntl[slot[0]] != 0 : X.C.cnt[tile[0]] > most))
        for (int j = 0; j < 3; ++j) X.grad[3 * b + j] = 0;
}

template <bool PLACE>
__global__ void __launch_bounds__(BIN_THREADS) k_tile_bin(GridGeom G, TileGeom T, int64_t N, PosView P, int32_t *cell,
                                                          int32_t *num, const ListPlace *base, int32_t *list,
                                                          SplitBeads X)
{
    tile_bin<PLACE, true, false>(G, T, N, P, cell, num, base, list, X);
}

}  // namespace
}  // namespace chromo
