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
// own cells.  Neither the densities nor dE/drho ever reach HBM.
//
// What bounds it: at 10^6 beads, B = 4, 128^3 voxels a third of the time is the adds (8
// corners x species x 2 words per bead and tile, a third of them conflicting), a quarter
// turning sums into dE/drho, a sixth the gather at the beads, the rest loads, weights and
// the barriers between; two blocks of eight wavefronts share a compute unit's LDS.
// Tiles of 8 x 8 x 4 with four smaller blocks take the same time (less waiting, more
// halo).  One evaluation there: 417 us as bucketed records, a gather of every record by
// its eight voxels and passes for the voxel and bead terms; 280 us so.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "chromo_device.hpp"

namespace chromo {
namespace {

// Tiles of at most 8 x 8 x 8 voxels.  Tile t of an axis of n voxels cut into nt tiles
// starts at t n / nt: tiles of at least half the size when there are several, so a cell
// touches at most one face per axis and the lists hold at most twice the beads per axis.
// An axis that fits one tile is one tile that wraps onto itself.
// The scatter needs no upper neighbours, and smaller tiles keep more wavefronts on a
// compute unit.
constexpr int TILE_MAX[3] = {8, 8, 8};
constexpr int FOLD_MAX[3] = {4, 4, 4};
constexpr int TILE_SX = 9, TILE_SY = 9, TILE_SZ = 9;    // a tile's voxels and their upper neighbours
constexpr int TILE_VOX = TILE_SX * TILE_SY * TILE_SZ;
constexpr int TILE_THREADS = 512;
constexpr int TILE_OWN = 1024;              // beads of its own cells a tile notes down in LDS
constexpr int TILE_BLOCKS = 1024;           // blocks of the tile kernel, at most

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

__device__ __forceinline__ int tile_start(int n, int nt, int t) { return (int)((int64_t)t * n / nt); }
__device__ __forceinline__ int tile_of(int n, int nt, int c) { return (int)(((int64_t)(c + 1) * nt - 1) / n); }

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

// The tiles of one axis that list a bead of cell c: its own and, when the cell lies on
// a face, the neighbour behind that face (UPPER: behind either face, for tiles that
// need their voxels' upper neighbours; else only behind the upper one, whose voxels the
// bead's upper corners reach).  Returns how many.
template <bool UPPER>
__device__ __forceinline__ int axis_tiles(int n, int nt, int c, int t[2])
{
    t[0] = nt == 1 ? 0 : tile_of(n, nt, c);
    t[1] = t[0];
    if (nt == 1) return 1;
    if (UPPER && c == tile_start(n, nt, t[0])) {
        t[1] = t[0] == 0 ? nt - 1 : t[0] - 1;
        return 2;
    }
    if (c + 1 == tile_start(n, nt, t[0] + 1)) {
        t[1] = t[0] + 1 == nt ? 0 : t[0] + 1;
        return 2;
    }
    return 1;
}

// Where a list begins in the array of all lists, which hold a bead up to eight times: 64
// bits (268,435,456 beads in one-voxel tiles pass 2^31 entries).
using ListPlace = unsigned long long;

// Clears the lists' counters and the list cursor.
__global__ void k_tile_clear(int32_t *cnt, int32_t *fill, ListPlace *cursor, int n)
{
    const int i = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    if (i < n) cnt[i] = fill[i] = 0;
    if (i == 0) *cursor = 0;
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

__global__ void k_tile_base(const int32_t *cnt, ListPlace *base, ListPlace *cursor, int n)
{
    tile_bases(cnt, base, cursor, n);
}

// PLACE false: each bead's cell into cell[], and the lists' lengths into num.  PLACE
// true: the beads into their lists, num counting the entries placed.  A block counts its beads per
// list in LDS first (consecutive beads lie in a few tiles), so that a list costs it one
// global atomic; a list that finds no room in the block's table takes its entries from
// the global counter one by one.  STABLE: what a block places in a list through its
// table is in bead order (a bit per bead and list in LDS, the rank the bits below).
// Otherwise the order within a list is any.
constexpr int TILE_TABLE = 512, TILE_PROBES = 16, BIN_THREADS = 256;

template <bool PLACE, bool UPPER, bool STABLE>
__device__ __forceinline__ void tile_bin(const GridGeom &G, const TileGeom &T, int64_t N, const PosView &P,
                                         int32_t *cell, int32_t *num, const ListPlace *base, int32_t *list)
{
    constexpr int W = BIN_THREADS / WAVE;
    __shared__ int32_t key[TILE_TABLE], cntl[TILE_TABLE], from[TILE_TABLE];
    __shared__ unsigned long long bits[STABLE && PLACE ? TILE_TABLE * W : 1];
    const int t = (int)threadIdx.x, wv = t / WAVE, lane = t % WAVE;
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
}

template <bool PLACE>
__global__ void __launch_bounds__(BIN_THREADS) k_tile_bin(GridGeom G, TileGeom T, int64_t N, PosView P, int32_t *cell,
                                                          int32_t *num, const ListPlace *base, int32_t *list)
{
    tile_bin<PLACE, true, false>(G, T, N, P, cell, num, base, list);
}

// Place of a cell on one axis of a tile of `size` voxels from `start`: 0 .. size - 1
// inside, -1 and size for the neighbours below and above.
__device__ __forceinline__ int tile_local(int n, int start, int size, int c)
{
    int d = c - start;
    if (d >= 0 && d < size) return d;
    if (d < 0) d += n;
    return d == size ? size : -1;
}

}  // namespace
}  // namespace chromo
