// chromo_index.hpp -- index arithmetic of beads, tiles and their parts: whole numbers only,
// so that a test can compile it for the host.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace chromo {

// Place of component j of bead b in an N x 3 array: past 2^31 from 715,827,883 beads on.
__host__ __device__ __forceinline__ int64_t row3(int32_t b, int j) { return 3 * (int64_t)b + j; }

// An axis of n voxels cut into nt tiles: tile t starts at t n / nt, and cell c lies in tile
// tile_of.
__host__ __device__ __forceinline__ int tile_start(int n, int nt, int t) { return (int)((int64_t)t * n / nt); }
__host__ __device__ __forceinline__ int tile_of(int n, int nt, int c) { return (int)(((int64_t)(c + 1) * nt - 1) / n); }

// The tiles of one axis that list a bead of cell c: its own and, when the cell lies on
// a face, the neighbour behind that face (UPPER: behind either face, for tiles that
// need their voxels' upper neighbours; else only behind the upper one, whose voxels the
// bead's upper corners reach).  Returns how many.  UPPER needs tiles of two voxels or
// more, so that a cell lies on one face only.
template <bool UPPER>
__host__ __device__ __forceinline__ int axis_tiles(int n, int nt, int c, int t[2])
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

// Halves of one axis of a tile, `which` 0 or 1; a tile of fewer than 4 voxels is not
// halved and has no second half (size 0).  Halves have two voxels or more, and two
// voxels or more lie outside them: the neighbours below and above are different cells.
__host__ __device__ __forceinline__ void tile_half(int which, int &start, int &size)
{
    const int lower = size < 4 ? size : size / 2;
    start += which ? lower : 0;
    size = which ? size - lower : lower;
}

// Place of a cell on one axis of a tile or part of `size` voxels from `start`, for a cell
// that is known to be inside or a neighbour: 0 .. size - 1 inside, -1 and size for the
// neighbours below and above.
__host__ __device__ __forceinline__ int tile_local(int n, int start, int size, int c)
{
    int d = c - start;
    if (d >= 0 && d < size) return d;
    if (d < 0) d += n;
    return d == size ? size : -1;
}

// Whether cell c is inside or a neighbour.  A part of the whole axis has no neighbours.
__host__ __device__ __forceinline__ bool tile_near(int n, int start, int size, int c)
{
    int d = c - start;
    if (d < 0) d += n;
    return d <= size || d == n - 1;
}

}  // namespace chromo
