"""The initial densities, bit for bit against the oracle's bead-order loop, on every tile
shape of the scatter (4 x 4 x 4 voxels on large grids, down to single voxels on small ones)
with uneven axes, so that tiles are ragged, for every binder count (the fold's lanes are
grouped by it); chains across the periodic faces, and one crowded enough that a tile's list
has to be sorted."""
import copy

import numpy as np
import pytest

from chromo_amd import _lib as L
from chromo_amd import workloads as W

SHAPES = [(4, 4, 4), (4, 4, 2), (2, 2, 2), (1, 1, 1)]
TILES = 2048
GRIDS = [(53, 55, 54), (47, 49, 45), (23, 25, 27), (13, 11, 14)]


def _shape(n):
    """The scatter's rule: the largest shape that still makes TILES tiles, else the smallest."""
    for s in SHAPES:
        if np.prod([-(-a // b) for a, b in zip(n, s)]) >= TILES:
            return s
    return SHAPES[-1]


def test_grids_cover_the_shapes():
    assert [_shape(n) for n in GRIDS] == SHAPES
    assert all(a % b for n, s in zip(GRIDS, SHAPES) for a, b in zip(n, s) if b > 2)


def _system(n, B, N, seed, scale):
    s = W.make_system(N, B, 8, seed=seed)
    f = s.field
    f.nx, f.ny, f.nz = n
    f.x_width, f.y_width, f.z_width = 30.0 * n[0], 30.0 * n[1], 30.0 * n[2]
    # around a corner of the box: beads on both sides of three faces
    s.chain.r = s.chain.r * scale + 15.0 * np.array(n)
    s.chain.states = np.random.RandomState(seed).randint(0, 3, size=(N, B))
    return s


@pytest.mark.gpu
@pytest.mark.parametrize("B", [1, 2, 3, 4])
@pytest.mark.parametrize("n", GRIDS)
def test_shapes_bitwise(n, B, oracle):
    from chromo_amd.engine import DeviceReplicas
    print("scatter shape", _shape(n), n, B, flush=True)
    for N, scale in ((4000, 1.0), (1500, 0.1)) + (((40000, 1e-3),) if B == 3 else ()):
        s = _system(n, B, N, 70 + B, scale)
        dr = DeviceReplicas([s.chain], [s.field], [copy.deepcopy(s.ctrls)], rng_mode=L.RNG_PHILOX, seeds=[1])
        assert np.array_equal(dr.density_of(0), oracle.OracleSim(s.chain, s.field).density()), (N, scale)
