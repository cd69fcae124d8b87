"""The initial densities, bit for bit against the oracle's bead-order loop, on small and
uneven grids, which the scatter folds in tiles of one voxel or 2 x 2 x 2 (the larger
shapes: test_gpu_scatter_shapes.py): one-voxel axes (corners of a bead share a voxel),
axes of two voxels, ragged tiles; lists of so many runs that they are sorted in global
memory; every binder count; many replicas in one call."""
import copy

import numpy as np
import pytest

from chromo_amd import _lib as L
from chromo_amd import workloads as W

pytestmark = pytest.mark.gpu


def _system(n, B, N, seed, scale=1.0):
    s = W.make_system(N, B, 8, seed=seed)
    s.chain.r = s.chain.r * scale
    s.chain.states = np.random.RandomState(seed).randint(0, 3, size=(N, B))
    f = s.field
    f.nx, f.ny, f.nz = n
    f.x_width, f.y_width, f.z_width = 30.0 * n[0], 30.0 * n[1], 30.0 * n[2]
    return s


CASES = [((1, 1, 1), 1, 60, 1.0), ((1, 9, 5), 2, 400, 1.0), ((2, 3, 4), 3, 500, 1.0), ((8, 8, 4), 4, 900, 1.0),
         ((9, 10, 5), 4, 1500, 1.0), ((16, 17, 8), 2, 2, 1.0), ((23, 7, 31), 1, 6000, 1.0), ((40, 33, 27), 3, 5000, 0.2),
         ((12, 12, 12), 2, 4000, 1e-3), ((64, 2, 1), 4, 257, 1.0)]


def test_scatter_tiles_bitwise(oracle):
    from chromo_amd.engine import DeviceReplicas
    systems = [_system(n, B, N, 60 + i, scale) for i, (n, B, N, scale) in enumerate(CASES)]
    want = [oracle.OracleSim(s.chain, s.field).density() for s in systems]
    print("scatter, all replicas in one call", flush=True)
    dr = DeviceReplicas([s.chain for s in systems], [s.field for s in systems],
                        [copy.deepcopy(s.ctrls) for s in systems], rng_mode=L.RNG_PHILOX, seeds=[1] * len(systems))
    for i, w in enumerate(want):
        assert np.array_equal(dr.density_of(i), w), CASES[i]
    for i, s in enumerate(systems):
        print("scatter", CASES[i], flush=True)
        one = DeviceReplicas([s.chain], [s.field], [copy.deepcopy(s.ctrls)], rng_mode=L.RNG_PHILOX, seeds=[1])
        assert np.array_equal(one.density_of(0), want[i]), CASES[i]
        one.density.fill_(7.0)
        L.check(one.lib.chromo_density_init(one.tab_ptr, 1, None))
        assert np.array_equal(one.density_of(0), want[i]), CASES[i]
