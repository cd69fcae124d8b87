"""A replica record without beads has no densities to scatter: the calls succeed and leave
its grid alone (no launch is made, so this runs without a GPU)."""
import ctypes

from chromo_amd import _lib as L


def test_density_init_without_beads():
    h = L.lib()
    reps = (L.ChromoReplica * 2)()
    for R in reps:
        R.N, R.B, R.field_on, R.nx, R.ny, R.nz, R.vol_bin = 0, 2, 1, 4, 4, 4, 1.0
        for j in range(3):
            R.width[j], R.dxyz[j], R.half_width[j], R.half_step[j] = 4.0, 1.0, 2.0, 0.5
    a = ctypes.addressof(reps)
    for n in (1, 2):
        assert h.chromo_density_init_bytes(a, n) == 0
        assert h.chromo_density_init_ws(a, n, None, 0, None) == 0
