"""Index arithmetic at the largest chains taken (csrc/chromo_index.hpp, compiled for the
host, and the sizes of the workspaces)."""
import subprocess
from pathlib import Path

ROOT = Path(__file__).resolve().parents[1]

MAIN = """
#include "chromo_index.hpp"
#include <stdio.h>
#include <stdlib.h>
int main(int n, char **a)
{
    for (int i = 1; i < n; ++i)
        for (int j = 0; j < 3; ++j) printf("%lld\\n", (long long)chromo::row3((int32_t)atol(a[i]), j));
}
"""


def test_bead_rows(tmp_path):
    (tmp_path / "main.cpp").write_text(MAIN)
    subprocess.run(["g++", "-O1", "-std=c++17", "-fsanitize=undefined", "-fno-sanitize-recover",
                    "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", f"-I{ROOT / 'chromo_amd' / 'csrc'}",
                    "-o", str(tmp_path / "rows"), str(tmp_path / "main.cpp")], check=True, capture_output=True)
    beads = [0, 1, 715827881, 715827882, 715827883, 2 ** 31 - 2]
    out = subprocess.run([str(tmp_path / "rows"), *map(str, beads)], check=True, capture_output=True).stdout.split()
    assert [int(x) for x in out] == [3 * b + j for b in beads for j in range(3)]


def test_kernels_index_beads_through_it():
    """The tiles' code holds beads in 32 bits: no product of one with 3 outside row3."""
    src = (ROOT / "chromo_amd" / "csrc" / "chromo_energy.hip").read_text()
    tile = src[src.index("// ---- field terms"):src.index("// ---- bead / bond terms")]
    assert "int32_t b" in tile and "3 * b" not in tile and tile.count("row3(b, j)") >= 3


def test_list_places_have_64_bits():
    """The workspaces hold, per bead, its cell and its entries in the lists, and per tile
    two counters of 32 bits and the place of its list in 64: the lists of the largest
    chains hold more than 2^31 entries."""
    import ctypes

    from chromo_amd import _lib as L
    h = L.lib()
    # a long flat grid: so many tiles that 4 bytes of each outweigh the rest of the scratch
    n, N = 2 ** 22, 2 ** 31 - 2
    m = L.ChromoEnergyModel()
    m.N, m.B, m.nx, m.ny, m.nz = N, 1, n, 1, 1
    m.x_width, m.y_width, m.z_width, m.bead_vol = 30.0 * n, 30.0, 30.0, 1.0
    assert h.chromo_energy_adjoint_bytes(ctypes.byref(m)) >= 4 * N + 4 * 2 * N + (4 + 4 + 8) * (n // 8)
    rep = (L.ChromoReplica * 1)()
    R = rep[0]
    R.N, R.B, R.field_on, R.nx, R.ny, R.nz = N, 1, 1, n, 1, 1
    for j in range(3):
        R.width[j] = (30.0 * n, 30.0, 30.0)[j]
        R.dxyz[j], R.half_width[j], R.half_step[j] = 30.0, R.width[j] / 2, 15.0
    R.vol_bin = 27000.0
    assert h.chromo_density_init_bytes(ctypes.addressof(rep), 1) >= 4 * N + 4 * 2 * N + (4 + 4 + 8) * (n // 4)
