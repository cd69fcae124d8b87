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
    """The tile kernel holds beads in 32 bits: no product of one with 3 outside row3."""
    src = (ROOT / "chromo_amd" / "csrc" / "chromo_energy.hip").read_text()
    tile = src[src.index("k_e_tile(EModel"):src.index("// ---- bead / bond terms")]
    assert "3 * b" not in tile and tile.count("row3(b, j)") == 3
