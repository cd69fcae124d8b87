"""The tiles of an axis and their halves (csrc/chromo_index.hpp, compiled for the host): on
every axis of up to 70 voxels each cell lies in one tile and one half of it, a tile lists
every cell that its halves need, and the places of a bead's corners in a range are those
of the voxels."""
import subprocess
from pathlib import Path

ROOT = Path(__file__).resolve().parents[1]

MAIN = r"""
#include "chromo_index.hpp"
#include <stdio.h>
#include <set>
#include <vector>
using namespace chromo;
static int bad = 0;
#define CHECK(x) do { if (!(x)) { printf("n %d nt %d tile %d half %d: %s\n", n, nt, t, h, #x); ++bad; } } while (0)
int main()
{
    for (int n = 1; n <= 70; ++n) {
        const int nt = (n + 7) / 8;
        std::vector<std::set<int>> lists(nt);
        for (int c = 0; c < n; ++c) {
            int at[2];
            const int k = axis_tiles<true>(n, nt, c, at);
            for (int i = 0; i < k; ++i) lists[at[i]].insert(c);
        }
        std::vector<int> owner(n, 0), owner_whole(n, 0);
        for (int t = 0; t < nt; ++t)
            for (int h = -1; h < 2; ++h) {          // -1: the whole tile
                int start = tile_start(n, nt, t), size = tile_start(n, nt, t + 1) - start;
                if (h >= 0) tile_half(h, start, size);
                CHECK(size >= 0 && size <= 8 && (h == 1 || size > 0));
                if (size == 0) continue;
                const bool whole = size == n;
                CHECK(whole || size >= 2);
                CHECK(whole || n - size >= 2);
                for (int c = 0; c < n; ++c) {
                    // the range's voxels that a bead of cell c reaches: its own and the next
                    const int up = (c + 1) % n;
                    auto place = [&](int v) {       // inside, or the first voxel behind the range
                        for (int i = 0; i < size + (whole ? 0 : 1); ++i)
                            if ((start + i) % n == v) return i;
                        return -1;
                    };
                    const bool near = place(c) >= 0 || place(up) >= 0;
                    if (near) CHECK(lists[t].count(c));
                    CHECK(tile_near(n, start, size, c) == near);
                    const bool own = c >= start && c < start + size;
                    if (own) ++(h < 0 ? owner_whole : owner)[c];
                    if (whole || !near) continue;   // a whole axis wraps onto itself: places are the cells
                    const int l = tile_local(n, start, size, c);
                    CHECK(own == (l >= 0 && l < size));
                    CHECK((l >= 0 ? l : -1) == place(c));
                    CHECK((l >= size ? -1 : l + 1) == place(up));
                }
            }
        for (int c = 0; c < n; ++c) {
            const int t = -1, h = c;
            CHECK(owner[c] == 1 && owner_whole[c] == 1);
        }
    }
    return bad != 0;
}
"""


def test_tiles_and_halves(tmp_path):
    (tmp_path / "main.cpp").write_text(MAIN)
    subprocess.run(["g++", "-O1", "-std=c++17", "-fsanitize=undefined", "-fno-sanitize-recover",
                    "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", f"-I{ROOT / 'chromo_amd' / 'csrc'}",
                    "-o", str(tmp_path / "tiles"), str(tmp_path / "main.cpp")], check=True, capture_output=True)
    r = subprocess.run([str(tmp_path / "tiles")], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout[:2000] + r.stderr[:2000]
