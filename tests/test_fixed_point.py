"""The energy adjoint's corner weights as integers (csrc/chromo_fixed.hpp, compiled for the
host): the nearest multiple of 2^-60 for any weight, ties and their neighbours included,
and words whose products and sums stay inside their types."""
import subprocess
from fractions import Fraction
from pathlib import Path

import numpy as np
import pytest

from chromo_amd import _lib as L

ROOT = Path(__file__).resolve().parents[1]

MAIN = """
#include "chromo_fixed.hpp"
#include <stdio.h>
int main()
{
    double w;
    while (fread(&w, 8, 1, stdin) == 1) {
        const chromo::Fixed60 f = chromo::fixed60(w * chromo::FIXED60_SCALE);
        const double back = chromo::from_fixed60(f.hi, (uint64_t)(int64_t)f.lo);
        printf("%u %d %a\\n", f.hi, f.lo, back);
    }
}
"""


def _weights():
    """Weights at and beside the ties of a high word of 20 to 32 bits, of the low word, the
    ends of the range and random products of three."""
    rs = np.random.RandomState(0)
    w = [0.0, 1.0, 2.0 ** -1074, 2.0 ** -61, 2.0 ** -60, 3 * 2.0 ** -61, 1 - 2.0 ** -53]
    for bits in range(20, 33):
        for k in list(range(4)) + list(rs.randint(0, 2 ** bits, size=20)) + [2 ** bits - 1]:
            w.append((2 * int(k) + 1) * 2.0 ** -(bits + 1))
    w += list(rs.randint(0, 2 ** 31, size=50) * 2.0 ** -31 + (2 * rs.randint(0, 2 ** 20, size=50) + 1) * 2.0 ** -52)
    w += list(np.prod(rs.random_sample((2000, 3)), axis=1))
    w = np.array(w)
    w = np.concatenate([w, np.nextafter(w, 2), np.maximum(np.nextafter(w, -1), 0)])
    return w[w <= 1]


@pytest.fixture(scope="module")
def words(tmp_path_factory):
    d = tmp_path_factory.mktemp("fixed")
    (d / "main.cpp").write_text(MAIN)
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    f"-I{ROOT / 'include'}", f"-I{ROOT / 'chromo_amd' / 'csrc'}", "-o", str(d / "fixed"),
                    str(d / "main.cpp")], check=True, capture_output=True)
    w = _weights()
    out = subprocess.run([str(d / "fixed")], input=w.tobytes(), check=True, capture_output=True).stdout.decode()
    rows = [line.split() for line in out.splitlines()]
    assert len(rows) == len(w)
    return w, [(int(h), int(lo), float.fromhex(b)) for h, lo, b in rows]


def test_nearest_multiple(words):
    for w, (hi, lo, back) in zip(*words):
        exact = Fraction(float(w))
        total = Fraction(hi * 2 ** 30 + lo, 2 ** 60)
        assert total >= 0 and abs(total - exact) <= Fraction(1, 2 ** 61), float(w).hex()
        assert back == float(total), float(w).hex()


def test_words_in_range(words):
    """Times the largest binder state the words fit 32 bits, summed over the largest chain
    (2^31 beads in one voxel) 64."""
    hi = max(h for h, _, _ in words[1]) * L.MAX_SITES
    lo = max(abs(x) for _, x, _ in words[1]) * L.MAX_SITES
    assert hi < 2 ** 32 and lo < 2 ** 31
    assert hi * 2 ** 31 < 2 ** 64 and lo * 2 ** 31 < 2 ** 63
