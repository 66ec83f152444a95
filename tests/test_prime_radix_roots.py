"""The odd primes' float32 cosines of the two-stage transforms (sk_rdft.h, RootTable), both tables, against the source's
own constants: compiled on the host, they sum to -1/2 over half a turn to a step of the smallest, so that a constant line
leaves nothing at the other frequencies, and each stays within three steps of its value.
"""
import os
import shutil
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PROGRAM = r"""
#include <cstdio>
#include "sk_rdft.h"
template <int R, bool BACK> void show() {
  constexpr sk::RootTable<R, BACK> t{};
  for (int m = 0; m < R; ++m) printf("%d %d %d %.17g %.17g\n", R, int(BACK), m, t.c[m], t.s[m]);
}
int main() {
  show<7, false>(); show<7, true>(); show<11, false>(); show<11, true>(); show<13, false>(); show<13, true>();
}
"""


@pytest.fixture(scope="module")
def tables(tmp_path_factory):
    if shutil.which("hipcc") is None:
        pytest.skip("no hipcc")
    d = tmp_path_factory.mktemp("roots")
    (d / "roots.hip").write_text(PROGRAM)
    subprocess.run(["hipcc", "-std=c++17", "--cuda-host-only", "-I", os.path.join(ROOT, "simulatokit_amd", "csrc"), "-I",
                    os.path.join(ROOT, "include"), str(d / "roots.hip"), "-o", str(d / "roots")], check=True,
                   capture_output=True, timeout=100)
    out = subprocess.run([str(d / "roots")], check=True, capture_output=True, text=True, timeout=20).stdout
    t = {}
    for line in out.splitlines():
        r, back, m, c, s = line.split()
        t.setdefault((int(r), int(back)), []).append((float(c), float(s)))
    return t


@pytest.mark.parametrize("r", [7, 11, 13])
@pytest.mark.parametrize("back", [0, 1])
def test_cosines_of_a_prime_sum_to_minus_a_half(tables, r, back):
    c, s = np.array(tables[r, back]).T
    angle = 2 * np.pi * np.arange(r) / r
    half = c[1:r // 2 + 1]
    assert np.array_equal(half, c[:r // 2:-1]) and np.allclose(s[1:], -s[:0:-1], rtol=0, atol=0)
    assert abs(half.sum() + 0.5) <= np.spacing(np.float32(np.abs(half).min()))
    assert np.abs(c - np.cos(angle)).max() <= 3 * 2.0 ** -25 and np.abs(s - np.sin(angle)).max() <= 3 * 2.0 ** -25
