"""What a two-stage transform there and back does to each frequency (pair_round_trip, which the propagators divide by):
against a line taken through both layouts with the source's own radices and float32 constants in float64, compiled on the
host. And the compact groups of the row pass: none holds low and high kept columns at once.
"""
import os
import shutil
import subprocess

import numpy as np
import pytest

from tests.test_pair_index_math import pair_ra

import simulatokit_amd as sk

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LENGTHS = [65, 91, 121, 225, 486, 600, 1000, 1008]
PROGRAM = r"""
#include <cstdio>
#include <vector>
#include "sk_pair.h"
namespace sk {
std::vector<float2> pair_roots_of(int m);
std::vector<double> pair_round_trip(int m, bool columns);
}
using V = double2;
static V mul(V a, V b) { return {a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x}; }
template <int M, int SIGN>
void there(const V* in, V* out, const float2* w) {  // elements (layout I) to frequencies (layout Q)
  constexpr int RA = sk::pair_ra(M), RB = M / RA;
  static V lds[RA][RB];
  for (int i = 0; i < RB; ++i) {
    V u[RA];
    for (int r = 0; r < RA; ++r) u[r] = in[i + RB * r];
    sk::rdft<RA, SIGN>(u);
    for (int q = 0; q < RA; ++q) lds[q][i] = u[q];
  }
  for (int q = 0; q < RA; ++q) {
    V v[RB];
    for (int p = 0; p < RB; ++p) v[p] = mul(lds[q][p], {w[RA * p + q].x, SIGN < 0 ? w[RA * p + q].y : -w[RA * p + q].y});
    sk::rdft<RB, SIGN>(v);
    for (int p = 0; p < RB; ++p) out[q + RA * p] = v[p];
  }
}
template <int M, int SIGN>
void back(const V* in, V* out, const float2* w) {  // layout Q to layout I
  constexpr int RA = sk::pair_ra(M), RB = M / RA;
  static V lds[RA][RB];
  for (int q = 0; q < RA; ++q) {
    V v[RB];
    for (int p = 0; p < RB; ++p) v[p] = in[q + RA * p];
    sk::rdft<RB, SIGN, true>(v);
    for (int p = 0; p < RB; ++p)
      lds[q][p] = mul(v[p], {w[M + RA * p + q].x, SIGN < 0 ? w[M + RA * p + q].y : -w[M + RA * p + q].y});
  }
  for (int i = 0; i < RB; ++i) {
    V u[RA];
    for (int q = 0; q < RA; ++q) u[q] = lds[q][i];
    sk::rdft<RA, SIGN, true>(u);
    for (int r = 0; r < RA; ++r) out[i + RB * r] = u[r];
  }
}
template <int M>
void show() {
  const auto w = sk::pair_roots_of(M);
  const auto gc = sk::pair_round_trip(M, true), gr = sk::pair_round_trip(M, false);
  std::vector<V> e(M), f(M), g(M);
  for (int k = 0; k < M; ++k) {
    for (int j = 0; j < M; ++j) e[j] = {j == k ? 1.0 : 0.0, 0.0};
    back<M, +1>(e.data(), f.data(), w.data());   // a column pass: to the rows of the grid, then to the frequencies
    there<M, -1>(f.data(), g.data(), w.data());
    const double c = g[k].x / M;
    there<M, +1>(e.data(), f.data(), w.data());  // a row pass
    back<M, -1>(f.data(), g.data(), w.data());
    printf("%d %d %.17g %.17g %.17g %.17g\n", M, k, c, gc[k], g[k].x / M, gr[k]);
  }
}
int main() { LINES }
"""


@pytest.fixture(scope="module")
def gains(tmp_path_factory):
    lib = sk._native.LIB_PATH
    if shutil.which("hipcc") is None or not os.path.exists(lib):
        pytest.skip("no hipcc, or the library is not built")
    d = tmp_path_factory.mktemp("gains")
    (d / "gains.hip").write_text(PROGRAM.replace("LINES", " ".join(f"show<{m}>();" for m in LENGTHS)))
    subprocess.run(["hipcc", "-O1", "-std=c++17", "--cuda-host-only", "-I", os.path.join(ROOT, "simulatokit_amd", "csrc"),
                    "-I", os.path.join(ROOT, "include"), str(d / "gains.hip"), "-L", os.path.dirname(lib),
                    "-lsimulato_hip", f"-Wl,-rpath,{os.path.dirname(lib)}", "-o", str(d / "gains")], check=True, capture_output=True, timeout=110)
    out = subprocess.run([str(d / "gains")], check=True, capture_output=True, text=True, timeout=100).stdout
    return np.array([[float(v) for v in line.split()] for line in out.splitlines()])


@pytest.mark.parametrize("m", LENGTHS)
def test_gains_are_those_of_the_lines(gains, m):
    _, k, col, want_col, row, want_row = gains[gains[:, 0] == m].T
    assert np.array_equal(k, np.arange(m))
    # the diagonal's terms are rounded in float64, m of them at most
    assert np.abs(col - want_col).max() <= m * 2.0 ** -52 and np.abs(row - want_row).max() <= m * 2.0 ** -52
    # float32 constants, not exact ones, and not the same for rows and columns where the radices differ
    assert np.abs(want_col - 1).max() > 1e-9 and np.abs(want_col - 1).max() < 3e-7
    assert m in (121, 225) or np.abs(want_col - want_row).max() > 1e-9


@pytest.mark.parametrize("m", [m for m in range(65, 1025) if pair_ra(m)])
def test_no_compact_group_is_low_and_high(m):
    ra = pair_ra(m)
    rb, k = m // ra, m // 3
    assert not any(rb * r <= k and rb * (r + 1) - 1 >= m - k for r in range(ra))
