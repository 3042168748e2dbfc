"""The layout of a level-scheduled sweep's packed entries, without a device: a
small program runs the library's planning code over level sizes and row widths
and checks that the steps cover every row once, that their places do not
overlap, and how many there are."""
import os
import shutil
import subprocess

import numpy as np
import pytest

SRC = os.path.join(os.path.dirname(__file__), "..", "mixsolver_amd", "csrc")

PROGRAM = r"""
#include <cstdio>
#include "ms_sweep_plan.hpp"
using namespace ms;
int main() {   // number of levels; per level its rows; per row its entries
  int nl;
  if (std::scanf("%d", &nl) != 1) return 1;
  std::vector<int> lev(1, 0), w;
  for (int l = 0, x; l < nl && std::scanf("%d", &x) == 1; l++) lev.push_back(lev.back() + x);
  for (int t = 0, x; t < lev.back() && std::scanf("%d", &x) == 1; t++) w.push_back(x);
  std::vector<LevSeg> segs;
  for (int l = 0, e; l < nl; l = e) {
    e = l + 1;
    const bool narrow = lev[l + 1] - lev[l] <= kNarrowRows;
    while (narrow && e < nl && lev[e + 1] - lev[e] <= kNarrowRows) e++;
    segs.push_back({l, e, narrow});
  }
  const SweepSteps S = sweep_steps(lev, segs, [&](int t) { return w[t]; });
  long long end = 0;
  int row = 0;
  for (const auto &g : segs) {
    const int last = g.s1;
    for (int s = g.s0; s < last; s++) {
      const SweepStep &d = S.st[s];
      if (d.t0 != row || d.n < 1 || d.base < end || (g.narrow && d.n > g.block)) return 2;
      for (int t = d.t0; t < d.t0 + d.n; t++)
        if (w[t] > d.w) return 3;
      row += d.n;
      end = d.base + (long long)d.w * d.stride;
      if (d.stride < d.n) return 4;
    }
    for (int s = last; g.narrow && s < last + kTailSteps; s++)
      if (s >= (int)S.st.size() || S.st[s].n != 0) return 5;
  }
  if (row != lev.back() || end != S.nent) return 6;
  std::printf("%lld %d\n", S.nent, (int)sweep_packs(2 * S.nent, 0));
  return 0;
}
"""


@pytest.fixture(scope="module")
def places(tmp_path_factory):
    if not shutil.which("g++"):
        pytest.skip("no host compiler")
    d = tmp_path_factory.mktemp("plan")
    (d / "plan.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", SRC, "plan.cpp", "-o", "plan"], cwd=d, check=True)

    def run(levels, widths):
        text = " ".join(map(str, [len(levels), *levels, *widths]))
        r = subprocess.run([str(d / "plan")], input=text, capture_output=True, text=True)
        assert r.returncode == 0, r.returncode
        nent, packs = map(int, r.stdout.split())
        return nent, bool(packs)
    return run


@pytest.mark.parametrize("rows", [1, 2, 3, 63])
@pytest.mark.parametrize("width", [1, 3, 9])
def test_narrow_levels_take_no_more_than_their_entries(places, rows, width):
    """Chains and bands: levels of a few rows, whose places follow the entries
    and not the number of levels."""
    nl = 20000 // rows
    nent, _ = places([rows] * nl, [width] * (rows * nl))
    assert nent == rows * nl * width


@pytest.mark.parametrize("widest", [2, 4, 5, 9])
def test_levels_of_all_sizes(places, widest):
    """Levels on both sides of a wavefront, a workgroup and a run: at most
    twice their rows' widest, and one wavefront per step to align it."""
    rng = np.random.default_rng(widest)
    levels = [1, 64, 2048, 2049, 65, 1024, 1025, 63, 5000] + [int(x) for x in rng.integers(1, 3000, 60)]
    n = sum(levels)
    nent, _ = places(levels, rng.integers(0, widest + 1, n))
    assert nent <= 2 * widest * n + 64 * (n // 64 + len(levels))


def test_a_long_row_in_a_wide_level_is_not_packed(places):
    """One row of 3,000 entries among 100,000 of one: its level would take
    3,000 places a row."""
    nent, packs = places([100000], [1] * 99999 + [3000])
    assert nent > 1e8 and not packs
    nent, packs = places([100000], [3] * 100000)
    assert nent <= 300200 and packs
