"""Level-scheduled natural-order sweeps on patterns that reach every form of
their step: one-row levels, levels wider than a workgroup, rows with more
entries than are fetched ahead, and neighbours further back in the level
order than the workgroup's ring of recent values (16384 positions), with
vectors in row order (narrow levels) and in level order (wide ones).

The sweeps keep the reference's order of operations, so after k iterations
x differs from the oracle's only by the rounding of the solver's dot
products: bars as for the reference's solver histories (CG 1e-10,
BiCGSTAB 1e-9)."""
import numpy as np
import pytest

from mixsolver_amd import linsolver

pytestmark = pytest.mark.gpu


def _couplings(name):
    """(n, list of (row, lower neighbour) arrays)."""
    def chain(n, *lags):
        i = np.arange(n)
        return n, [(i[lag:], i[:-lag]) for lag in lags]
    if name == "one":
        return 1, []
    if name == "two":
        return chain(2, 1)
    if name == "more":          # nine lower entries in most rows
        return chain(700, 1, 2, 3, 5, 8, 13, 21, 34, 55)
    if name == "far":           # one-row levels, neighbours 17000 positions back
        return chain(20000, 1, 17000)
    if name == "edge":          # the ring's last and first position, and one beyond
        return chain(17000, 1, 16383, 16384, 16385)
    if name == "wide":          # 60 levels of 600 rows, neighbours 24000 back: level order
        return chain(36000, 600, 24000)
    assert name == "split"      # levels of 1100 rows: two steps each
    return chain(12100, 1100)


@pytest.mark.parametrize("kind", ["cg_ic0", "bicgstab_ilu0"])
@pytest.mark.parametrize("name", ["one", "two", "more", "far", "edge", "wide", "split"])
def test_sweeps_against_oracle(name, kind):
    from oracle import pyoracle
    rng = np.random.default_rng(11)
    n, pairs = _couplings(name)
    rows, cols, vals = [np.arange(n)], [np.arange(n)], [np.zeros(n)]
    for i, j in pairs:
        w = rng.uniform(0.5, 1.5, len(i))
        skew = 0.0 if kind == "cg_ic0" else 0.3
        rows += [i, j]
        cols += [j, i]
        vals += [-w * (1 + skew), -w * (1 - skew)]
    rows, cols, vals = (np.concatenate(v) for v in (rows, cols, vals))
    diag = np.bincount(rows, np.abs(vals), n) * rng.uniform(1.01, 1.2, n) + 0.1
    vals[:n] = diag
    o = np.lexsort((cols, rows))
    rp = (np.concatenate([[0], np.cumsum(np.bincount(rows, minlength=n))]) + 1).astype(np.int32)
    ci, val = (cols[o] + 1).astype(np.int32), vals[o]
    b = rng.normal(size=n)
    bar = 1e-10 if kind == "cg_ic0" else 1e-9
    for k in (1, 2, 4):
        x, it, res, ierr = getattr(linsolver, kind)(rp, ci, val, b, np.zeros(n), 1e-13, k)
        xr, itr, resr, ierrr = pyoracle.solve(kind, rp, ci, val, b, np.zeros(n), 1e-13, k)
        assert (it, ierr) == (itr, ierrr), k
        assert np.linalg.norm(x - xr) <= bar * np.linalg.norm(xr), k
    x, _, res, ierr = linsolver.solve(rp, ci, val, b, np.zeros(n), 1e-10, 2000,
                                      solver="pcg" if kind == "cg_ic0" else "bicgstab", precond="natural",
                                      precision="mixed", inner_tol=0.1)
    assert ierr == 0 and res <= 1e-10
