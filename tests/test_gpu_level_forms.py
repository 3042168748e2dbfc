"""Natural-order factorizations and sweeps in the forms that the patterns of
test_gpu_levels.py do not reach.  x after k iterations against the oracle's:
the order of operations is the reference's, so it differs by the rounding of
the solver's dot products only (bars as there: CG 1e-10, BiCGSTAB 1e-9)."""
import numpy as np
import pytest

from mixsolver_amd import linsolver

pytestmark = pytest.mark.gpu


def _against_oracle(kind, n, pairs, one_sided=(), seed=11):
    """pairs: (row, lower neighbour) arrays of a symmetric pattern; one_sided:
    (row, column) arrays without their transpose"""
    from oracle import pyoracle
    rng = np.random.default_rng(seed)
    skew = 0.0 if kind == "cg_ic0" else 0.3
    rows, cols, vals = [np.arange(n)], [np.arange(n)], [np.zeros(n)]
    for i, j in pairs:
        w = rng.uniform(0.5, 1.5, len(i))
        rows += [i, j]
        cols += [j, i]
        vals += [-w * (1 + skew), -w * (1 - skew)]
    for i, j in one_sided:
        rows.append(i)
        cols.append(j)
        vals.append(-rng.uniform(0.5, 1.5, len(i)))
    rows, cols, vals = (np.concatenate(v) for v in (rows, cols, vals))
    vals[:n] = np.bincount(rows, np.abs(vals), n) * rng.uniform(1.01, 1.2, n) + 0.1
    o = np.lexsort((cols, rows))
    rp = (np.concatenate([[0], np.cumsum(np.bincount(rows, minlength=n))]) + 1).astype(np.int32)
    ci, val = (cols[o] + 1).astype(np.int32), vals[o]
    b = rng.normal(size=n)
    bar = 1e-10 if kind == "cg_ic0" else 1e-9
    for k in (1, 2, 4):
        x, it, _, ierr = getattr(linsolver, kind)(rp, ci, val, b, np.zeros(n), 1e-13, k)
        xr, itr, _, ierrr = pyoracle.solve(kind, rp, ci, val, b, np.zeros(n), 1e-13, k)
        assert (it, ierr) == (itr, ierrr), k
        assert np.linalg.norm(x - xr) <= bar * np.linalg.norm(xr), k
    if not one_sided:   # the FP32 factor and sweeps
        x, _, res, ierr = linsolver.solve(rp, ci, val, b, np.zeros(n), 1e-10, 2000,
                                          solver="pcg" if kind == "cg_ic0" else "bicgstab", precond="natural",
                                          precision="mixed", inner_tol=0.1)
        assert ierr == 0 and res <= 1e-10


@pytest.mark.parametrize("kind", ["cg_ic0", "bicgstab_ilu0"])
def test_long_rows_among_short_ones(kind):
    """A level of 20,000 rows of one lower entry and a few of 200, beside runs
    of narrow levels: too wide a step to pack, so the sweeps read the matrix's
    own layout, wide levels and runs both."""
    m, w, t = 10000, 20000, 3000
    n = m + w + t
    rng = np.random.default_rng(2)
    i = np.arange(m, m + w)
    pairs = [(i, rng.integers(0, m, w))]
    for r in (m + 7, m + 10000, m + w - 1):   # 200 more neighbours, none of them the first
        first = pairs[0][1][r - m]
        j = rng.permutation(np.delete(np.arange(m), first))[:200]
        pairs.append((np.full(200, r), j))
    c = np.arange(m + w, n)
    pairs += [(c, c - 1), (c, rng.integers(0, m, t))]
    _against_oracle(kind, n, pairs)


def _grid(m):
    """rows and lower neighbours of an m^3 seven-point grid, and of the (-1, -1,
    0) diagonal, which closes triangles; every level is a plane of up to 3 m^2 /
    4 rows, so narrow runs and levels of over 2,048 rows follow one another"""
    i = np.arange(m ** 3)
    x, y, z = i % m, i // m % m, i // (m * m)
    axes = [(i[x > 0], i[x > 0] - 1), (i[y > 0], i[y > 0] - m), (i[z > 0], i[z > 0] - m * m)]
    d = (x > 0) & (y > 0)
    return axes, (i[d], i[d] - 1 - m)


@pytest.mark.parametrize("kind", ["cg_ic0", "bicgstab_ilu0"])
def test_general_factor_of_wide_and_narrow_levels(kind):
    """A pattern with triangles takes the general elimination: a launch per
    wide level, one workgroup per run of narrow ones, in turn."""
    axes, diagonal = _grid(64)
    _against_oracle(kind, 64 ** 3, axes + [diagonal])


@pytest.mark.parametrize("where", ["lower", "upper"])
def test_general_factor_of_an_asymmetric_pattern(where):
    """Entries without a transpose (ILU(0) only), with their triangles."""
    axes, (i, j) = _grid(64)
    _against_oracle("bicgstab_ilu0", 64 ** 3, axes, [(i, j) if where == "lower" else (j, i)])
