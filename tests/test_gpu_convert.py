"""The device conversion of a caller's CSR: ragged rows, a last slice that is
not full, row pointers that do not start at 1, patterns without symmetry,
column spans on both sides of the 16-bit window, and every kind of invalid
matrix refused."""
import numpy as np
import pytest

from mixsolver_amd import linsolver
from mixsolver_amd._lib import MixSolverError

pytestmark = pytest.mark.gpu


def _ragged(n, seed, symmetric, span=None):
    """Diagonally dominant CSR (1-based) with 0..12 off-diagonals per row."""
    rng = np.random.default_rng(seed)
    m = rng.integers(0, 7 if symmetric else 13, n)
    i = np.repeat(np.arange(n), m)
    j = rng.integers(0, n, len(i))
    if span is not None:   # one entry exactly `span` columns away from another of its slice
        i, j = np.append(i % 64, [0, 0]), np.append(j % 64, [1, 1 + span])
    k = i != j
    i, j = i[k], j[k]
    if symmetric:
        i, j = np.concatenate([i, j]), np.concatenate([j, i])
    key = np.unique(i.astype(np.int64) * n + j)
    i, j = key // n, key % n
    w = rng.uniform(0.1, 1.0, len(i))
    if symmetric:
        lo, hi = np.minimum(i, j), np.maximum(i, j)
        w = 0.1 + ((lo * 7919 + hi * 104729) % 1000) / 1000.0
    rows, cols = np.concatenate([i, np.arange(n)]), np.concatenate([j, np.arange(n)])
    vals = np.concatenate([-w, np.bincount(i, w, n) * 1.2 + 0.5])
    o = np.lexsort((cols, rows))
    rp = (np.concatenate([[0], np.cumsum(np.bincount(rows, minlength=n))]) + 1).astype(np.int32)
    return rp, (cols[o] + 1).astype(np.int32), vals[o], rng.normal(size=n)


def _residual(rp, ci, val, b, x):
    row = np.repeat(np.arange(len(b)), np.diff(rp))
    return np.linalg.norm(b - np.bincount(row, val * x[ci - 1], len(b))) / np.linalg.norm(b)


@pytest.mark.parametrize("n,span", [(1, None), (63, None), (64, None), (65, None), (1000, None), (70000, 65533),
                                    (70000, 65534)])
def test_converted_systems_solve(n, span):
    for symmetric in (True, False):
        rp, ci, val, b = _ragged(n, n, symmetric, span)
        runs = [("bicgstab", "jacobi", "fp64")]
        if span is None:
            runs.append(("bicgstab", "natural", "fp64"))
        if symmetric:
            runs += [("pcg", "jacobi", "fp64")] + ([("pcg", "jacobi", "mixed")] if n >= 1000 else [])
        for solver, pc, prec in runs:
            x, it, res, ierr = linsolver.solve(rp, ci, val, b, np.zeros(n), 1e-10, 2000, solver=solver, precond=pc,
                                               precision=prec, inner_tol=0.1)
            assert ierr == 0 and res <= 1e-10, (solver, pc, prec, it, res, ierr)
            # the recursive residual and the true one part by rounding only
            assert _residual(rp, ci, val, b, x) <= 1.05e-10, (solver, pc, prec)


def test_row_pointers_may_start_later():
    rp, ci, val, b = _ragged(300, 5, True)
    x0 = linsolver.cg_jacobi(rp, ci, val, b, np.zeros(300), 1e-12, 500)[0]
    junk = np.full(7, 999999, np.int32)
    x1 = linsolver.cg_jacobi(rp + 7, np.concatenate([junk, ci]), np.concatenate([np.ones(7), val]), b, np.zeros(300),
                             1e-12, 500)[0]
    assert np.array_equal(x0, x1)


@pytest.mark.parametrize("fault", ["low", "high", "order", "twice", "diagonal", "pointer", "negative"])
def test_invalid_matrices_are_refused(fault):
    rp, ci, val, b = _ragged(200, 3, True)
    rp, ci = rp.copy(), ci.copy()
    a = rp[100] - 1
    r = next(i for i in range(100, 200) if rp[i + 1] - rp[i] >= 3)
    a = rp[r] - 1
    if fault == "low":
        ci[a] = 0
    elif fault == "high":
        ci[rp[r + 1] - 2] = 201
    elif fault == "order":
        ci[a], ci[a + 1] = ci[a + 1], ci[a]
    elif fault == "twice":
        ci[a + 1] = ci[a]
    elif fault == "diagonal":
        keep = np.ones(len(ci), bool)
        keep[a + np.flatnonzero(ci[a:rp[r + 1] - 1] == r + 1)[0]] = False
        ci, val = ci[keep], val[keep]
        rp[r + 1:] -= 1
    elif fault == "pointer":
        rp[r] = rp[-1] + 50
    else:
        rp[r] = -4
    with pytest.raises(MixSolverError):
        linsolver.cg_jacobi(rp, ci, val, b, np.zeros(200), 1e-10, 100)
