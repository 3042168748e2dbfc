"""Fields of a system read from other threads: while one thread runs a driver,
the run stays what it is without readers, bit for bit, and two threads that
read different fields at once each get their own."""
import threading
import time

import numpy as np
import pytest

from mixsolver_amd import meshgen
from mixsolver_amd.solver import Case

pytestmark = pytest.mark.gpu

CTL = """rho = 1.0
mu = 0.0055
transient = true
dt = 0.005
n_time_max = 1
n_correct = 2
time_scheme = 2
lin_tol = 1e-10
lin_max = 20000
ppe_precond = jacobi
body_force = 1.0 0.0 0.0
bc = 5 wall
periodic = 7 6
periodic = 9 8
"""


def _case(**over):
    m = meshgen.channel(32, 20, 12, periodic=True)
    cs = Case.from_control(m, CTL, gpu_mom_precond=2, gpu_coarse=16, **over)
    u = np.random.default_rng(5).uniform(-0.5, 0.5, size=(m.ncells, 3))
    u[:, 0] += 15.0
    cs.set_field("u", u)
    return cs


@pytest.mark.parametrize("over", [dict(gpu_ppe_precond=2, gpu_precision=0),
                                  dict(gpu_ppe_precond=0, gpu_ppe_solver=2, gpu_precision=1)])
def test_reading_beside_a_run_changes_nothing(over):
    res = []
    for readers in (0, 2):
        cs = _case(**over)
        assert cs.info["renumbered"]
        stop, reads, errors = threading.Event(), [0] * 2, []

        def read(i):
            try:
                while not stop.is_set():
                    for k in (("u", "flux"), ("p", "gu"))[i]:
                        assert np.all(np.isfinite(cs.get(k)))
                    reads[i] += 1
                    time.sleep(1e-3)
            except BaseException as e:   # noqa: B902 -- reported by the main thread
                errors.append(e)
        ts = [threading.Thread(target=read, args=(i,)) for i in range(readers)]
        for t in ts:
            t.start()
        ier = cs.piso_run(4)
        stop.set()
        for t in ts:
            t.join()
        assert ier == 0 and not errors, errors
        assert min(reads[:readers], default=1) > 0
        res.append([cs.get(k) for k in ("u", "p", "flux")] + [cs.history()])
        cs.close()
    for a, b in zip(*res):
        assert np.array_equal(a, b)


def test_threads_read_their_own_fields():
    cs = _case(gpu_ppe_precond=2)
    rng = np.random.default_rng(6)
    want = {k: rng.normal(size=cs.get(k).shape) for k in ("u", "p", "gu", "T")}
    for k, v in want.items():
        cs.set_field(k, v)
    bad = []

    def read(k):
        for _ in range(50):
            if not np.array_equal(cs.get(k), want[k]):
                bad.append(k)
    ts = [threading.Thread(target=read, args=(k,)) for k in want]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad, bad
    cs.close()


def test_systems_end_beside_a_server():
    """Systems are destroyed while a server's worker runs and captures its
    rounds on the library stream: every request is solved, and as alone."""
    from mixsolver_amd.serve import LaplacianPattern, Server, request_mesh
    P = LaplacianPattern(request_mesh(5000, "hex", seed=1))
    rng = np.random.default_rng(8)
    reqs = [(P.values(rng), P.rhs(rng)) for _ in range(3)]
    systems = [_case(gpu_ppe_precond=2) for _ in range(12)]
    srv = Server(precond="dilu", coarse=0, round_iters=4)
    pid = srv.add_pattern(P.row_ptr, P.col_idx, P.xc)
    alone = [srv.result(srv.submit(pid, v, b, tol=1e-10, maxit=5000), timeout_ms=-1)["x"] for v, b in reqs]
    stop, bad, solved = threading.Event(), [], [0]

    def serve():
        try:
            while not stop.is_set():
                tickets = [srv.submit(pid, v, b, tol=1e-10, maxit=5000) for v, b in reqs]
                for t, x in zip(tickets, alone):
                    r = srv.result(t, timeout_ms=-1)
                    if r["ierr"] != 0 or not np.array_equal(r["x"], x):
                        bad.append(r["ierr"])
                    solved[0] += 1
        except BaseException as e:   # noqa: B902 -- reported by the main thread
            bad.append(e)
    th = threading.Thread(target=serve)
    th.start()
    for cs in systems:
        time.sleep(5e-3)
        cs.close()
    stop.set()
    th.join()
    srv.close()
    assert not bad and solved[0] >= 3, bad
