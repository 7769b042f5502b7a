"""Calls on one system from several threads: downloads beside each other and
beside a solve, and gradients of several lattices, return what they return
alone, bit for bit (vectors and gradient inputs pass through kept buffers of
the system)."""
import threading

import numpy as np
import pytest

import parmoon_amd as pa
from parmoon_amd import prm as P

pytestmark = pytest.mark.gpu


def run_threads(calls, reps):
    """Each of `calls` `reps` times in a thread of its own, started together:
    its results in the order of the calls."""
    out = [[] for _ in calls]
    errors = []
    start = threading.Barrier(len(calls))

    def work(call, res):
        try:
            start.wait(30)
            for _ in range(reps):
                res.append(call())
        except Exception as e:
            errors.append(e)

    threads = [threading.Thread(target=work, args=a) for a in zip(calls, out)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors
    return out


def test_downloads_beside_each_other_and_a_solve(ctx):
    print("[case] rhs of two levels, solution and solve in four threads, 33^3 Q1", flush=True)
    S = pa.System(ctx, 3, 3, 1)
    S.assemble(P.config1b())
    rhs = S.rhs()
    n, na = int(S.dims()[0]), int(S.dims()[1])
    sol0 = np.zeros(n)
    sol0[na:] = rhs[na:]
    opt = P.solver_opt(solver=16, restart=20, maxit=12, res_norm_min=0.0, red_factor=0.0, smoother=3, omega=1.0)
    S.solve_resident(opt, check=False)
    want = [S.rhs(), S.rhs(level=0), S.solution()]
    # downloads of vectors that no call changes
    got = run_threads([S.rhs, lambda: S.rhs(level=0), S.solution], 40)
    for w, g in zip(want, got):
        assert len(g) == 40 and all(np.array_equal(w, a) for a in g)
    # beside solves with a caller's vectors (the cycle is captured by now)
    b = 0.5 * rhs
    alone, _, _ = S.solve(opt, b, sol0, check=False)
    got = run_threads([lambda: S.solve(opt, b, sol0, check=False)[0], S.rhs, lambda: S.rhs(level=1)], 12)
    assert all(np.array_equal(alone, a) for a in got[0])
    assert all(np.array_equal(want[0], a) for a in got[1])
    assert all(np.array_equal(S.rhs(level=1), a) for a in got[2])
    S.close()


def test_gradients_of_several_lattices(ctx):
    """129^3 is beyond the size whose buffers stay allocated."""
    print("[case] network gradients on 129^3, 33^3 and 5^3 in three threads", flush=True)
    S = pa.System(ctx, 1, 2, 1)
    S.assemble(P.config1b())
    S.learned_init(11)
    rng = np.random.default_rng(4)
    data = [(rng.standard_normal((M, M, M, 16), np.float32), rng.standard_normal((M, M, M), np.float32))
            for M in (129, 33, 5)]
    want = [S.learned_gradient(u, t) for u, t in data]
    got = run_threads([lambda u=u, t=t: S.learned_gradient(u, t) for u, t in data], 6)
    for (g, l), res in zip(want, got):
        assert all(np.array_equal(g, a) and l == b for a, b in res)
    S.close()
