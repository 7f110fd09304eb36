"""GPU: an iteration of the solve is enqueued ahead of the one whose residual is
awaited; what is enqueued past the last must change nothing: the iteration
counts and solutions of limits and tolerances around where it stops."""
import ctypes as C

import numpy as np
import pytest

import fluidtissue_amd as fa
import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [3, 14])
def test_limits_around_the_last_iteration(n):
    m = fa.kuhn_mesh(n, jitter=0.1, seed=1)
    N = len(m.xyz)
    rng = np.random.default_rng(7)
    phi = m.xyz[:, 0].astype(np.float64) - 0.4
    flow = np.concatenate([rng.standard_normal(3 * N), np.zeros(N)])
    r = fa.Reinit(0)
    r.set_mesh(m)
    got, info = r.advect(phi, flow, 0.01, tol=1e-10)
    last = info["iterations"]
    assert info["converged"] and last >= 2
    same, again = r.advect(phi, flow, 0.01, tol=1e-10, max_iters=last)   # nothing may be enqueued past it
    assert again["iterations"] == last and np.array_equal(same.view(np.uint64), got.view(np.uint64))
    for short in (1, last - 1):
        with pytest.raises(fa._lib.FtError) as e:
            r.advect(phi, flow, 0.01, tol=1e-10, max_iters=short)
        assert e.value.code == fa._lib.FT_ERR_SOLVER
    # loose tolerances: fewer iterations, each stop's residual above the next's
    counts = [r.advect(phi, flow, 0.01, tol=t)[1] for t in (0.5, 1e-2, 1e-4, 1e-10)]
    assert all(a["iterations"] <= b["iterations"] and a["error"] >= b["error"]
               for a, b in zip(counts, counts[1:]))
    assert counts[-1]["iterations"] == last and counts[-1]["error"] == info["error"]
    r.close()


@pytest.mark.parametrize("n,kind", [(2, "rotation"), (3, "rotation"), (5, "random"), (9, "random"), (14, "rotation")])
def test_restart(n, kind):
    """A tolerance below what r0 can tell (|r0.r| < eps^2 |r0|^2, reached near
    |r| = 1e-32 |b|) makes the solve restart from its true residual; iterations
    that were enqueued past that point must change nothing."""
    m = fa.kuhn_mesh(n, jitter=0.1 if n > 2 else 0.0, seed=1)
    N = len(m.xyz)
    x = m.xyz.astype(np.float64)
    phi = x[:, 0] - 0.4 + 0.1 * np.sin(5 * x[:, 1])
    v = (np.random.default_rng(7).standard_normal(3 * N) if kind == "random" else
         np.concatenate([-(x[:, 1] - 0.5), x[:, 0] - 0.5, 0.3 * np.sin(3 * x[:, 0])]))
    flow = np.concatenate([v, np.zeros(N)])
    dt, tol = 0.01, 1e-40
    ref, rinfo = oracle.advect(m.xyz, m.tets, phi, flow, dt, tol=tol, max_iters=400)
    assert rinfo["converged"] and rinfo["restarts"] > 0
    with fa.Reinit(0) as r:
        r.set_mesh(m)
        got, info = r.advect(phi, flow, dt, tol=tol, max_iters=400)
        last = info["iterations"]
        assert info["converged"] and info["error"] <= tol and info["restarts"] > 0
        assert np.max(np.abs(got - ref)) <= 1e-8 * np.max(np.abs(phi))
        ro, co, L, b = oracle.advect_system(m.xyz, m.tets, phi, flow, dt)
        assert np.linalg.norm(b - oracle.spmv(ro, co, L, got)) <= 1e-13 * np.linalg.norm(b)
        # limits from one iteration to one past the last: the count starts again
        # at the first restart, and a limit reached before it, or between it and
        # the last iteration, stops exactly there
        stopped = {}
        for limit in range(1, last + 2):
            out = phi.copy()
            i = fa._lib.FtAdvectInfo()
            rc = fa._lib.lib.ft_advect(r._h, out.ctypes.data, flow.ctypes.data, dt, tol, limit, C.byref(i))
            if rc == 0:
                assert i.converged and i.iterations == last and np.array_equal(out.view(np.uint64), got.view(np.uint64))
            else:
                assert rc == fa._lib.FT_ERR_SOLVER and i.iterations == limit and not i.converged
                assert i.error > tol and np.array_equal(out, phi)
                stopped[limit] = (i.restarts, i.error)
        before = [k for k, s in stopped.items() if s[0] == 0]        # limits reached before the first restart
        assert before == list(range(1, len(before) + 1)) and len(before) > 0
        if last > len(before):                                        # a limit between the two: the restart has happened
            assert all(stopped[k][0] > 0 for k in range(len(before) + 1, last))
            assert last not in stopped and last + 1 not in stopped
