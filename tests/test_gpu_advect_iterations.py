"""GPU: an iteration of the solve is enqueued ahead of the one whose residual is
awaited; what is enqueued past the last must change nothing: the iteration
counts and solutions of limits and tolerances around where it stops."""
import numpy as np
import pytest

import fluidtissue_amd as fa

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
