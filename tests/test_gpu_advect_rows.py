"""GPU: the solver's sparse products over row slices that share few diagonals
(col - row, one mask per row), over slices with too many of them (columns per
entry), and over meshes with both, against the oracle."""
import numpy as np
import pytest

import fluidtissue_amd as fa
import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,shuffled", [
    ((2, 2, 2), 0.0),          # one slice, 8 rows
    ((5, 4, 3), 0.0),          # 60 rows: rows of several lines and planes in one slice
    ((64, 4, 4), 0.0),         # slices that are whole lines
    ((13, 11, 9), 0.0),        # 1287 rows: 20 slices and 7 rows
    ((13, 11, 9), 0.4),        # the first nodes renumbered at random: both kinds of slice
    ((13, 11, 9), 1.0),        # all of them
])
def test_products_match_the_oracle(n, shuffled):
    m = fa.kuhn_mesh(n, jitter=0.15, seed=5)
    N = len(m.xyz)
    rng = np.random.default_rng(3)
    new_of = np.arange(N, dtype=np.int32)
    k = int(shuffled * N)
    new_of[:k] = rng.permutation(k)
    xyz = np.empty_like(m.xyz)
    xyz[new_of] = m.xyz
    m = fa.Mesh(xyz=xyz, tets=np.ascontiguousarray(new_of[m.tets]),
                edges=np.ascontiguousarray(new_of[m.edges]), t2e=m.t2e)
    x = m.xyz.astype(np.float64)
    phi = x[:, 0] - 0.4 + 0.1 * np.sin(5 * x[:, 1])
    flow = np.concatenate([rng.standard_normal(3 * N), np.zeros(N)])
    dt, tol = 0.01, 1e-11
    r = fa.Reinit(0)
    r.set_mesh(m)
    got, info = r.advect(phi, flow, dt, tol=tol, max_iters=500)
    r.close()
    # as for other meshes: both stop at |b - L x| <= tol |b|, 1e-8 of |phi|
    ref, rinfo = oracle.advect(m.xyz, m.tets, phi, flow, dt, tol=tol, max_iters=500)
    assert info["converged"] and rinfo["converged"] and not info["skipped"]
    assert np.max(np.abs(got - ref)) <= 1e-8 * np.max(np.abs(phi))
    ro, co, L, b = oracle.advect_system(m.xyz, m.tets, phi, flow, dt)
    res = b - oracle.spmv(ro, co, L, got)
    assert np.linalg.norm(res) <= 1.01 * tol * np.linalg.norm(b)


@pytest.mark.parametrize("pair", [(0, 1), (1, 2), (2, 3), (0, 3)])
def test_tets_that_name_a_node_twice(pair):
    """Their determinant is rarely computed as exactly 0 on a jittered mesh, and
    then both of the node's terms go into one entry, one after the other."""
    m = fa.kuhn_mesh(9, jitter=0.2, seed=3)
    N = len(m.xyz)
    rng = np.random.default_rng(1)
    tets = m.tets.copy()
    k = rng.choice(len(tets), 200, replace=False)
    tets[k, pair[1]] = tets[k, pair[0]]
    tets[k[:20], :] = tets[k[:20], :1]                     # one node four times
    vel = rng.standard_normal(3 * N)
    ro, co = oracle.fem_pattern(N, tets)
    with fa.Reinit(0) as r:
        r.set_mesh(fa.Mesh(xyz=m.xyz, tets=tets, edges=m.edges, t2e=m.t2e))
        for form, args in ((0, ()), (1, (vel,))):
            off, cols, got = r.fem_matrix(form, *args)
            want, _ = oracle.fem_assemble(form, m.xyz, tets, ro, co, *args)
            assert np.array_equal(off, ro) and np.array_equal(cols, co)
            assert np.array_equal(got.view(np.uint64), want.view(np.uint64))
