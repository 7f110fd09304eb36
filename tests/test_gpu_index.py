"""GPU: the index's tree where its shape changes, against the oracle.  Bins per
axis that give 1 to 4 levels of nodes (1, 2, 4, 5, 16, 17, 64, 71), bins that
hold one primitive or all of them, tiles split over waves and whole, narrow
bands, and interfaces the scaled coordinates do not hold (points far outside
the mesh, non-finite ones)."""
import numpy as np
import pytest

import fluidtissue_amd as fa
import oracle

pytestmark = pytest.mark.gpu


def _check_points(m, ifn, nodes, ifp):
    d, _ = oracle.point_distance(m.xyz, ifp, nodes)
    assert np.array_equal(np.abs(ifn[nodes]), d.astype(np.float64))


def _check_triangles(m, h, ifn, near, nodes, itf):
    """Within 1e-5 h of the FP64 brute force, the nearest triangle outside ties."""
    d64, f64 = oracle.triangle_distance(m.xyz, itf[0], itf[1], nodes)
    err = np.abs(np.abs(ifn[nodes]) - d64)
    assert err.max() <= 1e-5 * h
    for k in np.nonzero(near[nodes] != f64)[0]:
        dg = oracle.node_triangle_distance(nodes[k], m.xyz, itf[0], itf[1], near[nodes][k])
        assert abs(dg - d64[k]) <= 1e-5 * h


@pytest.mark.parametrize("n,bin_scale", [(9, 1e6), (9, 4.0), (9, 2.0), (9, 1.6), (17, 1.0), (18, 1.0), (33, 0.5),
                                         (72, 1.0), (21, 20.0), ((5, 40, 3), 1.0), ((300, 12, 10), 2.0)])
@pytest.mark.parametrize("field", ["sphere_wave", "ellipsoids"])
def test_tree_shapes_match_the_oracle(n, bin_scale, field):
    dims = (n, n, n) if np.isscalar(n) else n
    h = 1.0 / (max(dims) - 1)
    m = fa.kuhn_mesh(dims, spacing=h, jitter=0.2, seed=2)
    phi = fa.phi_field(field, m.xyz, seed=4)
    ifp, ifp2e = oracle.find_interface_nodes(m.edges, m.xyz, phi)
    if len(ifp) == 0:                              # the field misses this thin slab: cut its long side by a plane
        phi = m.xyz[:, int(np.argmax(dims))].astype(np.float64) - 0.37
        ifp, ifp2e = oracle.find_interface_nodes(m.edges, m.xyz, phi)
    tris, _, _ = oracle.reconstruct_interface(m.tets, m.t2e, m.edges, m.xyz, phi, ifp, ifp2e)
    nodes = np.random.default_rng(1).permutation(m.n_nodes)[:4000]
    with fa.Reinit(0) as r:
        r.set_mesh(m)
        _, ifn, _ = r.reset_phi(phi, mode="points", bin_scale=bin_scale)
        _check_points(m, ifn, nodes, ifp)
        out, ifn, _ = r.reset_phi(phi, mode="triangles", bin_scale=bin_scale, want_nearest=True)
        _check_triangles(m, h, ifn, r.nearest(), nodes, (ifp, tris))
        whole, _, _ = r.reset_phi(phi, mode="triangles", bin_scale=bin_scale, schedule="queue")   # no tile is split
        assert np.array_equal(out.view(np.uint64), whole.view(np.uint64))
        band = 2.5 * h
        _, bnd, cnt = r.reset_phi(phi, mode="triangles", bin_scale=bin_scale, band=band)
        # in the band the distance is the full domain's; beyond it +-band
        inside = np.abs(ifn) < np.float32(band)
        assert np.array_equal(bnd[inside].view(np.uint64), ifn[inside].view(np.uint64))
        beyond = np.abs(ifn) > np.float32(band) * (1 + 1e-6)
        assert np.array_equal(np.abs(bnd[beyond]), np.full(beyond.sum(), np.float64(np.float32(band))))
        assert cnt.n_clamped >= beyond.sum()


@pytest.mark.parametrize("scale", [1.0, 3.0, 100.0, 1e7])
def test_points_outside_the_mesh(scale):
    """EuclideanDistance::resetPhi takes any points, also far from the mesh."""
    m = fa.kuhn_mesh(20, jitter=0.1, seed=3)
    rng = np.random.default_rng(5)
    ifp = ((rng.random((500, 3)) - 0.5) * 2 * scale).astype(np.float32)
    phi = rng.standard_normal(m.n_nodes)
    ref = oracle.reset_phi_points(m.xyz, ifp, phi.copy())
    ref = ref[0] if isinstance(ref, tuple) else ref
    with fa.EuclideanDistance(0) as d:
        d.init(m.xyz)
        got = phi.copy()
        d.reset_phi(ifp, len(ifp), got)
    assert np.array_equal(got.view(np.uint64), ref.view(np.uint64))


def test_non_finite_points_do_not_hide_the_others():
    """A NaN or infinite point never wins, and the finite points that share its
    bin are still found."""
    m = fa.kuhn_mesh(16)
    rng = np.random.default_rng(6)
    good = rng.random((300, 3)).astype(np.float32)
    bad = good[:40].copy()
    bad[::2, 0] = np.nan
    bad[1::2, 1] = np.inf
    ifp = np.concatenate([bad, good])
    phi = rng.standard_normal(m.n_nodes)
    ref = oracle.reset_phi_points(m.xyz, good, phi.copy())
    ref = ref[0] if isinstance(ref, tuple) else ref
    with fa.EuclideanDistance(0) as d:
        d.init(m.xyz)
        got = phi.copy()
        d.reset_phi(ifp, len(ifp), got)
    assert np.array_equal(got.view(np.uint64), ref.view(np.uint64))


@pytest.mark.parametrize("n", [16, 24])
def test_scattered_nodes_that_count_and_bound_like_a_grid(n):
    """n^3 nodes over the unit cube, its corners among them, but not a grid:
    blocks of 4 x 4 x 4 spacings hold any number of nodes."""
    rng = np.random.default_rng(n)
    xyz = rng.random((n ** 3, 3)).astype(np.float32)
    xyz[:8] = [[i, j, k] for i in (0, 1) for j in (0, 1) for k in (0, 1)]
    xyz[8:200] = xyz[8]                                   # more than a tile in one place
    ifp = rng.random((400, 3)).astype(np.float32)
    phi = rng.standard_normal(n ** 3)
    ref = oracle.reset_phi_points(xyz, ifp, phi.copy())
    ref = ref[0] if isinstance(ref, tuple) else ref
    with fa.EuclideanDistance(0) as d:
        d.init(xyz)
        got = phi.copy()
        d.reset_phi(ifp, len(ifp), got)
    assert np.array_equal(got.view(np.uint64), ref.view(np.uint64))
