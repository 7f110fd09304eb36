"""GPU: crossing points and nodes that are not finite: such points are nobody's
nearest, such nodes have none, and neither changes anything for the rest."""
import ctypes as C

import numpy as np
import pytest

import fluidtissue_amd as fa
import oracle
from fluidtissue_amd._lib import check, lib

pytestmark = pytest.mark.gpu

FLT_MAX = float(np.finfo(np.float32).max)


@pytest.mark.parametrize("n_bad", [1, 3, 17, 63, 64, 65, 200])
def test_only_nan_points_after_a_larger_call(n_bad):
    """A leaf of NaN points alone, where the call before left its points."""
    m = fa.kuhn_mesh(16, jitter=0.1, seed=3)
    rng = np.random.default_rng(6)
    phi = rng.standard_normal(m.n_nodes)
    with fa.EuclideanDistance(0) as d:
        d.init(m.xyz)
        good = rng.random((300, 3)).astype(np.float32)
        d.reset_phi(good, len(good), phi.copy())
        got = phi.copy()
        d.reset_phi(np.full((n_bad, 3), np.nan, np.float32), n_bad, got)
        near = np.empty(m.n_nodes, np.int32)
        check(lib.ft_get_nearest(d._h, near.ctypes.data_as(C.c_void_p)))
    assert np.array_equal(got, np.where(phi < 0, -FLT_MAX, FLT_MAX))
    assert np.all(near == -1)


@pytest.mark.parametrize("mode", ["points", "triangles"])
def test_field_with_only_nan_points_in_a_batch(mode):
    """phi infinite on both sides of every crossing edge: the field's points are
    NaN, and the next field's are not its own."""
    small, big = fa.kuhn_mesh(2), fa.kuhn_mesh(12, jitter=0.1, seed=4)
    bad = np.full(small.n_nodes, np.inf)
    bad[0] = -np.inf
    fine = fa.phi_field("ellipsoids", big.xyz, seed=2)
    with fa.Reinit(0) as r:
        r.set_mesh(big)
        alone, _, _ = r.reset_phi(fine, mode=mode, want_nearest=True)
        near_alone = r.nearest()
    for first in (True, False):
        meshes, phis = ([small, big], [bad, fine]) if first else ([big, small], [fine, bad])
        with fa.Reinit(0) as r:
            r.set_batch(meshes)
            off, _, _ = r.batch_info()
            out, _, _ = r.reset_phi(np.concatenate(phis), mode=mode, want_nearest=True)
            near = r.nearest()
            cnt = r.field_counts()
        k = 0 if first else 1
        b, f = slice(off[k], off[k + 1]), slice(off[1 - k], off[2 - k])
        assert cnt[k].n_ifp > 0
        assert np.array_equal(out[b], np.where(bad < 0, -FLT_MAX, FLT_MAX)) and np.all(near[b] == -1)
        assert np.array_equal(out[f].view(np.uint64), alone.view(np.uint64))
        before = cnt[k].n_ifp if mode == "points" else cnt[k].n_tri
        assert np.array_equal(near[f], near_alone + (before if first else 0))


@pytest.mark.parametrize("share", [0.002, 0.3, 0.97, 1.0])
def test_nan_nodes_beside_others(share):
    """Nodes with a NaN coordinate share tiles with finite ones, as their first,
    last or most nodes."""
    m = fa.kuhn_mesh(17, jitter=0.1, seed=5)
    rng = np.random.default_rng(8)
    xyz = m.xyz.copy()
    bad = rng.random(len(xyz)) < share
    bad[:8] = True                                    # among the first nodes of the first tiles
    xyz[bad, rng.integers(0, 3, bad.sum())] = np.nan
    ifp = rng.random((700, 3)).astype(np.float32)
    phi = rng.standard_normal(len(xyz))
    ref = oracle.reset_phi_points(xyz, ifp, phi.copy())
    ref = ref[0] if isinstance(ref, tuple) else ref
    with fa.EuclideanDistance(0) as d:
        d.init(xyz)
        got = phi.copy()
        d.reset_phi(ifp, len(ifp), got)
    assert np.array_equal(got.view(np.uint64), ref.view(np.uint64))
    assert np.all(np.abs(got[bad]) == FLT_MAX) and np.all(np.abs(got[~bad]) < 2)


@pytest.mark.parametrize("mode", ["points", "triangles"])
@pytest.mark.parametrize("band", [0.0, 0.2])
def test_nan_nodes_away_from_the_interface(mode, band):
    m = fa.kuhn_mesh(18, jitter=0.1, seed=6)
    phi = np.linalg.norm(m.xyz.astype(np.float64) - 0.5, axis=1) - 0.2
    bad = np.zeros(m.n_nodes, bool)
    bad[[0, 3, 17, 40, 324, m.n_nodes - 1]] = True    # of tets that do not cross
    hurt = fa.Mesh(xyz=np.where(bad[:, None], np.float32(np.nan), m.xyz), tets=m.tets, edges=m.edges, t2e=m.t2e)
    res = []
    for mesh in (m, hurt):
        with fa.Reinit(0) as r:
            r.set_mesh(mesh)
            out, ifn, _ = r.reset_phi(phi, mode=mode, blend="update", band=band, want_nearest=True)
            res.append((out, ifn, r.nearest()))
    (o1, i1, n1), (o2, i2, n2) = res
    assert np.array_equal(o1[~bad].view(np.uint64), o2[~bad].view(np.uint64))
    assert np.array_equal(i1[~bad].view(np.uint64), i2[~bad].view(np.uint64))
    assert np.array_equal(n1[~bad], n2[~bad]) and np.all(n2[bad] == -1)


@pytest.mark.parametrize("mode", ["points", "triangles"])
@pytest.mark.parametrize("band", [0.0, 0.2])
@pytest.mark.parametrize("value", [np.inf, -np.inf, 3e38])
def test_box_without_a_size(mode, band, value):
    """A node at infinity, or two so far apart that their difference is: the
    others' results are those of the mesh without."""
    m = fa.kuhn_mesh(14, jitter=0.1, seed=7)
    phi = np.linalg.norm(m.xyz.astype(np.float64) - 0.5, axis=1) - 0.2
    far = np.array([m.n_nodes - 1, 0] if np.isfinite(value) else [m.n_nodes - 1])   # of tets that do not cross
    xyz = m.xyz.copy()
    xyz[far, 1] = value * np.array([1, -1])[:len(far)]
    res = []
    for mesh in (m, fa.Mesh(xyz=xyz, tets=m.tets, edges=m.edges, t2e=m.t2e)):
        with fa.Reinit(0) as r:
            r.set_mesh(mesh)
            out, ifn, _ = r.reset_phi(phi, mode=mode, band=band, want_nearest=True)
            res.append((np.delete(ifn, far), np.delete(r.nearest(), far)))
    assert np.array_equal(res[0][0].view(np.uint64), res[1][0].view(np.uint64))
    assert np.array_equal(res[0][1], res[1][1])


@pytest.mark.parametrize("value", [1e15, 1e20, 1e25, 1e37])
def test_huge_nodes_beside_others(value):
    """Nodes whose squares overflow (beyond 1.8e19) or dwarf the rest."""
    m = fa.kuhn_mesh(15, jitter=0.1, seed=5)
    rng = np.random.default_rng(8)
    xyz = m.xyz.copy()
    bad = rng.random(len(xyz)) < 0.05
    bad[:8] = True
    xyz[bad, rng.integers(0, 3, bad.sum())] = value * rng.choice([-1, 1], bad.sum())
    ifp = rng.random((500, 3)).astype(np.float32)
    phi = rng.standard_normal(len(xyz))
    ref = oracle.reset_phi_points(xyz, ifp, phi.copy())
    ref = ref[0] if isinstance(ref, tuple) else ref
    with fa.EuclideanDistance(0) as d:
        d.init(xyz)
        got = phi.copy()
        d.reset_phi(ifp, len(ifp), got)
    assert np.array_equal(got.view(np.uint64), ref.view(np.uint64))


@pytest.mark.parametrize("mode", ["points", "triangles"])
@pytest.mark.parametrize("band", [0.0, 0.2])
@pytest.mark.parametrize("value", [1e6, 1e22, 1e33, 3e38])
def test_one_node_far_off(mode, band, value):
    """A box whose size is one far node's: the others' results stay."""
    m = fa.kuhn_mesh(14, jitter=0.1, seed=7)
    phi = np.linalg.norm(m.xyz.astype(np.float64) - 0.5, axis=1) - 0.2
    xyz = m.xyz.copy()
    xyz[-1, 2] = value                                  # of tets that do not cross
    res = []
    for mesh in (m, fa.Mesh(xyz=xyz, tets=m.tets, edges=m.edges, t2e=m.t2e)):
        with fa.Reinit(0) as r:
            r.set_mesh(mesh)
            _, ifn, _ = r.reset_phi(phi, mode=mode, band=band, want_nearest=True)
            res.append((ifn[:-1], r.nearest()[:-1]))
    assert np.array_equal(res[0][0].view(np.uint64), res[1][0].view(np.uint64))
    assert np.array_equal(res[0][1], res[1][1])


@pytest.mark.parametrize("mode", ["points", "triangles"])
@pytest.mark.parametrize("band", [0.0, 0.12])
@pytest.mark.parametrize("share", [0.01, 0.4])
def test_level_sets_with_nan_and_infinity(mode, band, share):
    """Crossing points and triangles that are not finite among others: the
    finite ones' distances are the oracle's."""
    m = fa.kuhn_mesh(15, jitter=0.1, seed=2)
    rng = np.random.default_rng(3)
    phi = fa.phi_field("ellipsoids", m.xyz, seed=5)
    bad = rng.random(m.n_nodes) < share
    phi[bad] = rng.choice([np.nan, -np.nan, np.inf, -np.inf], bad.sum())
    with np.errstate(all="ignore"):
        ifp, ifp2e = oracle.find_interface_nodes(m.edges, m.xyz, phi)
        tris, _, _ = oracle.reconstruct_interface(m.tets, m.t2e, m.edges, m.xyz, phi, ifp, ifp2e)
    with fa.Reinit(0) as r:
        r.set_mesh(m)
        _, ifn, cnt = r.reset_phi(phi, mode=mode, band=band, want_nearest=True)
        near, itf = r.nearest(), r.interface()
    assert np.array_equal(itf.ifp, ifp, equal_nan=True) and cnt.n_tri == len(tris)
    assert not np.isfinite(ifp).all()
    h, nodes = 1.0 / 14, np.arange(m.n_nodes)
    limit = float(np.float32(band)) if band else FLT_MAX
    if mode == "points":
        d, j = oracle.point_distance(m.xyz, ifp, nodes)
        d = d.astype(np.float64)
        tol = 0.0
    else:
        ok = np.isfinite(ifp[tris[:, :3]]).all((1, 2))
        assert ok.any() and not ok.all()
        d, j = oracle.triangle_distance(m.xyz, ifp, np.ascontiguousarray(tris[ok]), nodes)
        d = np.where(np.isfinite(d), d, FLT_MAX)
        tol = 1e-5 * h
    none = near == -1
    if band:
        assert none[d > limit + 1e-5 * h].all() and not none[d < limit - 1e-5 * h].any()
    else:
        assert not none.any()
    assert np.all(np.abs(ifn[none]) == limit)
    assert np.max(np.abs(np.abs(ifn[~none]) - d[~none])) <= tol
    assert np.array_equal(np.signbit(ifn), phi < 0)
