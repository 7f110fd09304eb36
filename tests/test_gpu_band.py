"""GPU: what a narrow band's search leaves out -- the nodes clamped per field,
counted over runs of 1024 tiles that hold one field or several."""
import numpy as np
import pytest

import fluidtissue_amd as fa
import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", ["points", "triangles"])
@pytest.mark.parametrize("sizes", [[44], [45, 9, 3], [6, 44, 20, 45, 4]])
def test_clamped_nodes_are_those_without_a_nearest(mode, sizes):
    h = 1.0 / (max(sizes) - 1)
    meshes = [fa.kuhn_mesh(n, spacing=h, jitter=0.1, seed=2) for n in sizes]
    phis = [np.linalg.norm(m.xyz.astype(np.float64) - 0.4 * h * n, axis=1) - 0.2 * h * n for n, m in zip(sizes, meshes)]
    r = fa.Reinit(0)
    if len(sizes) == 1:
        r.set_mesh(meshes[0])
        off = np.array([0, meshes[0].n_nodes])
    else:
        r.set_batch(meshes)
        off, _, _ = r.batch_info()
    band = 2.5 * h
    _, ifn, cnt = r.reset_phi(np.concatenate(phis), mode=mode, band=band, want_nearest=True)
    none = r.nearest() == -1
    per_field = [int(none[off[k]:off[k + 1]].sum()) for k in range(len(sizes))]
    got = [c.n_clamped for c in r.field_counts()] if len(sizes) > 1 else [cnt.n_clamped]
    assert got == per_field and cnt.n_clamped == sum(per_field) > 0
    assert np.array_equal(np.abs(ifn[none]), np.full(none.sum(), np.float64(np.float32(band))))
    # every node the full search finds inside the band keeps its distance
    _, full, _ = r.reset_phi(np.concatenate(phis), mode=mode)
    sure = np.abs(np.abs(full) / band - 1) > 1e-5          # (rounding decides at the band's edge)
    inside = (np.abs(full) < band) & sure
    assert np.array_equal(inside[sure], ~none[sure])
    assert np.array_equal(ifn[inside].view(np.uint64), full[inside].view(np.uint64))
    r.close()


@pytest.mark.parametrize("mode", ["points", "triangles"])
@pytest.mark.parametrize("n,bin_scale,band_h", [(5, 1e6, 1.0), (9, 0.0, 0.2), (33, 0.0, 0.7), (33, 0.0, 100.0), (68, 0.5, 4.0),
                                                (68, 0.0, 9.0), ((130, 7, 5), 0.0, 3.0)])
def test_tiles_left_out_have_no_primitive_in_the_band(mode, n, bin_scale, band_h):
    """Tiles are left out whole, by boxes above the leaves: from one-leaf trees to
    three levels, bands below a spacing to the whole field."""
    dims = (n, n, n) if np.isscalar(n) else n
    h = 1.0 / (max(dims) - 1)
    m = fa.kuhn_mesh(dims, spacing=h, jitter=0.2, seed=3)
    mid = 0.5 * h * (np.array(dims) - 1)
    phi = np.linalg.norm((m.xyz - mid) / (mid + h), axis=1) - 0.55
    band = band_h * h
    with fa.Reinit(0) as r:
        r.set_mesh(m)
        _, full, _ = r.reset_phi(phi, mode=mode, bin_scale=bin_scale)
        out, ifn, cnt = r.reset_phi(phi, mode=mode, bin_scale=bin_scale, band=band, want_nearest=True)
        none = r.nearest() == -1
        again, _, _ = r.reset_phi(phi, mode=mode, bin_scale=bin_scale, band=band, schedule="queue", query_block=256)
    assert np.array_equal(out.view(np.uint64), again.view(np.uint64))
    sure = np.abs(np.abs(full) / band - 1) > 1e-5          # (rounding decides at the band's edge)
    inside = (np.abs(full) < band) & sure
    assert np.array_equal(inside[sure], ~none[sure]) and cnt.n_clamped == none.sum()
    assert np.array_equal(ifn[inside].view(np.uint64), full[inside].view(np.uint64))
    assert np.array_equal(np.abs(ifn[none]), np.full(none.sum(), np.float64(np.float32(band))))


@pytest.mark.parametrize("schedule", ["static", "queue", "bins"])
@pytest.mark.parametrize("band", [0.05, 0.13])
def test_band_of_a_batch_matches_the_oracle(schedule, band):
    """Every node of every field against the FP64 brute force over that field's
    triangles: the nodes within the band have their distance and nearest
    triangle (ties aside), the others +-band and none, and these are counted.
    (Rounding decides for nodes within 1e-5 h of the band's edge.)"""
    dims = [24, (30, 20, 13), 17, (9, 33, 21)]
    kinds = ["star", "spheres", "ellipsoids", "sphere_wave"]
    meshes = [fa.kuhn_mesh(d, jitter=0.15, seed=k) for k, d in enumerate(dims)]
    phis = [fa.phi_field(k, m.xyz, seed=9 + j) for j, (k, m) in enumerate(zip(kinds, meshes))]
    with fa.Reinit(0) as r:
        r.set_batch(meshes)
        off, _, _ = r.batch_info()
        _, ifn, cnt = r.reset_phi(np.concatenate(phis), mode="triangles", band=band, want_nearest=True, schedule=schedule)
        near, per = r.nearest(), r.field_counts()
    b32 = float(np.float32(band))
    first = 0
    for k, (m, phi) in enumerate(zip(meshes, phis)):
        h = 1.0 / (max(np.atleast_1d(dims[k])) - 1)
        ifp, ifp2e = oracle.find_interface_nodes(m.edges, m.xyz, phi)
        tris, _, _ = oracle.reconstruct_interface(m.tets, m.t2e, m.edges, m.xyz, phi, ifp, ifp2e)
        nodes = np.arange(m.n_nodes)
        d64, f64 = oracle.triangle_distance(m.xyz, ifp, tris, nodes)
        got, nr = ifn[off[k]:off[k + 1]], near[off[k]:off[k + 1]]
        none = nr == -1
        inside, beyond = d64 < b32 - 1e-5 * h, d64 > b32 + 1e-5 * h
        assert inside.any() and beyond.any()
        assert not none[inside].any() and none[beyond].all()
        assert np.array_equal(np.signbit(got), phi < 0)
        assert np.max(np.abs(np.abs(got[~none]) - d64[~none])) <= 1e-5 * h
        assert np.all(np.abs(got[none]) == b32)
        for i in np.nonzero(~none & (nr - first != f64))[0]:          # a tie: as near as the oracle's
            dg = oracle.node_triangle_distance(i, m.xyz, ifp, tris, nr[i] - first)
            assert abs(dg - d64[i]) <= 1e-5 * h
        assert per[k].n_clamped == none.sum() and per[k].n_tri == len(tris)
        first += len(tris)
    assert cnt.n_clamped == sum(c.n_clamped for c in per)


def test_bins_schedule_is_for_a_band_to_the_triangles():
    m = fa.kuhn_mesh(9)
    phi = m.xyz[:, 0].astype(np.float64) - 0.4
    with fa.Reinit(0) as r:
        r.set_mesh(m)
        r.reset_phi(phi, mode="triangles", band=0.2, schedule="bins")
        for mode, band in (("points", 0.2), ("triangles", 0.0), ("points", 0.0)):
            with pytest.raises(fa._lib.FtError) as e:
                r.reset_phi(phi, mode=mode, band=band, schedule="bins")
            assert e.value.code == fa._lib.FT_ERR_ARG


@pytest.mark.parametrize("mode", ["points", "triangles"])
@pytest.mark.parametrize("sizes", [[26], [24, 9, 31]])
def test_captured_band_replays(mode, sizes):
    """A band's two streams inside a captured graph: every replay, on other
    level sets and with eager work in between, equals the eager call."""
    import torch
    meshes = [fa.kuhn_mesh(n, jitter=0.1, seed=n) for n in sizes]
    xyz = np.concatenate([m.xyz for m in meshes]).astype(np.float64)
    band = 0.15
    with fa.Reinit(0) as r, fa.Reinit(0) as e:
        for h in (r, e):
            h.set_batch(meshes)
        d = torch.empty(len(xyz), dtype=torch.float64, device="cuda")
        di = torch.empty_like(d)
        for k in range(5):
            phi = np.linalg.norm(xyz - 0.5, axis=1) - (0.3, 0.31, 0.2, 0.42, 0.3)[k]
            want, ifn, cnt = e.reset_phi(phi, mode=mode, band=band)
            d.copy_(torch.from_numpy(phi))
            torch.cuda.synchronize()
            per = r.reset_phi_graph_device(d.data_ptr(), di.data_ptr(), mode=mode, band=band)
            torch.cuda.synchronize()
            assert np.array_equal(d.cpu().numpy().view(np.uint64), want.view(np.uint64))
            assert np.array_equal(di.cpu().numpy().view(np.uint64), ifn.view(np.uint64))
            clamped = [c.n_clamped for c in e.field_counts()]
            assert [c.n_clamped for c in per] == clamped and sum(clamped) == cnt.n_clamped > 0
