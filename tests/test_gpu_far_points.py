"""GPU: EuclideanDistance's points far outside the mesh, where the index takes
larger units, in turn with points inside it (and with reinits) on one handle,
against the oracle."""
import numpy as np
import pytest

import fluidtissue_amd as fa
import oracle
from fluidtissue_amd._lib import check, lib

pytestmark = pytest.mark.gpu


def _points(rng, n, at, radius):
    v = rng.standard_normal((n, 3))
    return (np.array(at) + radius * v / np.linalg.norm(v, axis=1)[:, None]).astype(np.float32)


def _oracle(xyz, ifp, phi):
    ref = oracle.reset_phi_points(xyz, ifp, phi.copy())
    return ref[0] if isinstance(ref, tuple) else ref


@pytest.mark.parametrize("dims,shift", [((14, 14, 14), 0.0), ((25, 9, 3), 0.0), ((14, 14, 14), 300.0)])
def test_far_and_near_points_in_turn(dims, shift):
    m = fa.kuhn_mesh(dims, jitter=0.1, seed=3)
    xyz = (m.xyz + np.float32(shift)).astype(np.float32)
    mid = np.full(3, shift) + 0.5 * m.xyz.max(0)
    rng = np.random.default_rng(4)
    phi = rng.standard_normal(len(xyz))
    outlier = _points(rng, 1, mid, 1e6)
    clouds = [
        _points(rng, 400, mid, 0.3),                              # inside
        _points(rng, 400, mid + [8, 0, 0], 1.0),                  # to one side
        _points(rng, 400, mid, 2.0),                              # about where the units change
        _points(rng, 400, mid, 3.1),
        np.concatenate([outlier, _points(rng, 400, mid, 0.3)]),   # the first point says nothing of the rest
        _points(rng, 400, mid - [0, 40, 40], 30.0),
        np.concatenate([np.full((5, 3), np.nan, np.float32), outlier, _points(rng, 50, mid + [0, 0, 900], 2.0)]),
        _points(rng, 3, mid, 1e19),
        _points(rng, 400, mid, 0.4),
    ]
    with fa.EuclideanDistance(0) as d:
        d.init(xyz)
        for ifp in clouds:
            got = phi.copy()
            d.reset_phi(ifp, len(ifp), got)
            assert np.array_equal(got.view(np.uint64), _oracle(xyz, ifp, phi).view(np.uint64))


def test_far_points_between_reinits():
    """The same handle's reinits, eager and captured, keep their results."""
    import torch
    m = fa.kuhn_mesh(20, jitter=0.1, seed=5)
    field = fa.phi_field("ellipsoids", m.xyz, seed=6)
    rng = np.random.default_rng(7)
    phi = rng.standard_normal(m.n_nodes)
    far = _points(rng, 300, [12, 0, 0], 1.0)
    with fa.Reinit(0) as r:
        r.set_mesh(m)
        d0 = torch.from_numpy(field).cuda()
        d = d0.clone()
        want = None
        for _ in range(3):
            out, _, _ = r.reset_phi(field, mode="points", bin_scale=2.0)
            d.copy_(d0)
            torch.cuda.synchronize()
            r.reset_phi_graph_device(d.data_ptr(), None, mode="points", bin_scale=2.0)
            torch.cuda.synchronize()
            want = out if want is None else want
            assert np.array_equal(out.view(np.uint64), want.view(np.uint64))
            assert np.array_equal(d.cpu().numpy().view(np.uint64), want.view(np.uint64))
            got = phi.copy()
            check(lib.ft_reset_phi_points(r._h, far.ctypes.data, len(far), got.ctypes.data))
            assert np.array_equal(got.view(np.uint64), _oracle(m.xyz, far, phi).view(np.uint64))
