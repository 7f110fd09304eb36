"""GPU: the scans of a reinit on both sides of the sizes where one workgroup
does a whole scan (8192 elements: words of the edge bitmap at 42^3 and 43^3,
groups of tets at 71^3 and 72^3, points and triangles in between; 32768
leaves), against the oracle; and stages that outgrow what they were sized
for by the call before."""
import numpy as np
import pytest

import fluidtissue_amd as fa
import oracle
from tests.helpers import assert_interface_bit_exact

pytestmark = pytest.mark.gpu


def _interface(m, phi):
    ifp, ifp2e = oracle.find_interface_nodes(m.edges, m.xyz, phi)
    tris, elems, area = oracle.reconstruct_interface(m.tets, m.t2e, m.edges, m.xyz, phi, ifp, ifp2e)
    return dict(ifp=ifp, ifp2e=ifp2e, tris=tris, if_elems=elems, ifp_area=area)


@pytest.mark.parametrize("n", [2, 33, 42, 43, 71, 72])
def test_scans_match_the_oracle(n):
    m = fa.kuhn_mesh(n, jitter=0.2, seed=n)
    small = np.linalg.norm(m.xyz.astype(np.float64) - 0.5, axis=1) - 0.11
    large = fa.phi_field("star", m.xyz, seed=3)
    if n == 2:                                       # a corner cut off, then half of the cell
        small, large = (m.xyz.astype(np.float64) @ w - 0.4 for w in ([1.0, 1.1, 1.2], [1.0, 0.1, 0.2]))
    r = fa.Reinit(0)
    r.set_mesh(m)
    # the first call reads its totals back; the second is sized by the first,
    # which it outgrows; the third runs within the second's sizes
    for phi in (small, large, small):
        ref = _interface(m, phi)
        out, ifn, cnt = r.reset_phi(phi, mode="triangles")
        assert (cnt.n_ifp, cnt.n_tri, cnt.n_if_elems) == (len(ref["ifp"]), len(ref["tris"]), len(ref["if_elems"]))
        assert_interface_bit_exact(r.interface(), ref)
        out, ifn, cnt = r.reset_phi(phi, mode="points")
        nodes = np.random.default_rng(n).permutation(m.n_nodes)[:2000]
        d, _ = oracle.point_distance(m.xyz, ref["ifp"], nodes)
        assert np.array_equal(np.abs(ifn[nodes]), d.astype(np.float64))
    r.close()
