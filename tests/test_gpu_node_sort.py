"""GPU: the node sort of a batch whose fields' bin counts follow one another
unsorted: structured grids with a tile per block, grids without, a field that
only looks like a grid (which sends all of them to the packed order), small
after large, and the same handle set up again."""
import numpy as np
import pytest

import fluidtissue_amd as fa

pytestmark = pytest.mark.gpu


def _looks_like_a_grid(n, seed):
    """n^3 nodes with a unit box that are no grid; the tets of one, which need
    not be well shaped."""
    m = fa.kuhn_mesh(n)
    xyz = np.random.default_rng(seed).random((n ** 3, 3)).astype(np.float32)
    xyz[:8] = [[i, j, k] for i in (0, 1) for j in (0, 1) for k in (0, 1)]
    return fa.Mesh(xyz=xyz, tets=m.tets, edges=m.edges, t2e=m.t2e)


@pytest.mark.parametrize("mode", ["points", "triangles"])
@pytest.mark.parametrize("scattered", [False, True])
def test_batches_sort_as_their_fields_alone(mode, scattered):
    meshes = [fa.kuhn_mesh(d, jitter=0.1, seed=k) for k, d in enumerate((36, 2, (20, 8, 16), 5, (66, 4, 4), 17, 9))]
    if scattered:
        meshes.insert(3, _looks_like_a_grid(16, 1))
    phis = [np.linalg.norm(m.xyz.astype(np.float64) - 0.4 * m.xyz.max(0), axis=1) - 0.45 * m.xyz.max() for m in meshes]
    alone = []
    for m, phi in zip(meshes, phis):
        with fa.Reinit(0) as r:
            r.set_mesh(m)
            alone.append(r.reset_phi(phi, mode=mode)[0])
    with fa.Reinit(0) as r:
        for order in (range(len(meshes)), reversed(range(len(meshes))), range(len(meshes))):
            order = list(order)
            r.set_batch([meshes[k] for k in order])
            out, _, _ = r.reset_phi(np.concatenate([phis[k] for k in order]), mode=mode)
            assert np.array_equal(out.view(np.uint64), np.concatenate([alone[k] for k in order]).view(np.uint64))
