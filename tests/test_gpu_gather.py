"""The leaf levels' two forms of the triangle gather (tree_util.h: a wave picks by
how its leaves' triangles lie): meshes in order, shuffled, and half of each, whose
waves take either, against the oracle's build."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def meshes(lb, n):
    side = int(np.sqrt(n / 2)) + 1
    near = lb.wl_heightfield(n, side, side)[:n]  # neighbours in the mesh are neighbours in space
    far = near[np.random.default_rng(n).permutation(n)]
    return [near, far, np.concatenate([near[:n // 2], far[:n - n // 2]])]


# waves, tiles of 256 and 512 leaves: one short, whole, one past
@pytest.mark.parametrize("tile", [0, 512])
@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 127, 255, 257, 511, 513, 1023, 1025, 40003, 300001])
def test_builds(lb, ora, n, tile):
    with lb.Context(0) as c:
        if tile:  # k_tree.hip's leaf level
            c.set_tuning(lb.TUNE_TREE_TILE, tile)
        for tri in meshes(lb, n):
            bvh, otri = c.build_arrays(tri, None)[:2]
            wb, wo = ora.build(tri, None, 0)[:2]
            assert np.array_equal(bvh, wb)
            assert np.array_equal(otri.view(np.uint32), wo.view(np.uint32))
