"""Meshes of triangles with no number in them: every node's boxes are NaN, those
that a leaf tile makes and those of the levels above it, as the oracle has them
(a union that begins with an empty box would make the latter infinite)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("budget", [0, 8 << 30], ids=["free", "under a budget"])
@pytest.mark.parametrize("n", [1, 2, 257, 2140, 24000, 100003])
def test_boxes_of_nothing(lb, ora, n, budget):
    tri = np.full((n, 12), np.nan, np.float32)
    for bounds in (None, np.array([0, 0, 0, 1, 1, 1], np.float32)):
        with lb.Context(0, hbm_budget=budget) as c:
            bvh, _, sk, pm = c.build_arrays(tri, bounds, keep_topology=True)
        wb, _, wsk, wpm = ora.build(tri, bounds, 0)
        assert np.array_equal(sk, wsk) and np.array_equal(pm, wpm)
        assert np.array_equal(bvh, wb)
