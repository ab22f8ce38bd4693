"""The tree levels of small meshes on the GPU (csrc/k_forest.hip), where their
tiles, levels and stores change: builds and refits against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# one tile, two; 64 and 65 leaf tiles (one item level, two); the last size
# with direct node stores, then past it
SIZES = [1, 2, 63, 65, 255, 256, 257, 16384, 16385, 40001, 131072, 131073, 1 << 21, (1 << 21) + 1]


@pytest.mark.parametrize("n", SIZES)
def test_build_and_refit(ctx, lb, ora, n):
    kinds = [lb.wl_uniform(n, n, 0.01)]
    if n < 1 << 20:  # one key: deltas from the positions alone; few keys
        kinds += [np.tile(lb.wl_uniform(1, 1, 0.01), (n, 1)), lb.wl_uniform(n, 7, 0.01)[np.arange(n) * 5 % 7]]
    for tri in kinds:
        bvh, otri, sk, pm = ctx.build_arrays(tri, None, keep_topology=True)
        wb, wo, wsk, wpm = ora.build(tri, None, 0)
        assert np.array_equal(sk, wsk) and np.array_equal(pm, wpm)
        assert np.array_equal(bvh, wb)
        assert np.array_equal(otri.view(np.uint32), wo.view(np.uint32))
        moved = lb.wl_jitter(3, tri, 0.001)
        bufs = [ctx.to_device(x) for x in (moved, sk, pm)] + [ctx.alloc(64 * n), ctx.alloc(48 * n)]
        try:
            dt, ds, dp, db, do = bufs
            ctx.refit(dt, n, ds, dp, db, do)
            rb, ro = ora.refit(moved, wsk, wpm)
            assert np.array_equal(db.read(np.uint8, 64 * n), rb)
            assert np.array_equal(do.read(np.uint32, 12 * n), ro.view(np.uint32).ravel())
        finally:
            for b in bufs:
                b.destroy()


@pytest.mark.parametrize("n", [300, 100000, 7 << 19, (7 << 19) + 1, 1 << 23, (1 << 23) + 1])
def test_routes_agree(lb, n):
    """Free, under a budget (which takes the larger leaf tile) and with the
    tile fixed: the same words, up to the largest mesh and past it."""
    side = int(np.sqrt(n / 2)) + 1
    tri = lb.wl_heightfield(9, side, side)[:n]
    outs = []
    for budget, tile in [(0, 0), (64 << 30, 0), (0, 512)]:
        with lb.Context(0, hbm_budget=budget) as c:
            if tile:
                c.set_tuning(lb.TUNE_TREE_TILE, tile)
            outs.append(c.build_arrays(tri, None)[:2])
    for bvh, otri in outs[1:]:
        assert np.array_equal(outs[0][0], bvh)
        assert np.array_equal(outs[0][1].view(np.uint32), otri.view(np.uint32))
