"""The routes of a batched build: sort tiles of 1,024 keys up to 2^23 triangles
in all and k_forest.hip's leaf tiles up to 7 * 2^19, larger tiles and k_tree.hip's
past them or under an HBM budget; meshes that begin at any offset, whole and part tiles."""
import numpy as np
import pytest

from test_gpu_batched import make_batch, run_batch

pytestmark = pytest.mark.gpu

SMALL = [1, 1023, 1024, 1025, 3, 4096, 4097, 4095, 255, 257, 16385, 2, 70001]
MIDDLE = SMALL + [262144, 131073, 100003] * 7  # 3.6M
LARGE = SMALL + [262144, 131073, 100003] * 16  # 7.9M
# meshes of more sort tiles than bounds blocks, and empty ones
FEW = [3, 600001, 0, 0, 1030, 524289, 0, 7] + [0] * 300 + [2]
LARGER = LARGE + [262144, 262143]              # past 2^23


@pytest.mark.parametrize("bits", [8, 10])
@pytest.mark.parametrize("with_bounds", [False, True])
@pytest.mark.parametrize("sizes", [SMALL, FEW, MIDDLE, LARGE, LARGER], ids=["small", "few", "middle", "large", "larger"])
def test_routes_agree(lb, ora, sizes, with_bounds, bits):
    meshes, offsets, tri = make_batch(lb, sizes, 300)
    bounds = None
    if with_bounds:
        bounds = np.concatenate([lb.wl_bounds(m) if len(m) else np.zeros(6, np.float32) for m in meshes])
    outs = []
    for budget in (0, 64 << 30):
        with lb.Context(0, hbm_budget=budget) as c:
            c.set_tuning(lb.TUNE_SORT_BITS, bits)
            outs.append(run_batch(c, tri, offsets, bounds))
    for a, b in zip(*outs):
        assert np.array_equal(a.view(np.uint8), b.view(np.uint8))
    bvh, otri, sk, pm = outs[0]
    for k in list(range(len(SMALL))) + [len(sizes) - 1]:
        a, b = int(offsets[k]), int(offsets[k + 1])
        if a == b:
            continue
        wb, wo, wsk, wpm = ora.build(meshes[k], None if bounds is None else bounds[6 * k:6 * k + 6], 0)
        assert np.array_equal(sk[a:b], wsk) and np.array_equal(pm[a:b], wpm), k
        assert np.array_equal(bvh[64 * a:64 * b], wb), k
        assert np.array_equal(otri[a:b].view(np.uint32), wo.view(np.uint32)), k
