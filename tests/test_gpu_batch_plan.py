"""The plan of a batch (tile tables on the device) after a call that ran out of
budget while it made one: the same call again makes it anew."""
import numpy as np
import pytest

from test_gpu_batched import make_batch

pytestmark = pytest.mark.gpu

BUDGET = 64 << 20


@pytest.mark.parametrize("before", [False, True], ids=["first", "after another batch"])
@pytest.mark.parametrize("with_bounds", [False, True])
def test_no_room_for_the_tables(lb, ora, with_bounds, before):
    meshes, offsets, tri = make_batch(lb, [3, 1, 0, 4097] + [5] * 300 + [1025], 40)
    bounds = None
    if with_bounds:
        bounds = np.concatenate([lb.wl_bounds(m) if len(m) else np.zeros(6, np.float32) for m in meshes])
    total = int(offsets[-1])
    with lb.Context(0, hbm_budget=BUDGET) as c:
        d, bvh, otri = c.to_device(tri), c.alloc(64 * total), c.alloc(48 * total)
        if before:
            c.build_batched(d, offsets[:4], None, bvh, otri)
        hog = c.alloc(BUDGET - c.bytes_in_use() - 64)
        for _ in range(2):
            with pytest.raises(lb.LBVHError) as err:
                c.build_batched(d, offsets, bounds, bvh, otri)
            assert err.value.code == lb.ERR_OUT_OF_BUDGET
        hog.destroy()
        c.build_batched(d, offsets, bounds, bvh, otri)
        got, gtri = bvh.read(np.uint8, 64 * total), otri.read(np.uint32, 12 * total)
    for k, m in enumerate(meshes):
        a, b = int(offsets[k]), int(offsets[k + 1])
        if a == b:
            continue
        wb, wo = ora.build(m, None if bounds is None else bounds[6 * k:6 * k + 6], 0)[:2]
        assert np.array_equal(got[64 * a:64 * b], wb), k
        assert np.array_equal(gtri[12 * a:12 * b], wo.view(np.uint32).ravel()), k
