"""The per-stage tree kernels where their launches change (csrc/k_tree.hip):
the radix tree's few-tile resolve and the up pass's fan-in, against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# radix tree tiles of 4,096 gaps: 1, 2, 64 (the most without a scan), 65;
# up pass blocks of 1,024 leaves: 33 and 64 (one level by 64s), 65 and 1,024
# (two by 32s), 1,025 (two by 64s)
SIZES = [2, 4097, 4098, 33000, 65536, 65537, 64 * 4096 + 1, 64 * 4096 + 2, 1 << 20, (1 << 20) + 1]


@pytest.mark.parametrize("n", SIZES)
def test_parents_and_nodes(ctx, lb, ora, n):
    for tri in (lb.wl_uniform(n, n, 0.01), lb.wl_uniform(n, 7, 0.01)[np.arange(n) * 5 % 7]):
        b = lb.wl_bounds(tri)
        wb, _, wsk, _ = ora.build(tri, b, 0)
        d = ctx.to_device(tri)
        bufs = [ctx.alloc(k * n) for k in (32, 4, 4, 8, 64)]
        aabb, keys, idx, par, bvh = bufs
        try:
            ctx.aabb_morton(d, n, b, aabb, keys)
            ctx.sort(keys, idx, n)
            ctx.radix_tree(keys, n, par)
            ctx.up_pass(idx, aabb, par, n, bvh)
            ctx.synchronize()
            assert np.array_equal(par.read(np.int32, 2 * n), ora.radix_tree(wsk))
            assert np.array_equal(bvh.read(np.uint8, 64 * n), wb)
        finally:
            for x in [d] + bufs:
                x.destroy()
