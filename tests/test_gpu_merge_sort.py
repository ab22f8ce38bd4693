"""The merge sort of small meshes on the GPU, where its tiles, chunks, rounds
and searches change: against numpy's stable sort and the oracle's build."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# a wave's keys, the tile, the runs of a round (8, 16, 32 tiles), two rounds
# (8 and 16 runs left), the largest, and the first that takes radix passes
SIZES = [1, 2, 127, 129, 2047, 2048, 2049, 4095, 16384, 16385, 32769, 65535, 65536, 65537, 131073, 262143, 262144,
         262145]


@pytest.mark.parametrize("n", SIZES)
def test_sort(ctx, n):
    rng = np.random.default_rng(n)
    half = np.arange(n) < n // 2
    for keys in (rng.integers(0, 1 << 32, n), rng.integers(0, 9, n), np.full(n, 0xFFFFFFFF),
                 np.where(half, 0xFFFFFFFF, rng.integers(0, 1 << 32, n)), np.arange(n)[::-1],
                 rng.integers(0, 1 << 12, n) << 20 | np.arange(n) % 3):
        keys = keys.astype(np.uint32)
        dk, di = ctx.to_device(keys), ctx.alloc(4 * n)
        try:
            ctx.sort(dk, di, n)
            want = np.argsort(keys, kind="stable")
            assert np.array_equal(di.read(np.int32, n), want)
            assert np.array_equal(dk.read(np.uint32, n), keys[want])
        finally:
            dk.destroy()
            di.destroy()


@pytest.mark.parametrize("bounds", ["gpu", "caller"])
@pytest.mark.parametrize("n", SIZES)
def test_build(ctx, lb, ora, n, bounds):
    for tri in (lb.wl_uniform(n, n, 0.01), lb.wl_heightfield(n, 150, (n + 299) // 300)[:n]):
        b = lb.wl_bounds(tri) if bounds == "caller" else None
        bvh, otri, sk, pm = ctx.build_arrays(tri, b, keep_topology=True)
        wb, wo, wsk, wpm = ora.build(tri, b, 0)
        assert np.array_equal(sk, wsk) and np.array_equal(pm, wpm)
        assert np.array_equal(bvh, wb)
        assert np.array_equal(otri.view(np.uint32), wo.view(np.uint32))
        assert np.array_equal(ctx.build_arrays(tri, b)[0], wb)  # keys in scratch


# where the tile grows: one tile of 512, 1,024 or 2,048 keys, then several
@pytest.mark.parametrize("n", [511, 512, 513, 1023, 1024, 1025, 1537, 3000, 4096, 4097, 8192, 8193, 16383, 32768])
def test_small_tiles(ctx, lb, ora, n):
    test_sort(ctx, n)
    for bounds in ("gpu", "caller"):
        test_build(ctx, lb, ora, n, bounds)


# two rounds of 16: one tile past 8 and 16 groups, the largest build, the first
# that takes radix passes
@pytest.mark.parametrize("n", [65537, 262145, 300001, 393215, 393216, 393217])
def test_two_rounds(ctx, lb, ora, n):
    for bounds in ("gpu", "caller"):
        test_build(ctx, lb, ora, n, bounds)
