"""The sort tiles of a batch by its largest mesh: 1,024 keys up to the line that its
size in all, its digits and its number of meshes give (batch_small_mesh of
csrc/lbvh_internal.h), 4,096 beyond, where one block's scan of a mesh's small tiles
would be the longer chain.  The tiles show in the scratch that the
context holds, beside one under a budget, which always takes the large ones."""
import numpy as np
import pytest

from test_gpu_batched import make_batch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("past", [False, True], ids=["at the line", "past it"])
@pytest.mark.parametrize("bits,most,rest", [
    (8, 3 << 16, []), (8, 3 << 16, [2000] * 40), (8, 65536, [7, 0, 1025] * 100), (8, 65536, [2000] * 200),
    (8, 32768, [3000] * 400), (10, 5 << 12, []), (10, 5 << 12, [20000] * 4), (10, 16384, [7, 0, 1025] * 100),
    (10, 4096, [3000] * 400)])
def test_tiles_follow_the_largest_mesh(lb, ora, bits, most, rest, past):
    meshes, offsets, tri = make_batch(lb, rest[:3] + [most + past] + rest[3:], 70)
    total = int(offsets[-1])
    held, outs = [], []
    for budget in (0, 8 << 30):
        with lb.Context(0, hbm_budget=budget) as c:
            c.set_tuning(lb.TUNE_SORT_BITS, bits)
            c.set_tuning(lb.TUNE_TREE_TILE, 1024)  # the same tree either way
            d, bvh, otri = c.to_device(tri), c.alloc(64 * total), c.alloc(48 * total)
            c.build_batched(d, offsets, None, bvh, otri)
            outs.append((bvh.read(np.uint8, 64 * total), otri.read(np.uint32, 12 * total)))
            held.append(c.bytes_in_use())
    assert (held[0] == held[1]) == past, held
    for a, b in zip(*outs):
        assert np.array_equal(a, b)
    for k in (0, min(3, len(meshes) - 1), len(meshes) - 1):
        a, b = int(offsets[k]), int(offsets[k + 1])
        wb, wo = ora.build(meshes[k], None, 0)[:2]
        assert np.array_equal(outs[0][0][64 * a:64 * b], wb), k
        assert np.array_equal(outs[0][1][12 * a:12 * b], wo.view(np.uint32).ravel()), k


@pytest.mark.parametrize("bits", [8, 10])
@pytest.mark.parametrize("budget", [0, 1 << 30], ids=["small tiles", "large tiles"])
def test_part_tiles(lb, ora, budget, bits):
    """Meshes that end at, before and past a row of a tile (256 keys), the last
    row's end and the tile's."""
    sizes = [255, 256, 257, 511, 512, 513, 767, 768, 769, 3839, 3840, 3841, 4095, 4096, 4097, 1]
    meshes, offsets, tri = make_batch(lb, sizes, 120)
    total = int(offsets[-1])
    with lb.Context(0, hbm_budget=budget) as c:
        c.set_tuning(lb.TUNE_SORT_BITS, bits)
        d, bvh, otri = c.to_device(tri), c.alloc(64 * total), c.alloc(48 * total)
        c.build_batched(d, offsets, None, bvh, otri)
        got, gtri = bvh.read(np.uint8, 64 * total), otri.read(np.uint32, 12 * total)
    for k, m in enumerate(meshes):
        a, b = int(offsets[k]), int(offsets[k + 1])
        wb, wo = ora.build(m, None, 0)[:2]
        assert np.array_equal(got[64 * a:64 * b], wb), k
        assert np.array_equal(gtri[12 * a:12 * b], wo.view(np.uint32).ravel()), k
