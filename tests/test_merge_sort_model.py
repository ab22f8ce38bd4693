"""CPU restatement of the merge sort of small meshes (csrc/k_merge_sort.hip):
the merge rounds inside a tile, the runs per round, the sample search and the
windowed rank search of k_merge, each read checked to lie inside its run.
Tiles of 128 keys and samples of 2 stand for the kernel's 2,048 and 32 (64
samples a tile), so that a few thousand keys take several rounds."""
import numpy as np
import pytest

TILE_LOG = 7
TILE = 1 << TILE_LOG
SAMPLE_LOG, WINDOW, STEPS = 1, 12, 4
SAMPLE = 1 << SAMPLE_LOG


def tile_sort(keys, full):
    """One tile: runs of two, then merge rounds by ranks in the sibling."""
    past = 0xFFFFFFFF if full else 0x7FFFFFFF
    k = np.full(TILE, past, np.int64)
    k[:len(keys)] = keys
    idx = np.arange(TILE)
    swap = k[1::2] < k[0::2]
    order = np.arange(TILE).reshape(-1, 2)
    order[swap] = order[swap][:, ::-1]
    k, idx = k[order.ravel()], idx[order.ravel()]
    length = 2
    while length < TILE:
        p = np.arange(TILE)
        sib = (p ^ length) & ~(length - 1)
        second = (p & length) != 0
        pos = sib.copy()
        below = lambda v: np.where(second, v <= k, v < k)  # noqa: E731
        h = length // 2
        while h:
            assert np.all((pos + h - 1 >= sib) & (pos + h - 1 < sib + length))
            pos = np.where(below(k[pos + h - 1]), pos + h, pos)
            h //= 2
        assert np.all((pos >= sib) & (pos < sib + length))
        pos = pos + below(k[pos])
        to = (p & ~(2 * length - 1)) + (p & (length - 1)) + pos - sib
        assert np.array_equal(np.sort(to), p)
        k2, i2 = np.empty_like(k), np.empty_like(idx)
        k2[to], i2[to] = k, idx
        k, idx = k2, i2
        length *= 2
    assert np.all(idx[:len(keys)] < len(keys))  # the padding stays behind
    return k[:len(keys)], idx[:len(keys)]


def merge_plan(n):
    """(run_log, log2 of the runs merged together) of each round."""
    runs, rounds, log = -(-n // TILE), [], TILE_LOG
    while runs > 1:
        g = 4
        if runs <= (16 if rounds else 32):
            g = 3
            while 1 << g < runs:
                g += 1
        rounds.append((log, g))
        runs = -(-runs // (1 << g))
        log += g
    return rounds


def chunk_positions(keys, n, c0, run_log, group_log):
    """Where the 64 keys at c0 go, and the widest window searched."""
    smp, lane = keys[SAMPLE - 1::SAMPLE], np.arange(64)
    if not len(smp):
        smp = np.full(1, -5)
    key = keys[np.minimum(c0 + lane, n - 1)]
    run = c0 >> run_log
    runs = 1 << group_log
    g0 = run & ~(runs - 1)
    x, have = max(run_log - TILE_LOG, 0), n >> SAMPLE_LOG  # a short run has fewer samples
    assert x <= 6
    rank, widest, rng = np.zeros(64, np.int64), 0, np.random.default_rng(c0)
    for s in range(g0, g0 + runs):
        b = s << run_log
        length = 0 if s == run or b >= n else min(1 << run_log, n - b)
        le = s < run
        ns = length >> SAMPLE_LOG

        def count(at, k, c, le=le):
            v = smp[np.where(at < have, at, 0)]
            return int(np.sum(((v <= k) if le else (v < k)) & (lane < c)))

        ends = []
        for k in (key[0], key[63]):
            c = count((b >> SAMPLE_LOG) + ((lane + 1) << x) - 1, k, ns >> x) << x
            if x:
                c += count((b >> SAMPLE_LOG) + c + lane, k, min(ns - c, (1 << x) - 1))
            ends.append(c)
        lo = ends[0] << SAMPLE_LOG
        m = min((ends[1] << SAMPLE_LOG) + SAMPLE - 1, length) - lo
        assert 0 <= m <= length - lo
        widest = max(widest, m)
        w = keys[b + lo:b + lo + m] if m else keys[:1]
        below = (lambda y: y <= key) if le else (lambda y: y < key)
        pos = np.zeros(64, np.int64)
        if m < WINDOW:
            win = np.full(1 << STEPS, key.max() + 1)  # anything past the window
            win[WINDOW:] = rng.integers(0, key.max() + 2, (1 << STEPS) - WINDOW)
            win[:WINDOW] = w[np.minimum(np.arange(WINDOW), max(m, 1) - 1)]
            h = 1 << (STEPS - 1)
            while h:
                pos = np.where(below(win[pos + h - 1]), pos + h, pos)
                h //= 2
            pos = np.minimum(pos, m)
        else:
            # every lane on its own: samples 2^x apart, those between, keys
            def halve(p, left, read, steps):
                left = np.broadcast_to(left, 64).copy()
                for _ in range(steps):
                    h = (left + 1) >> 1
                    p = p + np.where((h > 0) & below(read(np.where(h > 0, p + h - 1, 0))), h, 0)
                    left >>= 1
                assert not left.any()
                return p

            coarse = smp[np.minimum((b >> SAMPLE_LOG) + ((lane + 1) << x) - 1, have - 1)]
            p = halve(np.zeros(64, np.int64), ns >> x, lambda q: coarse[q], 7) << x
            p = halve(p, np.minimum((1 << x) - 1, ns - p), lambda q: smp[(b >> SAMPLE_LOG) + q], x)
            p <<= SAMPLE_LOG
            assert np.all(p <= length)
            p = halve(p, np.minimum(SAMPLE - 1, length - p), lambda q: keys[np.minimum(b + q, n - 1)], SAMPLE_LOG)
            pos = p - lo
        rank += lo + pos
    i = np.arange(c0, min(c0 + 64, n))
    return i, (g0 << run_log) + (i - (run << run_log)) + rank[:len(i)], widest


def merge_sort(keys, full):
    n = len(keys)
    k, idx = np.empty(n, np.int64), np.empty(n, np.int64)
    for b in range(0, n, TILE):
        kk, ii = tile_sort(keys[b:b + TILE], full)
        k[b:b + TILE], idx[b:b + TILE] = kk, ii + b
    for run_log, g in merge_plan(n):
        k2, i2 = np.full(n, -1, np.int64), np.full(n, -1, np.int64)
        for c0 in range(0, n, 64):
            i, to, _ = chunk_positions(k, n, c0, run_log, g)
            assert np.all(to < n) and np.all(i2[to] == -1)
            k2[to], i2[to] = k[i], idx[i]
        k, idx = k2, i2
    return k, idx


@pytest.mark.parametrize("full", [False, True])
@pytest.mark.parametrize("n", [1, 2, 63, 64, 127, 128, 129, 1000, 1024, 1025, 2049, 4095, 4097, 8192, 8193, 9001])
def test_merge_sort_is_the_stable_sort(n, full):
    rng = np.random.default_rng(n)
    top = 0xFFFFFFFF if full else (1 << 30) - 1
    kinds = [rng.integers(0, top + 1, n), rng.integers(0, 5, n), np.full(n, top), np.arange(n),
             np.arange(n)[::-1], np.where(np.arange(n) % 3 == 0, top, rng.integers(0, 9, n)),
             np.sort(rng.integers(0, n // 2 + 1, n))]
    for keys in kinds:
        keys = np.asarray(keys, np.int64)
        k, idx = merge_sort(keys, full)
        want = np.argsort(keys, kind="stable")
        assert np.array_equal(idx, want)
        assert np.array_equal(k, keys[want])


@pytest.mark.parametrize("run_log", [6, 7, 10, 13])
def test_uneven_runs_take_every_search(run_log):
    """One and two readings of the samples, narrow and wide windows."""
    rng = np.random.default_rng(7)
    L = 1 << run_log
    n = 5 * L + 77
    keys = rng.integers(0, 1 << 12, n)
    keys[L:2 * L] = 1000  # a run inside one key
    keys[2 * L:3 * L:2] = 0  # chunks of it span the others
    for b in range(0, n, L):
        keys[b:b + L].sort()
    inv = np.empty(n, np.int64)
    inv[np.argsort(keys, kind="stable")] = np.arange(n)
    widths = []
    for c0 in range(0, n, 64 if run_log < 13 else 64 * 13):
        i, to, widest = chunk_positions(keys, n, c0, run_log, 3)
        assert np.array_equal(to, inv[i])
        widths.append(widest)
    assert max(widths) >= WINDOW
