"""The tree levels of small meshes (csrc/k_forest.hip) restated on the CPU:
nearest smaller deltas from the waves' masks of gaps below each value, child
boxes from the waves' sparse tables of unions, the frontier ranked by the bits of its
first elements.  In place of the item levels' own method it must reproduce the
oracle's nodes byte for byte."""
import numpy as np
import pytest

import test_item_levels_model as base


TOP = 4  # the tables' highest level


def below_masks(deltas, m, W):
    """[wave][u]: bits of the wave's gaps whose delta is below u, by planes."""
    masks = []
    for w in range(W):
        lanes = range(64 * w, 64 * w + 64)
        ends = sum(1 << i for i, t in enumerate(lanes) if t < m and deltas[t] < 0)
        v = [deltas[t] if t < m and deltas[t] >= 0 else 63 for t in lanes]
        pl = [sum((v[i] >> b & 1) << i for i in range(64)) for b in range(6)]
        row = []
        for u in range(64):
            lt, eq = 0, (1 << 64) - 1
            for b in range(5, -1, -1):
                vb = (1 << 64) - 1 if u >> b & 1 else 0
                lt |= eq & vb & ~pl[b]
                eq &= ~(pl[b] ^ vb)
            row.append(lt | ends)
        masks.append(row)
    return masks


def forest_round(items, skeys, n, nodes, T=256, LOG=None):
    m = len(items)
    assert 0 < m <= T
    W = T // 64
    il, ir = [i[0] for i in items], [i[1] for i in items]
    dm = [items[0][4]] + [i[5] for i in items]
    d = dm[1:]
    own = [(np.asarray(i[2], np.float32), np.asarray(i[3], np.float32)) for i in items]
    union = lambda p, q: (np.minimum(p[0], q[0]), np.maximum(p[1], q[1]))  # noqa: E731
    none = (np.full(3, np.nan, np.float32),) * 2  # past the elements: poison
    tabs, wholes = [], []
    for w in range(W):
        tab = [[own[t] if t < m else none for t in range(64 * w, 64 * w + 64)]]
        for k in range(TOP):
            tab.append([union(tab[k][i], tab[k][i + (1 << k)]) for i in range(64 - (2 << k) + 1)])
        tabs.append(tab)
        whole = tab[TOP][0]
        for i in (16, 32, 48):
            whole = union(whole, tab[TOP][i])
        wholes.append(whole)

    def part(w, i, j):
        k = min(TOP, (j - i + 1).bit_length() - 1)
        # an IndexError is a read past the level
        r = union(tabs[w][k][i], tabs[w][k][j + 1 - (1 << k)])
        if j - i >= 2 << TOP:
            r = union(r, union(tabs[w][TOP][i + (1 << TOP)], tabs[w][TOP][j + 1 - (2 << TOP)]))
        return r

    def box(x, y):
        assert 0 <= x <= y < m
        wx, wy = x >> 6, y >> 6
        if wx == wy:
            return part(wx, x & 63, y & 63)
        r = union(part(wx, x & 63, 63), part(wy, 0, y & 63))
        for w in range(wx + 1, wy):
            r = union(r, wholes[w])
        assert not np.isnan(r[0]).any()
        return r

    masks = below_masks(d, m, W)
    span = {}
    for t in range(m - 1):
        w, lane = t >> 6, t & 63
        pl = pr = -1
        for q in range(W):
            lo = hi = masks[q][d[t]]
            if q == w:
                lo &= (1 << lane) - 1
                hi &= ~((2 << lane) - 1)
            if q <= w and lo:
                pl = q * 64 + lo.bit_length()
            if q >= w and hi and pr < 0:
                pr = q * 64 + (hi & -hi).bit_length()
        if pl < 0 and dm[0] < d[t]:
            pl = 0
        if pl >= 0:
            assert dm[pl] < d[t] and all(v >= d[t] for v in dm[pl + 1:t + 1])
        if pr >= 0:
            assert pr <= m and dm[pr] < d[t] and all(v >= d[t] for v in dm[t + 1:pr])
        if pl >= 0 and pr >= 0:
            span[t] = (pl, pr)
    roots = {}
    for t, (pl, pr) in span.items():
        x, y = pl, pr - 1
        (lmn, lmx), (rmn, rmx) = box(x, t), box(t + 1, y)
        lo, s, hi = il[x], ir[t], ir[y]
        whole = lo == 0 and hi == n - 1
        nd = np.zeros(16, np.int32)
        nd[0:3], nd[3] = lmn.view(np.int32), -(s + 1) if lo == s else s
        nd[4:7], nd[7] = lmx.view(np.int32), 2
        nd[8:11], nd[11] = rmn.view(np.int32), -(s + 2) if hi == s + 1 else s + 1
        nd[12:15] = rmx.view(np.int32)
        K = 0 if whole else (hi if dm[pr] > dm[pl] else lo)
        assert (nodes[K] == 0).all()
        nodes[K] = nd
        if not whole and (pr - 1 if dm[pr] > dm[pl] else pl - 1) not in span:
            assert x not in roots
            roots[x] = (lo, hi, np.minimum(lmn, rmn), np.maximum(lmx, rmx), dm[pl], dm[pr])
    for t in range(m):
        if il[t] == 0 and ir[t] == n - 1:
            continue
        if (t if dm[t + 1] > dm[t] else t - 1) not in span:
            assert t not in roots
            roots[t] = (il[t], ir[t], *own[t], dm[t], dm[t + 1])
    assert len(roots) <= base.FMAX
    return [roots[a] for a in sorted(roots)]


def run(monkeypatch, ora, tri, leaves, items):
    def level(elements, skeys, n, nodes, T=None, LOG=None):
        single = all(e[0] == e[1] for e in elements) and len(elements) <= leaves
        return forest_round(elements, skeys, n, nodes, leaves if single else items)
    monkeypatch.setattr(base, "item_level", level)
    return base.run(ora, tri, leaves, items)


CASES = {"uniform": lambda lb: lb.wl_uniform(6, 9000, 0.01),
         "clustered": lambda lb: lb.wl_clustered(5, 6000, 0.3),
         "all-equal": lambda lb: np.tile(lb.wl_uniform(9, 1, 0.01), (3000, 1)),
         "heightfield": lambda lb: lb.wl_heightfield(7, 32, 32)}
CASES.update({f"n{n}": (lambda lb, n=n: lb.wl_uniform(3, n, 0.01)) for n in (2, 3, 64, 65, 255, 256, 257, 513)})


@pytest.mark.parametrize("name", CASES)
def test_forest_levels_reproduce_oracle(monkeypatch, lb, ora, name):
    ok, n, levels = run(monkeypatch, ora, CASES[name](lb), 256, 512)
    assert ok, (name, n, levels)


def test_rounds_of_few_items(monkeypatch, lb, ora):
    """Leaf tiles of 64 and rounds of 256 items: most blocks take several."""
    ok, n, levels = run(monkeypatch, ora, lb.wl_uniform(12, 20000, 0.01), 64, 256)
    assert ok, (n, levels)
