"""Pair plans by a table of all pairs and by sorting the list's own: the same
plan (host only).  A list takes the table while it is no larger than a sort; the
same list among more shells than it names takes the sort."""
import numpy as np
import pytest

from bskit_amd import _lib as L
from bskit_amd.engine import PairPlan

pytestmark = pytest.mark.skipif(not L.built(), reason='libbskhip.so not built')


def plan(tri, nshell, mode, levels, **kw):
    p = PairPlan(tri, nshell, mode, upload=False, levels=levels, **kw)
    return p, p.tables(), p.slots()


@pytest.mark.parametrize('mode,f64,levels', [(0, False, False), (0, False, True), (0, True, False),
                                             (0, True, True), (1, False, True), (1, True, False),
                                             (2, True, True), (2, False, False)])
def test_table_and_sort(mode, f64, levels):
    rng = np.random.default_rng(10 * mode + f64)
    few = rng.integers(0, 8, (300, 3), dtype=np.int32)  # 64 pairs: table
    lv = rng.integers(0, 4, 301) if levels else None
    # one more triangle with a shell so far up that the table would be larger than
    # the sort: 80^2 > 4 * 301 + 4096 for the roles' lists
    top = 80
    many = np.concatenate([few, [[top, top, top]]]).astype(np.int32)
    a, ta, sa = plan(few, top + 1, mode, None if lv is None else lv[:300], f64=f64)
    b, tb, sb = plan(many, top + 1, mode, lv, f64=f64)
    # both find every triangle's pair and third side in the item of its slot
    for p, (items, outpos, pairs), slots, tri in ((a, ta, sa, few), (b, tb, sb, many)):
        prow = pairs.reshape(-1, 16)
        item = {}
        e0 = 0
        for g, (_, lo, _, npass, ni, rep) in enumerate(p.segments):
            for e in range(e0, e0 + 8 * npass * ni):
                if outpos[e] >= 0:
                    item[(g, outpos[e])] = (items[e] & 0xffff, (items[e] >> 16 & 0xff) + lo // 16)
            e0 += 8 * npass * ni
        for t, (i, j, k) in enumerate(tri):
            for g, s in enumerate(slots[t]):
                if s < 0:
                    continue
                s = int(s) & 0x0fffffff
                tile, kb = item[(g, s // 256)]
                w = int(prow[tile][s // 16 % 16])
                x, y, z = w & 0xffff, w >> 16 & 0xffff, 16 * kb + s % 16
                want = (i, j, k)
                if mode == 0:
                    assert sorted((x, y, z)) == sorted(want)
                elif mode == 1:
                    assert (max(x, y), min(x, y), z) == (max(i, j), min(i, j), k)
                else:
                    assert (x, y, z) == want


def test_grid_info_plan():
    """Grid info's four sums, with repeated sides, few and many shells."""
    rng = np.random.default_rng(3)
    for nb, ntri in ((6, 200), (70, 200), (136, 90)):
        tri = rng.integers(0, nb, (ntri, 3), dtype=np.int32)
        tri[::5, 1] = tri[::5, 0]
        p = PairPlan(tri, nb, L.MODE_AUTO, upload=False, gridinfo=True)
        items, outpos, pairs = p.tables()
        prow = pairs.reshape(-1, 16)
        lo = p.segments[0][1]
        item = {o: (i & 0xffff, (i >> 16 & 0xff) + lo // 16) for i, o in zip(items, outpos) if o >= 0}
        p.ntri = 4 * ntri
        slots = p.slots()
        for t in range(4 * ntri):
            s = int(slots[t, 0]) & 0x0fffffff
            tile, kb = item[s // 256]
            w = int(prow[tile][s // 16 % 16])
            got = sorted((w & 0xffff, w >> 16 & 0xffff, 16 * kb + s % 16))
            want = [int(v) for v in tri[t // 4]]
            if t % 4:
                want[t % 4 - 1] += nb
            assert got == sorted(want)
