"""SSSP and BFS rounds in one launch where many arcs of a round lead to few
vertices: one, several, more than a wave looks at, and more than a workgroup
remembers, with candidates in rising, falling and random order.  Exact against
the oracle, for drop-in, resident and repeated solves."""
import numpy as np
import pytest

import orc
import smdp

pytestmark = pytest.mark.gpu


def _csr(n, src, dst, w):
    order = np.argsort(src, kind="stable")
    row = np.concatenate([[0], np.cumsum(np.bincount(src, minlength=n))])
    return smdp.HostGraph(row, dst[order], w[order], 0)


def _fan(mid, sinks, order, seed=1):
    """0 -> mid vertices -> sinks -> back into the middle."""
    r = np.random.RandomState(seed)
    n = 1 + mid + sinks
    v = np.arange(1, mid + 1)
    s = 1 + mid + np.arange(sinks)
    w1 = {"rising": 1 + np.arange(mid) // 3, "falling": 1 + (mid - np.arange(mid)) // 3,
          "equal": np.full(mid, 5), "random": r.randint(1, 1000, mid)}[order]
    src = np.concatenate([np.zeros(mid, int), v, v, s])
    dst = np.concatenate([v, 1 + mid + r.randint(0, sinks, mid), 1 + mid + (v * 7) % sinks, 1 + r.randint(0, mid, sinks)])
    w = np.concatenate([w1, r.randint(1, 9, 2 * mid), np.ones(sinks, int)])
    return _csr(n, src, dst, w)


@pytest.mark.parametrize("sinks", [1, 2, 15, 16, 17, 64, 3000, 40000])
@pytest.mark.parametrize("order", ["rising", "falling", "equal", "random"])
def test_fans(ctx, sinks, order):
    g = _fan(60000, sinks, order)
    print(f"fan into {sinks}, {order}", flush=True)
    ref, lv = orc.dijkstra(g.row, g.col, g.w, 0), orc.bfs(g.row, g.col, 0)
    d, st = ctx.sssp(g, 0, smdp.SOL_TUNED)
    assert np.array_equal(d, ref) and st.kernel_launches == 2
    with smdp.Graph(ctx, g) as dg:
        for _ in range(2):
            dg.sssp(0, smdp.SOL_TUNED)
            assert np.array_equal(dg.read(smdp.RES_DIST), ref)
            dg.bfs(0, smdp.SOL_TUNED)
            assert np.array_equal(dg.read(smdp.RES_LEVEL), lv)


def test_negative_candidates(ctx):
    """Distances below zero, and targets lowered in many rounds."""
    r = np.random.RandomState(2)
    n, m = 40000, 300000
    a = r.randint(0, 200, m)
    layer = r.randint(0, 199, m)
    src = np.where(r.rand(m) < 0.5, layer, layer * 200 + a)  # layers of 200 vertices, hubs among the first
    dst = np.minimum((src // 200 + 1) * 200 + r.randint(0, 3, m), n - 1)
    keep = dst > src
    g = _csr(n, np.concatenate([[0] * 200, src[keep]]), np.concatenate([np.arange(200) + 1, dst[keep]]),
             np.concatenate([np.arange(200) % 11, r.randint(-40, 60, keep.sum())]))
    ref = orc.bellman_ford(g.row, g.col, g.w, 0)
    assert ref.min() < 0
    d, _ = ctx.sssp(g, 0, smdp.SOL_TUNED)
    assert np.array_equal(d, ref)
