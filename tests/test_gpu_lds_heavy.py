"""Vertices with many arcs in LDS solves: rounds with more chunks of them than
a round's list holds (512 of 256 arcs), chunk lengths around their limits, and
hubs of clusters.  Whole numbers: exact against the oracle."""
import numpy as np
import pytest

import orc
import smdp

pytestmark = pytest.mark.gpu


def _complete(n, lo, hi, seed=1):
    w = np.random.RandomState(seed).randint(lo, hi + 1, n * n)
    return smdp.HostGraph(np.arange(n + 1) * n, np.tile(np.arange(n), n), w, n // 2)


def _hubs(n, degs, seed, whi=50):
    """The first vertices have degs random arcs each, the others two."""
    r = np.random.RandomState(seed)
    deg = np.full(n, 2, np.int64)
    deg[:len(degs)] = degs
    row = np.concatenate([[0], np.cumsum(deg)])
    return smdp.HostGraph(row, r.randint(0, n, row[-1]), r.randint(1, whi + 1, row[-1]), 0)


def _check(ctx, g):
    ref = orc.dijkstra(g.row, g.col, g.w, g.source)
    d, st = ctx.sssp(g, g.source, smdp.SOL_TUNED)
    assert np.array_equal(d, ref)
    assert st.kernel_launches == 1 and st.m_reached == int(np.diff(g.row)[ref != orc.INF].sum())
    lv, _ = ctx.bfs(g, g.source, smdp.SOL_TUNED)
    assert np.array_equal(lv, orc.bfs(g.row, g.col, g.source))


@pytest.mark.parametrize("n", [63, 65, 200, 256, 257, 440, 513, 600, 627])
@pytest.mark.parametrize("lo,hi", [(0, 0), (1, 1), (1, 100), (1, 2 ** 20)])
def test_complete_graphs(ctx, n, lo, hi):
    print(f"complete {n} weights {lo}..{hi}", flush=True)
    _check(ctx, _complete(n, lo, hi))


@pytest.mark.parametrize("degs", [[256 * 512], [256 * 512 + 1], [256 * 128, 256 * 128 + 1, 256 * 129], [90000] * 4,
                                  [256] * 1400, [257] * 700, [300000]])
def test_chunk_lengths(ctx, degs):
    print(f"chunks {degs[:4]} x {len(degs)}", flush=True)
    _check(ctx, _hubs(3000, degs, 3))


@pytest.mark.parametrize("n,degs", [(500000, [500000]), (70000, [4000000, 1000000, 3]), (40000, [300] * 3000),
                                    (33000, [15000000])])
def test_hubs_of_clusters(ctx, n, degs):
    print(f"cluster n={n} hubs {degs[:3]}", flush=True)
    g = _hubs(n, degs, 4)
    small = _hubs(600, [300] * 600, 5)
    with smdp.Batch(ctx, [g, small], np.zeros(2, np.int32)) as b:
        for _ in range(2):
            b.run()
            for i, h in enumerate((g, small)):
                assert np.array_equal(b.read(i), orc.dijkstra(h.row, h.col, h.w, 0))
