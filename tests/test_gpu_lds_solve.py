"""SSSP and BFS of small graphs solved by one workgroup in LDS (the tuned
solution of graphs that fit): vertex counts around the scan blocks (256) and
the largest that fits, rows around the heavy and chunk sizes, hubs beyond a
round's chunk list, zero, large and negative weights (which go back to the
rounds), and each entry point.  Whole numbers: exact against the oracle."""
import numpy as np
import pytest

import orc
import smdp
from conftest import random_graph
from test_zz_no_alloc import DeviceArrays, noalloc_sssp

pytestmark = pytest.mark.gpu

FIT = 32768  # vertices one workgroup holds


def _hubs(n, degs, seed, whi=50):
    """Vertex i has degs[i] random arcs, the others two."""
    r = np.random.RandomState(seed)
    deg = np.full(n, 2, np.int64)
    deg[:len(degs)] = degs
    row = np.concatenate([[0], np.cumsum(deg)])
    return smdp.HostGraph(row, r.randint(0, n, row[-1]), r.randint(1, whi + 1, row[-1]), 0)


def _check(ctx, g, src=None):
    src = g.source if src is None else src
    ref = orc.dijkstra(g.row, g.col, g.w, src)
    d, st = ctx.sssp(g, src, smdp.SOL_TUNED)
    assert np.array_equal(d, ref)
    assert st.m_reached == int(np.diff(g.row)[ref != orc.INF].sum()) and st.rounds >= 1
    lv, _ = ctx.bfs(g, src, smdp.SOL_TUNED)
    assert np.array_equal(lv, orc.bfs(g.row, g.col, src))
    return st


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 255, 256, 257, 4095, 4096, 4097, FIT - 1, FIT, FIT + 1])
def test_vertex_counts(ctx, n):
    row, col, w = random_graph(n, 5 * n, n, 1, 60)
    g = smdp.HostGraph(row, col, w, 0)
    print(f"lds n={n}", flush=True)
    for src in {0, n // 2, n - 1}:
        st = _check(ctx, g, src)
    assert (st.kernel_launches == 1) == (n <= FIT)


@pytest.mark.parametrize("degs", [[255, 256, 257], [255, 511, 512, 513, 2047, 2048, 2049], [300] * 700, [140000, 3],
                                  [1000, 0, 0, 90000, 90000]])
def test_heavy_rows(ctx, degs):
    print(f"lds degs={degs[:5]}", flush=True)
    _check(ctx, _hubs(3000, degs, 11))


def test_long_path_and_grid(ctx):
    n = 5000  # one vertex a round
    path = smdp.HostGraph(np.minimum(np.arange(n + 1), n - 1), np.arange(1, n), np.arange(1, n) % 7 + 1, 0)
    _check(ctx, path)


@pytest.mark.parametrize("wlo,whi", [(0, 0), (0, 3), (1, 1), (1, 200000), (2 ** 20, 2 ** 27)])
def test_weights_in_range(ctx, wlo, whi):
    row, col, w = random_graph(3000, 20000, 5, wlo, whi)
    g = smdp.HostGraph(row, col, w, 7)
    d, st = ctx.sssp(g, 7, smdp.SOL_TUNED)
    assert np.array_equal(d, orc.dijkstra(row, col, w, 7)) and st.kernel_launches == 1


def test_candidates_at_and_beyond_the_sentinel(ctx):
    """Distances just below 2^30 hold, candidates at or above it do not count."""
    big = 2 ** 30 - 1
    row = [0, 3, 4, 5, 5, 5, 5]
    g = smdp.HostGraph(row, [1, 2, 3, 4, 5], [big - 5, 4, big, 4, big - 3], 0)
    d, _ = ctx.sssp(g, 0, smdp.SOL_TUNED)
    assert d.tolist() == [0, big - 5, 4, big, big - 1, orc.INF]


def test_weights_out_of_range_go_back_to_the_rounds(ctx):
    """A weight of 2^30 or more, or a negative one without a cycle."""
    for w, ref in (([5, 2 ** 30, 9, 2, 7, 2 ** 30], [0, 5, 7, 9, 14]),
                   ([50, 60, 9, -20, 7, 1], [0, 50, 30, 9, 10])):
        g = smdp.HostGraph([0, 3, 4, 5, 6, 6], [1, 2, 3, 2, 4, 4], w, 0)
        d, st = ctx.sssp(g, 0, smdp.SOL_TUNED)
        assert d.tolist() == ref and st.kernel_launches > 1


def test_resident_and_device_entry_points(ctx):
    g = smdp.gen_rmat(13, 16, wlo=1, whi=255, seed=4)
    srcs = smdp.gen_sources(g, 3, 2)
    with smdp.Graph(ctx, g) as dg:
        for s in srcs:
            dg.sssp(int(s), smdp.SOL_TUNED)
            assert np.array_equal(dg.read(smdp.RES_DIST), orc.dijkstra(g.row, g.col, g.w, int(s)))
            dg.bfs(int(s), smdp.SOL_TUNED)
            assert np.array_equal(dg.read(smdp.RES_LEVEL), orc.bfs(g.row, g.col, int(s)))
    d = DeviceArrays(g)
    try:
        rc, st = noalloc_sssp(ctx, d, int(srcs[0]), smdp.SOL_TUNED)
        assert rc == smdp.OK and np.array_equal(d.read_dist(), orc.dijkstra(g.row, g.col, g.w, int(srcs[0])))
    finally:
        d.close()
