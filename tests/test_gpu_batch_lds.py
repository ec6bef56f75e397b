"""Small-graph batches solved in LDS: graphs around the most vertices one
workgroup holds (32768) and a cluster (16 of them), clusters of several sizes,
more clusters than workgroups (each workgroup then takes several in turn),
hubs, and graphs whose weights keep them out of LDS in the same batch.  Whole
numbers: exact against the oracle, on every replay."""
import numpy as np
import pytest

import orc
import smdp
from conftest import random_graph

pytestmark = pytest.mark.gpu

FIT = 32768


def _graph(n, m, seed, wlo=1, whi=100):
    row, col, w = random_graph(n, m, seed, wlo, whi)
    return smdp.HostGraph(row, col, w, 0)


def _check(ctx, graphs, srcs=None, replays=2):
    srcs = np.zeros(len(graphs), np.int32) if srcs is None else np.asarray(srcs, np.int32)
    refs = [orc.dijkstra(g.row, g.col, g.w, int(s)) for g, s in zip(graphs, srcs)]
    with smdp.Batch(ctx, graphs, srcs) as b:
        for rep in range(replays):
            st = b.run()
            for i, ref in enumerate(refs):
                assert np.array_equal(b.read(i), ref), (rep, i, graphs[i].n, graphs[i].m)
    return st


@pytest.fixture
def share(ctx):
    old = ctx.get_params(smdp.APP_MSSSP)
    yield lambda v: ctx.set_params(smdp.APP_MSSSP, group_share=v)
    ctx.set_params(smdp.APP_MSSSP, **old.as_dict())


@pytest.mark.parametrize("pct", [10, 100, 1000])
def test_sizes_around_one_workgroup(ctx, share, pct):
    share(pct)
    graphs = [_graph(n, 4 * n, n) for n in (1, 63, 257, FIT - 1, FIT, FIT + 1, FIT + 64, 2 * FIT, 2 * FIT + 1, 100003)]
    print(f"batch lds share={pct}", flush=True)
    _check(ctx, graphs, [g.n // 3 for g in graphs])


@pytest.mark.parametrize("n", [16 * FIT - 1, 16 * FIT, 16 * FIT + 1])  # the last is solved in memory
def test_largest_cluster(ctx, n):
    print(f"batch cluster n={n}", flush=True)
    _check(ctx, [_graph(n, 2 * n, 3), _graph(500, 2000, 4)])


def test_many_arcs_and_hubs_in_a_cluster(ctx):
    r = np.random.RandomState(5)
    n = 40000
    deg = np.full(n, 8, np.int64)
    deg[[0, 1, 25000, n - 1]] = [300000, 70000, 200000, 600]
    row = np.concatenate([[0], np.cumsum(deg)])
    hubs = smdp.HostGraph(row, r.randint(0, n, row[-1]), r.randint(0, 40, row[-1]), 0)
    dense = _graph(20000, (1 << 20) + 77, 6)  # one workgroup holds its vertices, a cluster shares its arcs
    _check(ctx, [hubs, dense] + [_graph(300, 900, i) for i in range(5)], [1, 0] + [0] * 5)


def test_more_clusters_than_workgroups(ctx):
    graphs = [smdp.gen_small_graph(i, vlo=FIT + 1 + i, vhi=FIT + 1 + i, dlo=1.5, dhi=1.5, seed=8) for i in range(300)]
    print("batch: 300 clusters", flush=True)
    _check(ctx, graphs)


def test_weights_out_of_range_beside_lds_graphs(ctx):
    """Negative weights without a cycle and weights of 2^30 or more are solved
    in memory, as a group and by one workgroup; the rest of the batch in LDS."""
    n = 3000
    dag = np.sort(np.random.RandomState(7).randint(0, n - 1, 9000))
    col = dag + 1 + np.random.RandomState(8).randint(0, n, 9000) % (n - 1 - dag)
    row = np.concatenate([[0], np.cumsum(np.bincount(dag, minlength=n))])
    w = np.random.RandomState(9).randint(-20, 50, 9000)
    neg = smdp.HostGraph(row, col, w, 0)
    want = np.full(n, orc.INF, np.int64)
    want[0] = 0
    for u in range(n):  # vertices in topological order
        if want[u] < orc.INF:
            for e in range(row[u], row[u + 1]):
                want[col[e]] = min(want[col[e]], want[u] + w[e])
    big = _graph(200, 1000, 3, 1, 9)
    big.w[500] = 2 ** 30
    rest = [_graph(400, 1600, i) for i in range(4)] + [_graph(FIT + 5, 50000, 2)]
    graphs = [neg, big] + rest
    outs, _ = ctx.sssp_multi_graph(graphs, np.zeros(len(graphs), np.int32))
    assert np.array_equal(outs[0], want)
    for g, d in list(zip(graphs, outs))[1:]:
        assert np.array_equal(d, orc.dijkstra(g.row, g.col, g.w, 0))
