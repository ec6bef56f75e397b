"""Reading a batch's results: in order, backwards, twice, with gaps, graphs
larger than a piece read ahead, and after another run (nothing read ahead of an
earlier run is returned)."""
import numpy as np
import pytest

import orc
import smdp
from conftest import random_graph

pytestmark = pytest.mark.gpu


def test_read_orders_and_new_runs(ctx):
    sizes = [40, 3000, 1, 33000, 700, 600000, 20, 20, 9000] + [500 + 7 * i for i in range(60)]
    graphs = []
    for i, n in enumerate(sizes):
        row, col, w = random_graph(n, 2 * n, i, 1, 30)
        graphs.append(smdp.HostGraph(row, col, w, 0))
    refs = [orc.dijkstra(g.row, g.col, g.w, 0) for g in graphs]
    r = np.random.RandomState(3)
    with smdp.Batch(ctx, graphs, np.zeros(len(graphs), np.int32)) as b:
        for order in (range(len(sizes)), reversed(range(len(sizes))), [0, 1, 2, 2, 1, 5, 6, 7, 6, 3, 4, 5],
                      r.randint(0, len(sizes), 80), list(range(3, len(sizes))) * 2):
            b.run()
            for i in order:
                assert np.array_equal(b.read(int(i)), refs[i]), i


def test_results_follow_the_last_run(ctx):
    """A batch whose plan changes between runs and reads still returns the last run's results."""
    graphs = [smdp.gen_small_graph(i, vlo=64, vhi=2000, seed=5) for i in range(20)]
    refs = [orc.dijkstra(g.row, g.col, g.w, 0) for g in graphs]
    old = ctx.get_params(smdp.APP_MSSSP)
    try:
        with smdp.Batch(ctx, graphs, np.zeros(20, np.int32)) as b:
            b.run()
            assert all(np.array_equal(b.read(i), refs[i]) for i in range(10))
            b.autotune()
            b.run()
            assert all(np.array_equal(b.read(i), refs[i]) for i in range(20))
    finally:
        ctx.set_params(smdp.APP_MSSSP, **old.as_dict())
