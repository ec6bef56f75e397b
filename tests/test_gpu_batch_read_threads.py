"""Several threads reading the results of one batch at the same time: in order
(which reads ahead), backwards, and at random, each into buffers of its own."""
import threading

import numpy as np
import pytest

import orc
import smdp
from conftest import random_graph

pytestmark = pytest.mark.gpu


def test_threads_read_one_batch(ctx):
    graphs = []
    for i in range(200):
        row, col, w = random_graph(20 + 37 * (i % 11) + 400 * (i % 3), 900, i, 1, 30)
        graphs.append(smdp.HostGraph(row, col, w, 0))
    refs = [orc.dijkstra(g.row, g.col, g.w, 0) for g in graphs]
    errors = []
    with smdp.Batch(ctx, graphs, np.zeros(len(graphs), np.int32)) as b:
        def body(orders):
            try:
                for order in orders:
                    for i in order:
                        assert np.array_equal(b.read(int(i)), refs[i]), i
            except BaseException as e:  # noqa: BLE001 (reported below)
                errors.append(e)

        r = np.random.RandomState(2)
        k = len(graphs)
        orders = [[range(k)] * 8, [range(k // 2, k), range(k // 2)] * 8, [range(k - 1, -1, -1)] * 8,
                  [r.randint(0, k, 400) for _ in range(4)]]
        for _ in range(3):
            b.run()
            threads = [threading.Thread(target=body, args=(o,)) for o in orders]
            for t in threads:
                t.start()
            for t in threads:
                t.join(100)
            assert not errors, errors[0]
