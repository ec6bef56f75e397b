"""Batches whose graphs share teams of workgroups: clusters that follow one
another on a team while other teams take seconds, and solves in memory on
teams that also run clusters.  Whole numbers: exact on every replay."""
import numpy as np
import pytest

import orc
import smdp
from conftest import random_graph

pytestmark = pytest.mark.gpu


def _path(n):
    v = np.arange(n - 1, dtype=np.int32)
    return smdp.HostGraph(np.minimum(np.arange(n + 1), n - 1).astype(np.int32), v + 1, 1 + v % 5, 0)


def test_long_paths_wait_only_for_their_own_rounds(ctx):
    """20 clusters of 15 or 16 workgroups on 256, each a vertex a round: a
    barrier that also waited for another path's solve would give up."""
    graphs = [_path(490000 - 137 * i) for i in range(20)]
    print("batch: 20 long paths", flush=True)
    with smdp.Batch(ctx, graphs, np.zeros(len(graphs), np.int32)) as b:
        b.run()
        for i, g in enumerate(graphs):
            assert np.array_equal(b.read(i), np.concatenate([[0], np.cumsum(g.w)]))


def test_solves_in_memory_between_clusters(ctx):
    """Graphs with a negative weight are solved in memory; with more graphs for
    teams than workgroups, some by teams whose other graphs are clusters."""
    graphs, refs = [], []
    for i in range(90):
        n = 70000 + 100 * i
        row, col, w = random_graph(n, 4 * n, i, 1, 30)
        if i % 4 == 0:  # the last arc of a vertex that no arc reaches: negative, and never relaxed
            u = int(np.flatnonzero((np.bincount(col, minlength=n) == 0) & (np.diff(row) > 0))[-1])
            w[row[u + 1] - 1] = -3
        graphs.append(smdp.HostGraph(row, col, w, 0))
        src = int(np.argmax(np.diff(row)))
        h = w.copy()
        h[h < 0] = 1
        refs.append((src, orc.dijkstra(row, col, h, src)))
    print("batch: memory solves between clusters", flush=True)
    with smdp.Batch(ctx, graphs, np.array([s for s, _ in refs], np.int32)) as b:
        for _ in range(2):
            b.run()
            for i, (_, ref) in enumerate(refs):
                assert np.array_equal(b.read(i), ref), i
