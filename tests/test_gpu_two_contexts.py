"""Two host threads, a context each, on one GPU: solves whose workgroups wait
for one another take turns (or go to the host-driven rounds), so none stalls at
a barrier, and results are exact."""
import threading
import time

import numpy as np
import pytest

import orc
import smdp

pytestmark = pytest.mark.gpu

STALL = 0.5  # seconds; a barrier that gives up has waited for about one


def _together(workers):
    errors, slowest = [], []

    def body(work):
        try:
            with smdp.Context(0) as c:
                slowest.append(work(c))
        except BaseException as e:  # noqa: BLE001 (reported by the caller)
            errors.append(e)

    threads = [threading.Thread(target=body, args=(w,)) for w in workers]
    for t in threads:
        t.start()
    for t in threads:
        t.join(100)
    assert not errors and len(slowest) == len(workers), errors
    assert max(slowest) < STALL, slowest


def _timed(run, check, times):
    run(), check()  # the first run also builds plans
    worst = 0.0
    for _ in range(times):
        t0 = time.perf_counter()
        run()
        worst = max(worst, time.perf_counter() - t0)
        check()
    return worst


def _equal(a, b):
    assert np.array_equal(a, b)


def test_rounds_in_one_launch_side_by_side():
    g = smdp.gen_rmat(16, 16, wlo=1, whi=255, seed=3)
    ref, lv = orc.dijkstra(g.row, g.col, g.w, g.source), orc.bfs(g.row, g.col, g.source)

    def sssp(c):
        with smdp.Graph(c, g) as dg:
            return _timed(lambda: dg.sssp(g.source, smdp.SOL_TUNED), lambda: _equal(dg.read(smdp.RES_DIST), ref), 150)

    def bfs(c):
        with smdp.Graph(c, g) as dg:
            return _timed(lambda: dg.bfs(g.source, smdp.SOL_TUNED), lambda: _equal(dg.read(smdp.RES_LEVEL), lv), 150)

    print("two contexts: sssp and bfs", flush=True)
    _together([sssp, sssp, bfs])


def test_colouring_batch_and_sources_side_by_side():
    g = smdp.gen_rmat(13, 8, wlo=1, whi=255, seed=4, symmetrize=True)
    colors, _ = orc.color_closed(g.row, g.col)
    srcs = smdp.gen_sources(g, 20, 3)
    refs = np.stack([orc.dijkstra(g.row, g.col, g.w, int(s)) for s in srcs])
    graphs = [smdp.gen_small_graph(i, vlo=40000, vhi=40000, dlo=8.0, dhi=8.0, seed=6) for i in range(30)]
    last = orc.dijkstra(graphs[-1].row, graphs[-1].col, graphs[-1].w, 0)

    def color(c):
        with smdp.Graph(c, g) as dg:
            return _timed(lambda: dg.color(False, smdp.SOL_TUNED), lambda: _equal(dg.read(smdp.RES_COLOR), colors), 40)

    def sources(c):
        with smdp.Graph(c, g) as dg:
            return _timed(lambda: dg.sssp_multi_source(srcs),
                          lambda: _equal(dg.read(smdp.RES_MDIST, count=20 * g.n).reshape(20, g.n), refs), 40)

    def batch(c):
        with smdp.Batch(c, graphs, np.zeros(30, np.int32)) as b:
            return _timed(lambda: b.run(), lambda: _equal(b.read(29), last), 40)

    print("contexts: colouring, sources and a batch", flush=True)
    _together([color, sources, batch])
