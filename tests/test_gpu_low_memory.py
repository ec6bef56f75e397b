"""Calls that take extra device memory for speed, with the device nearly full:
they go on without it and stay exact."""
import contextlib
import ctypes as C

import numpy as np
import pytest

import orc
import smdp
from conftest import random_graph
from test_zz_no_alloc import hip

pytestmark = pytest.mark.gpu

MB = 1 << 20


def _free():
    free, total = C.c_size_t(), C.c_size_t()
    assert hip().hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


@contextlib.contextmanager
def device_left(mb):
    """About mb MB of device memory are free inside (within 16 MB below)."""
    fill = []

    def take(nbytes):
        p = C.c_void_p()
        assert hip().hipMalloc(C.byref(p), C.c_size_t(nbytes)) == 0
        fill.append(p)

    try:
        while _free() > (mb + 1100) * MB:
            take(_free() - (mb + 1024) * MB)
        while _free() > mb * MB:
            take(16 * MB)
        print(f"device memory left: {_free() // MB} MB", flush=True)
        yield
    finally:
        for p in fill:
            hip().hipFree(p)


def test_batch_without_memory_for_messages(ctx):
    """15M arcs between the 16 workgroups of a cluster: 215 MB of messages
    beside 126 MB for the batch itself."""
    row, col, w = random_graph(500000, 15000000, 3, 1, 50)
    g = smdp.HostGraph(row, col, w, 0)
    ref = orc.dijkstra(row, col, w, 0)
    with device_left(260):
        with smdp.Batch(ctx, [g], np.zeros(1, np.int32)) as b:
            for _ in range(2):
                b.run()
                assert np.array_equal(b.read(0), ref)
    with smdp.Batch(ctx, [g], np.zeros(1, np.int32)) as b:
        b.run()
        assert np.array_equal(b.read(0), ref)


def test_dropin_without_memory_for_round_queues(ctx):
    """The queues of the rounds in one launch (32 bytes per vertex) beside a
    graph of 8 million vertices."""
    n = 8_000_000
    row = np.minimum(np.arange(n + 1, dtype=np.int64) * 2, n - 1).astype(np.int32)
    col = np.arange(1, n, dtype=np.int32)  # a binary heap: vertex v has 2v + 1 and 2v + 2
    g = smdp.HostGraph(row, col, np.ones(n - 1, np.int32), 0)
    want = np.floor(np.log2(np.arange(1, n + 1))).astype(np.int32)
    with smdp.Context(0) as c, device_left(420):
        for _ in range(2):
            lv, _ = c.bfs(g, 0, smdp.SOL_TUNED)
            assert np.array_equal(lv, want)
    lv, st = ctx.bfs(g, 0, smdp.SOL_TUNED)
    assert np.array_equal(lv, want) and st.kernel_launches == 2


def test_multi_source_without_memory_for_bounds(ctx):
    """The bounds (12 bytes per vertex) that skip arcs, beside 274 bytes per
    vertex that the call cannot do without."""
    n = 3_000_000
    row, col, w = random_graph(n, 3_000_000, 9, 1, 90)
    g = smdp.HostGraph(row, col, w)
    srcs = np.array([0, 5, n - 1, 77], np.int32)
    refs = np.stack([orc.dijkstra(row, col, w, int(s)) for s in srcs])

    def solve(dg):
        st = dg.sssp_multi_source(srcs)
        assert np.array_equal(dg.read(smdp.RES_MDIST, count=4 * n).reshape(4, n), refs)
        return st

    with smdp.Graph(ctx, g) as dg:
        before = _free()
        solve(dg)
        used = before - _free()
    print(f"multi-source: {used // MB} MB", flush=True)
    with smdp.Graph(ctx, g) as dg:
        with device_left(used // MB - 6):
            for _ in range(2):
                assert solve(dg).arcs_skipped == 0
