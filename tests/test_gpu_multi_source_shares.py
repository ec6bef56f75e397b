"""Multi-source SSSP: equal shares of a round's arcs, and the bounds that let arcs be skipped."""
import numpy as np
import pytest
import orc
import smdp

pytestmark = pytest.mark.gpu


def _csr(n, src, dst, w):
    order = np.argsort(src, kind="stable")
    row = np.zeros(n + 1, np.int64)
    np.add.at(row, np.asarray(src) + 1, 1)
    return smdp.HostGraph(np.cumsum(row).astype(np.int32), np.asarray(dst)[order].astype(np.int32),
                          np.asarray(w)[order].astype(np.int32))


def _rmat_and_path():
    """A component that never reaches the vertex of most arcs: its sources are in no bound."""
    g = smdp.gen_rmat(12, 12, wlo=1, whi=255, seed=3)
    src = np.concatenate([np.repeat(np.arange(g.n), np.diff(g.row)), g.n + np.arange(299)])
    dst = np.concatenate([g.col, g.n + 1 + np.arange(299)])
    return _csr(g.n + 300, src, dst, np.concatenate([g.w, np.full(299, 7)])), [g.n, g.n + 150, g.n + 299]


def _tail_into_core():
    """Sources that reach the core only after many rounds: the bounds are made anew."""
    g = smdp.gen_rmat(12, 12, wlo=1, whi=255, seed=5)
    hub = int(np.argmax(np.diff(g.row)))
    src = np.concatenate([np.repeat(np.arange(g.n), np.diff(g.row)), g.n + np.arange(40)])
    dst = np.concatenate([g.col, g.n + 1 + np.arange(39), [hub]])
    return _csr(g.n + 40, src, dst, np.concatenate([g.w, np.full(40, 3)])), [g.n, g.n + 20, g.n + 33, g.n + 36]


def _sparse():
    """Long parts of the queue per workgroup, many of them vertices without arcs."""
    r = np.random.RandomState(2)
    n, m = 65536, 90000
    return _csr(n, np.minimum(r.randint(0, n, m), r.randint(0, n, m)), r.randint(0, n, m), r.randint(0, 99, m)), []


def _star():
    """One vertex of 100000 arcs, shared by every wave, its targets without arcs but one."""
    n = 100_002
    dst = np.arange(1, n - 1)
    return _csr(n, np.concatenate([np.zeros(len(dst), int), [n - 2, n - 1]]), np.concatenate([dst, [n - 1, 0]]),
                np.concatenate([1 + dst % 9, [4, 5]])), [0, n - 2, n - 1, 5]


def _grid():
    k = 70
    v = np.arange(k * k).reshape(k, k)
    a = np.concatenate([v[:, :-1].ravel(), v[:-1].ravel()])
    b = np.concatenate([v[:, 1:].ravel(), v[1:].ravel()])
    r = np.random.RandomState(4)
    return _csr(k * k, np.concatenate([a, b]), np.concatenate([b, a]), r.randint(1, 50, 2 * len(a))), []


def _one():
    return _csr(2, [0], [1], [9]), [0, 1]


@pytest.mark.parametrize("k", [1, 5, 64, 70])
@pytest.mark.parametrize("make", [_rmat_and_path, _tail_into_core, _sparse, _star, _grid, _one])
def test_every_source(make, k):
    g, first = make()
    srcs = np.array((first + list(np.random.RandomState(6).randint(0, g.n, 70)))[:k], np.int32)
    with smdp.Context(0) as ctx:
        d, _ = ctx.sssp_multi_source(g, srcs)
    for i in range(k):
        assert np.array_equal(d[i], orc.dijkstra(g.row, g.col, g.w, int(srcs[i]))), i


@pytest.mark.parametrize("k", [3, 64])
def test_negative_arcs_without_cycles(k):
    """Arcs from lower to higher ids with weights of both signs, over a core of many arcs."""
    r = np.random.RandomState(8)
    n, m = 3000, 60000
    a = (r.rand(m) ** 2 * (n - 1)).astype(int)
    b = a + 1 + (r.rand(m) * (n - 1 - a)).astype(int)
    w = r.randint(-200, 300, m)
    g = _csr(n, a, b, w)
    srcs = r.randint(0, 200, k).astype(np.int32)
    with smdp.Context(0) as ctx:
        d, _ = ctx.sssp_multi_source(g, srcs)
    ref = np.full((k, n), 1 << 30, np.int64)
    ref[np.arange(k), srcs] = 0
    for u in range(n):  # ids are a topological order
        for e in range(g.row[u], g.row[u + 1]):
            ok = ref[:, u] < 1 << 30
            ref[ok, g.col[e]] = np.minimum(ref[ok, g.col[e]], ref[ok, u] + g.w[e])
    assert np.array_equal(d, ref)
