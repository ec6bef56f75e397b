"""SSSP and BFS rounds in one launch: shares of a round's arcs, windows of its queue, parts of a
workgroup, the round cap, and the sizes at which the solve goes to them."""
import numpy as np
import pytest
import orc
import smdp
from test_zz_no_alloc import DeviceArrays, noalloc_sssp

pytestmark = pytest.mark.gpu


def _csr(n, src, dst, w):
    src, dst, w = np.asarray(src), np.asarray(dst), np.asarray(w)
    order = np.argsort(src, kind="stable")
    row = np.zeros(n + 1, np.int64)
    np.add.at(row, src + 1, 1)
    return smdp.HostGraph(np.cumsum(row).astype(np.int32), dst[order].astype(np.int32), w[order].astype(np.int32), 0)


def _random(n, m, seed, wlo=0, whi=40):
    r = np.random.RandomState(seed)
    return _csr(n, r.randint(0, n, m), r.randint(0, n, m), r.randint(wlo, whi, m))


def _path(n):
    v = np.arange(n - 1)
    return _csr(n, v, v + 1, 1 + v % 5)


def _star(leaves):
    """The source's leaves, each with an arc to one of 7 vertices."""
    v = 1 + np.arange(leaves)
    return _csr(leaves + 8, np.concatenate([np.zeros(leaves, int), v]),
                np.concatenate([v, leaves + 1 + v % 7]), np.concatenate([v % 11, 1 + v % 3]))


GRAPHS = {
    "one": lambda: smdp.HostGraph([0, 0], [], [], 0),
    "source without arcs": lambda: _csr(3, [1], [2], [4]),
    "loops and doubles": lambda: _csr(3, [0, 0, 0, 0, 1, 1], [0, 1, 1, 1, 1, 2], [0, 9, 7, 8, 0, 0]),
    "path": lambda: _path(700),
    "star 1023": lambda: _star(1023),
    "star 1024": lambda: _star(1024),
    "star 1025": lambda: _star(1025),
    "star 40000": lambda: _star(40000),
    "random": lambda: _random(20000, 70000, 3),
    "zero weights": lambda: _random(5000, 30000, 4, 0, 2),
    "dense": lambda: _random(600, 90000, 5),
    "rmat": lambda: smdp.gen_rmat(15, 24, wlo=1, whi=255, seed=6),
}


def _solve(ctx, g, bfs):
    """Rounds in one launch also where a smaller solver would take the graph (a round cap below what
    that one needs)."""
    app = smdp.APP_BFS if bfs else smdp.APP_SSSP
    old = ctx.get_params(app)
    try:
        ctx.set_params(app, max_rounds=2 * g.n + 1)
        with smdp.Graph(ctx, g) as dg:
            st = dg.bfs(g.source, smdp.SOL_TUNED) if bfs else dg.sssp(g.source, smdp.SOL_TUNED)
            return dg.read(smdp.RES_LEVEL if bfs else smdp.RES_DIST), st
    finally:
        ctx.set_params(app, **old.as_dict())


def _check(ctx, g, bfs):
    d, st = _solve(ctx, g, bfs)
    ref = orc.bfs(g.row, g.col, g.source) if bfs else orc.dijkstra(g.row, g.col, g.w, g.source)
    assert np.array_equal(d, ref)
    reached = ref != (smdp.BFS_UNDEF if bfs else smdp.SSSP_INF)
    assert st.m_reached == int(np.diff(g.row)[reached].sum())
    return st


@pytest.mark.parametrize("bfs", [False, True])
@pytest.mark.parametrize("name", list(GRAPHS))
def test_parity(ctx, name, bfs):
    st = _check(ctx, GRAPHS[name](), bfs)
    assert st.kernel_launches <= 2


@pytest.mark.parametrize("bfs", [False, True])
def test_a_workgroup_queues_several_parts(ctx, bfs):
    """A round of 3000000 arcs that each queue a vertex, over 15000 a workgroup."""
    st = _check(ctx, _star(3_000_000), bfs)
    assert st.rounds == 2 and st.kernel_launches == 2


def test_negative_arcs_without_cycles(ctx):
    r = np.random.RandomState(7)
    n, m = 3000, 40000
    a = r.randint(0, n - 1, m)
    b = a + 1 + (r.rand(m) * (n - 1 - a)).astype(int)
    g = _csr(n, a, b, r.randint(-90, 100, m))
    d, _ = _solve(ctx, g, False)
    ref = np.full(n, smdp.SSSP_INF, np.int64)
    ref[0] = 0
    for u in range(n):
        for e in range(g.row[u], g.row[u + 1]):
            if ref[u] < smdp.SSSP_INF:
                ref[g.col[e]] = min(ref[g.col[e]], ref[u] + g.w[e])
    assert np.array_equal(d, ref)


@pytest.mark.parametrize("bfs", [False, True])
def test_round_cap(ctx, bfs):
    """A path of 600 vertices takes 599 rounds (its last vertex has no arcs) and
    one that finds no work, which the cap counts as it does where the host
    drives the rounds."""
    app = smdp.APP_BFS if bfs else smdp.APP_SSSP
    g = _path(600)
    old = ctx.get_params(app)
    try:
        for cap, ok in ((598, False), (599, False), (600, True), (601, True)):
            ctx.set_params(app, max_rounds=cap)
            run = ctx.bfs if bfs else ctx.sssp
            if ok:
                assert run(g, 0, smdp.SOL_TUNED)[1].rounds == 599
            else:
                with pytest.raises(smdp.SmdpError) as e:
                    run(g, 0, smdp.SOL_TUNED)
                assert e.value.code == smdp.ERR_OVERFLOW
    finally:
        ctx.set_params(app, **old.as_dict())


@pytest.mark.parametrize("n", [32769, (1 << 18) - 1, 1 << 18, (1 << 18) + 1])
def test_device_csr_sizes(ctx, n):
    """The fixed array's queues hold 2^18 vertices; more go through the host-driven rounds."""
    g = _random(n, 4 * n, 9, 1, 200)
    d = DeviceArrays(g)
    try:
        for _ in range(2):
            rc, _ = noalloc_sssp(ctx, d, 0, smdp.SOL_TUNED)
            assert rc == smdp.OK and np.array_equal(d.read_dist(), orc.dijkstra(g.row, g.col, g.w, 0))
    finally:
        d.close()


def test_round_log(ctx):
    g = smdp.gen_rmat(16, 16, wlo=1, whi=255, seed=8)
    ctx.set_profiling(True)
    try:
        _, st = ctx.sssp(g, g.source, smdp.SOL_TUNED)
        q, arcs, ms = ctx.round_log()
    finally:
        ctx.set_profiling(False)
    assert len(q) == st.rounds and q[0] == 1
    assert sum(q) == st.vertices_expanded and sum(arcs) == st.edges_relaxed
    assert st.dominant_launches == 1 and 0 < sum(ms) <= st.ms_kernel
