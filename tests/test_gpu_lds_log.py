"""What an LDS solve reports of its rounds: the per-round log of a profiled call,
and a round count that means the same as that of the other kinds of rounds."""
import numpy as np
import pytest

import orc
import smdp

pytestmark = pytest.mark.gpu


def _chain(n, w=100):
    return smdp.HostGraph(np.minimum(np.arange(n + 1), n - 1), np.arange(1, n), np.full(n - 1, w), 0)


@pytest.mark.parametrize("bfs", [False, True])
@pytest.mark.parametrize("name", ["rmat", "uniform", "chain", "heavy", "one vertex", "long chain"])
def test_round_log(ctx, name, bfs):
    g = {"rmat": lambda: smdp.gen_rmat(13, 16, wlo=1, whi=255, seed=8),
         "uniform": lambda: smdp.gen_uniform(16384, 8, 1, 100, 3),
         "chain": lambda: _chain(50),
         "heavy": lambda: smdp.HostGraph(np.arange(301) * 300, np.tile(np.arange(300), 300), np.arange(90000) % 77, 0),
         "one vertex": lambda: smdp.HostGraph([0, 0], [], [], 0),
         "long chain": lambda: _chain(6000)}[name]()
    run = ctx.bfs if bfs else ctx.sssp
    _, plain = run(g, g.source, smdp.SOL_TUNED)
    ctx.set_profiling(True)
    try:
        d, st = run(g, g.source, smdp.SOL_TUNED)
        q, arcs, ms = ctx.round_log()
    finally:
        ctx.set_profiling(False)
    assert np.array_equal(d, orc.bfs(g.row, g.col, g.source) if bfs else orc.dijkstra(g.row, g.col, g.w, g.source))
    assert st.kernel_launches == 1 and st.dominant_launches == 1
    logged = min(int(st.rounds), 4095)  # entries of the log
    assert len(q) == logged and q[0] == 1 and all(a > 0 for a in arcs[1:])
    if st.rounds == logged:
        assert sum(q) == st.vertices_expanded and sum(arcs) == st.edges_relaxed
    assert all(t >= 0 for t in ms) and sum(ms) <= st.ms_kernel
    assert plain.rounds == st.rounds or name not in ("chain", "one vertex", "long chain")


@pytest.mark.parametrize("bfs", [False, True])
def test_round_cap_by_the_reported_rounds(bfs):
    """A chain's rounds do not depend on the order of relaxations: one more than
    the reported rounds suffices as a cap, the reported rounds do not, whichever
    kind of rounds reported them."""
    app = smdp.APP_BFS if bfs else smdp.APP_SSSP
    g = _chain(20)
    with smdp.Context(0) as c:
        run = c.bfs if bfs else c.sssp
        d, st = run(g, 0, smdp.SOL_TUNED)
        assert st.kernel_launches == 1 and st.rounds == 19
        c.set_params(app, max_rounds=20)
        assert np.array_equal(run(g, 0, smdp.SOL_TUNED)[0], d)
        c.set_params(app, max_rounds=19)
        with pytest.raises(smdp.SmdpError) as e:
            run(g, 0, smdp.SOL_TUNED)
        assert e.value.code == smdp.ERR_OVERFLOW
