"""The window of an LDS solve follows the weights over their whole range: as
weights and distances scale, rounds and relaxed arcs stay about the same."""
import numpy as np
import pytest

import orc
import smdp

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["uniform", "star"])
def test_rounds_do_not_grow_with_the_weights(ctx, kind):
    r = np.random.RandomState(3)
    if kind == "uniform":
        n, deg = 16384, 8
        row, col = np.arange(n + 1) * deg, r.randint(0, n, n * deg)
    else:
        n = 30000
        row, col = np.minimum(np.arange(n + 1) * (n - 1), n - 1), np.arange(1, n)
    base = r.randint(1, 64, len(col))
    rounds = {}
    # 20 times the largest weight stays below the 2^30 that marks an unreached vertex
    for shift in (0, 8, 14, 16, 18, 20) + ((23, 24) if kind == "star" else ()):
        g = smdp.HostGraph(row, col, base << shift, 0)
        d, st = ctx.sssp(g, 0, smdp.SOL_TUNED)
        assert np.array_equal(d, orc.dijkstra(g.row, g.col, g.w, 0)) and st.kernel_launches == 1
        rounds[shift] = int(st.rounds)
    print(kind, rounds, flush=True)
    # at a shift of 0 the window is rounded to a whole number: compare the others
    assert max(rounds.values()) <= 1.5 * rounds[8] + 2, rounds


def test_largest_weights(ctx):
    """A few light paths beside weights just below 2^30, and the mean over all of them."""
    r = np.random.RandomState(5)
    n, m = 4000, 40000
    src, dst = r.randint(0, n, m), r.randint(0, n, m)
    order = np.argsort(src, kind="stable")
    row = np.concatenate([[0], np.cumsum(np.bincount(src, minlength=n))])
    for w in (r.randint(2 ** 29, 2 ** 30, m), np.where(r.rand(m) < 0.5, 2 ** 30 - 1, 1), np.full(m, 2 ** 30 - 1)):
        g = smdp.HostGraph(row, dst[order], w, 0)
        d, _ = ctx.sssp(g, 0, smdp.SOL_TUNED)
        assert np.array_equal(d, orc.dijkstra(g.row, g.col, g.w, 0))
