"""Tuned frontier rounds whose queue fills the launch's tiles exactly, one
entry short or one over: up to one tile (256 entries) per workgroup each
workgroup takes its own tile, beyond that tiles are claimed.  The same line for
the grid-queue chunks.  Whole-number results: exact against the oracle."""
import numpy as np
import pytest

import orc
import smdp

pytestmark = pytest.mark.gpu


def _fan(k, deg):
    """0 -> k children, each with deg arcs to the last vertices."""
    sinks = max(deg, 1)
    n = 1 + k + sinks
    row = np.zeros(n + 1, np.int64)
    row[1] = k
    row[2:k + 2] = k + deg * np.arange(1, k + 1)
    row[k + 2:] = row[k + 1]
    col = np.concatenate([1 + np.arange(k), np.tile(1 + k + np.arange(deg), k)])
    w = (np.arange(len(col)) % 9 + 1).astype(np.int32)
    return smdp.HostGraph(row, col, w, 0)


@pytest.mark.parametrize("deg", [1, 40])  # 40: above the split of short queues, so chunks of the grid queue
@pytest.mark.parametrize("extra", [-256, -1, 0, 1, 256, 2000])
def test_tiles_around_the_grid(ctx, deg, extra):
    cus = ctx.info()["cus"]
    k = (cus * 256 if deg == 1 else cus * 8) + extra
    g = _fan(k, deg)
    print(f"fan k={k} deg={deg}", flush=True)
    old = {a: ctx.get_params(a) for a in (smdp.APP_SSSP, smdp.APP_BFS)}
    try:
        for app in old:
            ctx.set_params(app, wg_per_cu=1, split_threshold=64, chunk=64)
        d, _ = ctx.sssp(g, 0, smdp.SOL_TUNED)
        assert np.array_equal(d, orc.dijkstra(g.row, g.col, g.w, 0))
        lv, _ = ctx.bfs(g, 0, smdp.SOL_TUNED)
        assert np.array_equal(lv, orc.bfs(g.row, g.col, 0))
    finally:
        for app, p in old.items():
            ctx.set_params(app, **p.as_dict())
