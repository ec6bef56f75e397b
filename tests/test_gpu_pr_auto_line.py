"""The automatic PageRank layout: a graph that stays on the device takes the
binned layout (two launches an iteration) once its merge tiles do not run all
at once, a call on host arrays stays on tiles (one launch) up to 2^22 arcs."""
from contextlib import contextmanager

import numpy as np
import pytest

import orc
import smdp
from test_gpu_pr_merge import D, TOL

pytestmark = pytest.mark.gpu


def _uniform(n, m, seed=3):
    r = np.random.RandomState(seed)
    row = np.concatenate([[0], np.cumsum(np.bincount(r.randint(0, n, m), minlength=n))])
    return smdp.HostGraph(row, r.randint(0, n, m), None, 0)


@contextmanager
def _layout(ctx, layout):
    old = ctx.get_params(smdp.APP_PAGERANK)
    ctx.set_params(smdp.APP_PAGERANK, layout=layout)
    try:
        yield
    finally:
        ctx.set_params(smdp.APP_PAGERANK, **old.as_dict())


# rows + arcs at the line of 2^22 on 256 CUs, and just above and below 2^21 arcs beyond it
@pytest.mark.parametrize("n,m,binned", [(1 << 20, 3 << 20, False), ((1 << 20) + 1, 3 << 20, True),
                                        ((2 << 20) + 99, 2 << 20, False), ((2 << 20) + 99, (2 << 20) + 1, True),
                                        (1000, (1 << 22) - 1000, False), (1001, (1 << 22) - 1000, True)])
def test_resident_and_drop_in(ctx, n, m, binned):
    ig = _uniform(n, m)
    print(f"n {n}, m {m}", flush=True)
    od = np.bincount(ig.col, minlength=n).astype(np.int32)
    opts = smdp.pr_opts(D, 1.0, 0.0, 12)
    resident = {}
    with smdp.Graph(ctx, ig) as dg:
        dg.set_outdeg(od)
        for layout in (smdp.LAYOUT_AUTO, smdp.LAYOUT_CSR, smdp.LAYOUT_BINNED, smdp.LAYOUT_AUTO):
            with _layout(ctx, layout):
                st = dg.pagerank(opts, smdp.SOL_TUNED)
            resident[layout] = st.kernel_launches, dg.read(smdp.RES_RANK, np.float32)
    tiles, bins = resident[smdp.LAYOUT_CSR], resident[smdp.LAYOUT_BINNED]
    assert bins[0] - tiles[0] == 12  # one launch more an iteration
    like = bins if binned else tiles
    assert resident[smdp.LAYOUT_AUTO][0] == like[0]
    assert np.array_equal(resident[smdp.LAYOUT_AUTO][1], like[1])
    rank, st = ctx.pagerank(ig, od, opts, smdp.SOL_TUNED)
    assert st.kernel_launches == tiles[0] and np.array_equal(rank, tiles[1])
    ref, _, _ = orc.pagerank(ig.row, ig.col, od, d=float(np.float32(D)), T=1.0, fixed_iters=12)
    for _, r in (tiles, bins):
        assert np.all(np.abs(r.astype(np.float64) - ref) <= TOL * ref)
