"""Parameters whose layout names the renumbered copy (set, or tuned for a
resident graph) do not keep calls on host or device arrays, which have no
copy, from the solves in one launch."""
import numpy as np
import pytest

import orc
import smdp
from test_zz_no_alloc import DeviceArrays, noalloc_sssp

pytestmark = pytest.mark.gpu

SMALL = smdp.gen_uniform(16384, 8, 1, 100, 1)
MIDDLE = smdp.gen_rmat(16, 8, wlo=1, whi=255, seed=2)


@pytest.mark.parametrize("layout", [smdp.LAYOUT_AUTO, smdp.LAYOUT_HOT, smdp.LAYOUT_BUCKETS])
@pytest.mark.parametrize("g,launches", [(SMALL, 1), (MIDDLE, 2)], ids=["lds", "rounds"])
def test_calls_on_arrays(g, launches, layout):
    ref, lv = orc.dijkstra(g.row, g.col, g.w, g.source), orc.bfs(g.row, g.col, g.source)
    with smdp.Context(0) as c:
        c.set_params(smdp.APP_SSSP, layout=layout)
        d, st = c.sssp(g, g.source, smdp.SOL_TUNED)
        assert np.array_equal(d, ref) and st.kernel_launches == launches
        if layout != smdp.LAYOUT_BUCKETS:
            c.set_params(smdp.APP_BFS, layout=layout)
        d, st = c.bfs(g, g.source, smdp.SOL_TUNED)
        assert np.array_equal(d, lv) and st.kernel_launches == launches
        arrays = DeviceArrays(g)
        try:
            rc, st = noalloc_sssp(c, arrays, g.source, smdp.SOL_TUNED)
            assert rc == smdp.OK and np.array_equal(arrays.read_dist(), ref) and st.kernel_launches == launches
        finally:
            arrays.close()
        with smdp.Graph(c, g) as dg:  # a resident graph follows the layout
            st = dg.sssp(g.source, smdp.SOL_TUNED)
            assert np.array_equal(dg.read(smdp.RES_DIST), ref)
            assert (st.kernel_launches == launches) == (layout == smdp.LAYOUT_AUTO)


def test_plain_csr_still_asks_for_the_hosts_rounds(ctx):
    old = ctx.get_params(smdp.APP_SSSP)
    try:
        ctx.set_params(smdp.APP_SSSP, layout=smdp.LAYOUT_CSR)
        d, st = ctx.sssp(SMALL, SMALL.source, smdp.SOL_TUNED)
        assert np.array_equal(d, orc.dijkstra(SMALL.row, SMALL.col, SMALL.w, SMALL.source))
        assert st.kernel_launches > 2
    finally:
        ctx.set_params(smdp.APP_SSSP, **old.as_dict())
