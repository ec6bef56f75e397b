"""PageRank by merge-path tiles on more arcs than the automatic layout leaves to
them (2^22): the plain in-CSR asked for, with the largest tiles (32 items a
thread), beside the binned layout that automatic takes."""
import pytest

import smdp
from test_gpu_pr_merge import _check, _rows

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("layout", [smdp.LAYOUT_CSR, smdp.LAYOUT_AUTO])
@pytest.mark.parametrize("name", ["rmat", "hub and empty rows"])
def test_above_the_automatic_line(ctx, name, layout):
    ig = {"rmat": lambda: smdp.invert(smdp.gen_rmat(18, 17, seed=9)),
          "hub and empty rows": lambda: _rows([1_500_000, 0, 3] + [0] * 70000 + [9] * 350000, 600000, 12)}[name]()
    assert ig.m > 1 << 22
    print(f"pagerank {name}, {ig.m} arcs, layout {layout}", flush=True)
    old = ctx.get_params(smdp.APP_PAGERANK)
    try:
        ctx.set_params(smdp.APP_PAGERANK, layout=layout)
        _check(ctx, ig)
    finally:
        ctx.set_params(smdp.APP_PAGERANK, **old.as_dict())
