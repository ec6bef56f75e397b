"""PageRank on the binned layout where workgroups sum one bin, two or none: the
loads issued after a workgroup's last bin, whose start falls on each place of a
group of 4 arcs, on arc 0, and behind the last arc."""
import numpy as np
import pytest

import orc
import smdp
from test_gpu_pr_auto_line import _layout
from test_gpu_pr_merge import D, TOL, _rows

pytestmark = pytest.mark.gpu

# a bin holds up to 1536 rows; a launch has 512 workgroups on 256 CUs
CASES = {
    "one_vertex": lambda: _rows([], 1, 1),
    "no_arcs": lambda: _rows([], 5000, 1),
    "one_bin": lambda: _rows([1, 2, 3, 4] * 384, 1536, 2),
    "two_bins": lambda: _rows([1] * 1537, 1537, 3),
    "arcs_then_none": lambda: _rows([7] * 1535 + [2], 20000, 4),
    "none_then_arcs": lambda: _rows([0] * 15000 + [5] * 1601, 16601, 5),
    "starts_1": lambda: _rows([1] + [4] * 12000, 12001, 6),
    "starts_2": lambda: _rows([2] + [4] * 12000, 12001, 7),
    "starts_3": lambda: _rows([3] + [4] * 12000, 12001, 8),
    "full_bins": lambda: _rows([16379, 1, 16379, 16000, 380, 3], 50, 9),
    "wide_and_rows": lambda: _rows([50000, 1, 0, 16380, 2] + [9] * 3000, 40000, 10),
    "a_bin_each": lambda: _rows([1] * (512 * 1536), 512 * 1536, 11),
    "a_bin_each_and_one": lambda: _rows([1] * (512 * 1536 + 1), 512 * 1536 + 1, 12),
    "two_bins_each": lambda: _rows([2, 0, 1, 1] * (256 * 1536), 1024 * 1536, 13),
}


@pytest.mark.parametrize("name", sorted(CASES))
def test_last_bins(ctx, name):
    ig = CASES[name]()
    print(f"binned {name} n={ig.n} m={ig.m}", flush=True)
    od = np.bincount(ig.col, minlength=ig.n).astype(np.int32)
    ref, _, _ = orc.pagerank(ig.row, ig.col, od, d=float(np.float32(D)), T=1.0, fixed_iters=12)
    with _layout(ctx, smdp.LAYOUT_BINNED), smdp.Graph(ctx, ig) as dg:
        dg.set_outdeg(od)
        got = []
        for _ in range(2):
            st = dg.pagerank(smdp.pr_opts(D, 1.0, 0.0, 12), smdp.SOL_TUNED)
            assert st.rounds == 12 and st.edges_relaxed == 12 * ig.m and st.vertices_expanded == 12 * ig.n
            got.append(dg.read(smdp.RES_RANK, np.float32))
    assert np.array_equal(got[0].view(np.uint32), got[1].view(np.uint32))
    assert np.all(np.abs(got[0].astype(np.float64) - ref) <= TOL * ref)
