"""Rows that cross many merge tiles, in SpMV and PageRank: more tiles than the
partials loaded at once, rows that begin or end on a tile's edge, behind empty
rows, and several of them.  SpMV is exact where every product and sum is a
whole number below 2^24; PageRank is compared with 64-bit ranks."""
import numpy as np
import pytest

import orc
import smdp

pytestmark = pytest.mark.gpu


def _rows(lengths, n, seed):
    r = np.random.RandomState(seed)
    deg = np.zeros(n, np.int64)
    deg[:len(lengths)] = lengths
    row = np.concatenate([[0], np.cumsum(deg)])
    return row.astype(np.int32), r.randint(0, n, row[-1]).astype(np.int32)


CASES = {
    "one row over 977 tiles": ([10 ** 6], 1000),
    "behind empty rows, from a tile's edge": ([0] * 1000 + [23, 16 * 1024, 5], 5000),  # 1023 items, then the row
    "one item into a tile": ([0] * 1000 + [24, 17 * 1024 + 1, 5], 5000),
    "ends on an edge": ([0] * 1024 + [33 * 1024 - 1, 7, 40000], 3000),
    "15, 16, 17 and 33 tiles": ([15 * 1024, 3, 16 * 1024, 17 * 1024, 0, 0, 33 * 1024, 1], 900),
    "tiles of 4096": ([3, 2_500_000, 1_000_000, 0, 9], 2000),
}


@pytest.mark.parametrize("name", list(CASES))
def test_spmv(ctx, name):
    lengths, n = CASES[name]
    row, col = _rows(lengths, n, 3)
    r = np.random.RandomState(4)
    val = r.choice([-1.0, 1.0, 2.0], len(col)).astype(np.float32)
    x = r.randint(0, 3, n).astype(np.float32)
    terms = np.concatenate([[0.0], np.cumsum(val.astype(np.float64) * x[col])])
    want = terms[row[1:]] - terms[row[:-1]]
    assert np.abs(want).max() < 2 ** 24
    with smdp.Graph(ctx, smdp.HostGraph(row, col)) as dg:
        dg.set_values(val)
        dg.set_x(x)
        for _ in range(2):
            dg.spmv(smdp.SOL_TUNED)
            assert np.array_equal(dg.read(smdp.RES_Y, np.float32).astype(np.float64), want)


@pytest.mark.parametrize("name", list(CASES))
def test_pagerank(ctx, name):
    lengths, n = CASES[name]
    row, col = _rows(lengths, n, 5)
    outdeg = np.bincount(col, minlength=n).astype(np.int32)
    ref, _, _ = orc.pagerank(row, col, outdeg, d=float(np.float32(0.85)), T=1.0, fixed_iters=8)
    with smdp.Graph(ctx, smdp.HostGraph(row, col)) as dg:
        dg.set_outdeg(outdeg)
        dg.pagerank(smdp.pr_opts(.85, 1.0, 0.0, 8), smdp.SOL_TUNED)
        rank = dg.read(smdp.RES_RANK, np.float32).astype(np.float64)
    # each rank is rounded to 24 bits once an iteration, and errors do not grow (damping below 1)
    assert np.abs(rank - ref).sum() <= 8 * 2.0 ** -23 and np.all(np.abs(rank - ref) <= 16 * 2.0 ** -23 * ref)
