"""PageRank by merge-path tiles (the tuned solution on the plain in-CSR):
graphs whose row ends and arcs fill tiles exactly, one item short or over, rows
that cross several tiles, long runs of empty rows, and both tile sizes, against
the FP64 oracle with the same number of iterations.

Tolerance: every term of a row's sum is non-negative, so relative errors do not
grow in a sum.  One iteration rounds a rank at most eight times (division,
compensated sum, fma, the two parts of the base term and their conversions),
and the iteration damps earlier errors by d, so ranks lie within
8 u / (1 - d) of the FP64 ones, u = 2^-24.
"""
import numpy as np
import pytest

import orc
import smdp

pytestmark = pytest.mark.gpu

D = 0.85
TOL = 8 * 2.0 ** -24 / (1 - D)


def _rows(lens, n, seed):
    """An in-CSR with the given row lengths (rest empty) and random sources."""
    deg = np.zeros(n, np.int64)
    deg[:len(lens)] = lens
    row = np.concatenate([[0], np.cumsum(deg)]).astype(np.int32)
    col = np.random.RandomState(seed).randint(0, n, row[-1]).astype(np.int32)
    return smdp.HostGraph(row, col)


def _cases():
    out = {"one_vertex": _rows([], 1, 1), "loop": _rows([1], 1, 1), "no_arcs": _rows([], 3000, 1)}
    for total in (255, 1023, 1024, 1025, 2047, 2048, 2049):  # tiles of 1024 items
        n = total // 3
        out[f"hub_{total}"] = _rows([total - n], n, total)
        lens = np.full(n, (total - n) // n)
        lens[: (total - n) % n] += 1
        out[f"even_{total}"] = _rows(lens, n, total)
    out["hub_first"] = _rows([9000] + [1] * 500, 2000, 3)
    out["hub_last"] = _rows([0] * 4000 + [7000], 4001, 4)
    out["hubs_apart"] = _rows([3000, 0, 0, 5000] + [0] * 2500 + [4096, 1, 1024], 4000, 5)
    out["rmat11"] = smdp.invert(smdp.gen_rmat(11, 16, seed=7))
    return out


CASES = _cases()


def _check(ctx, ig):
    od = np.bincount(ig.col, minlength=ig.n).astype(np.int32)
    r, st = ctx.pagerank(ig, od, smdp.pr_opts(D, 1.0, 0.0, 12), smdp.SOL_TUNED)
    assert st.rounds == 12 and st.edges_relaxed == 12 * ig.m and st.vertices_expanded == 12 * ig.n
    ref, _, _ = orc.pagerank(ig.row, ig.col, od, d=float(np.float32(D)), T=1.0, fixed_iters=12)
    assert np.all(np.abs(r.astype(np.float64) - ref) <= TOL * ref)
    r2, _ = ctx.pagerank(ig, od, smdp.pr_opts(D, 1.0, 0.0, 12), smdp.SOL_TUNED)
    assert np.array_equal(r.view(np.uint32), r2.view(np.uint32))


@pytest.mark.parametrize("name", sorted(CASES))
def test_small_tiles(ctx, name):
    print(f"pr merge {name}", flush=True)
    _check(ctx, CASES[name])


def test_large_tiles(ctx):
    """Above 2^21 merge items the tiles hold 4096 items (layout forced to CSR:
    automatic takes the binned one there)."""
    g = smdp.gen_rmat(17, 16, seed=9)
    old = ctx.get_params(smdp.APP_PAGERANK)
    try:
        ctx.set_params(smdp.APP_PAGERANK, layout=smdp.LAYOUT_CSR)
        _check(ctx, smdp.invert(g))
    finally:
        ctx.set_params(smdp.APP_PAGERANK, **old.as_dict())


# The largest matrix of each tile size (4, 8, 16 items a thread) on 256 CUs and the smallest of the next,
# with a hub over many tiles, empty rows and a ragged end; and the last size before the binned layout.
@pytest.mark.parametrize("total", [140800, 140801, 409600, 409601, 1280000, 1280001, 1 << 22])
def test_tile_sizes_of_a_pass(ctx, total):
    n = total // 9 + 1
    lens = np.random.RandomState(total % 1000).randint(0, 9, n - 200)
    lens[7] += total - n - lens.sum()
    ig = _rows(lens, n, 11)
    assert ig.n + ig.m == total and lens[7] > 4096
    _check(ctx, ig)
