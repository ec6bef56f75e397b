"""PageRank on the plain in-CSR where rows and arcs together exceed the merge
tiles' 32-bit positions: the tuned solution takes a wave per row there, and the
last rows end just below arc 2^31."""
import os

import numpy as np
import pytest

import smdp

pytestmark = pytest.mark.gpu

N, M = 32768, 2 ** 31 - 5


def test_rows_up_to_the_last_arc():
    if os.sysconf("SC_PAGE_SIZE") * os.sysconf("SC_AVPHYS_PAGES") < 40 << 30:
        pytest.skip("needs 40 GB of host memory")
    # Arc p comes from vertex p mod N, so a row of 2 N arcs has every vertex twice; the
    # rows before the last three have all theirs, those have an odd number of arcs.
    col = np.tile(np.arange(N, dtype=np.int32), 2 ** 31 // N)[:M]
    row = np.minimum(np.arange(N + 1, dtype=np.int64) * 2 * N, M)
    row[-3:-1] -= [77, 1001]
    outdeg = (1 + np.arange(N) % 97).astype(np.int32)
    print(f"pagerank on {M} arcs", flush=True)
    with smdp.Context(0) as c:
        c.set_params(smdp.APP_PAGERANK, layout=smdp.LAYOUT_CSR)
        with smdp.Graph(c, smdp.HostGraph(row.astype(np.int32), col)) as dg:
            dg.set_outdeg(outdeg)
            st = dg.pagerank(smdp.pr_opts(0.85, 1.0, 0.0, 1), smdp.SOL_TUNED)
            rank = dg.read(smdp.RES_RANK, np.float32)
    assert st.rounds == 1
    d, share = float(np.float32(0.85)), (1.0 / N) / outdeg
    upto = np.concatenate([[0.0], np.cumsum(np.tile(share, 2))])  # sums over runs of the sources
    whole = share.sum()
    first, length = row[:-1] % N, np.diff(row)
    want = (1 - d) / N + d * (length // N * whole + upto[first + length % N] - upto[first])
    # a compensated sum rounded once, and the rounded contributions of its terms
    assert np.all(np.abs(rank - want) <= 4 * 2.0 ** -24 * want)
    assert len(np.unique(rank[-4:])) >= 3  # rows of different lengths
