"""What the autotuner chooses among where the automatic layout runs kernels that
read few parameters: it never gives up the solve in one launch for a slower
layout, leaves parameters alone that change nothing, and does not take cache
entries found for other kernels."""
import json

import numpy as np
import pytest

import orc
import smdp

pytestmark = pytest.mark.gpu

G = smdp.gen_rmat(16, 8, wlo=1, whi=255, seed=3)


@pytest.fixture
def fresh():
    with smdp.Context(0) as c:
        yield c


def test_sssp_keeps_the_rounds_in_one_launch(fresh, tmp_path):
    cache = tmp_path / "t.json"
    with smdp.Graph(fresh, G) as dg:
        p = dg.autotune(smdp.APP_SSSP, G.source, cache)
        assert p.layout == smdp.LAYOUT_AUTO, p.as_dict()
        assert dg.sssp(G.source, smdp.SOL_TUNED).kernel_launches == 2
        assert np.array_equal(dg.read(smdp.RES_DIST), orc.dijkstra(G.row, G.col, G.w, G.source))
        key = list(json.loads(cache.read_text()))[0]
        assert ":rounds:" in key
        # an entry for this graph from when it was solved on the renumbered copy
        old = dict(p.as_dict(), layout=smdp.LAYOUT_BUCKETS, delta=64)
        fields = ["heavy_threshold", "split_threshold", "chunk", "wg_per_cu", "batch_rounds", "max_rounds", "layout",
                  "delta", "persistent", "group_share"]
        body = ", ".join(f'"{f}": {old[f]}' for f in fields)
        cache.write_text("{\n  \"%s\": {%s}\n}\n" % (key.replace("rounds:", ""), body))
        assert dg.autotune(smdp.APP_SSSP, G.source, cache).layout == smdp.LAYOUT_AUTO
        assert len(json.loads(cache.read_text())) == 2
        # while one under its own key is taken as it is
        cache.write_text("{\n  \"%s\": {%s}\n}\n" % (key, body))
        assert dg.autotune(smdp.APP_SSSP, G.source, cache).layout == smdp.LAYOUT_BUCKETS


def test_parameters_without_effect_stay(fresh):
    with smdp.Graph(fresh, G) as dg:
        for app in (smdp.APP_BFS, smdp.APP_MSSSP):
            base = fresh.get_params(app).as_dict()
            got = dg.autotune(app, G.source).as_dict()
            if app == smdp.APP_MSSSP:
                assert got["wg_per_cu"] in (base["wg_per_cu"], 4, 8)
                got["wg_per_cu"] = base["wg_per_cu"]
            assert got == base and fresh.get_params(app).split_threshold == base["split_threshold"]
        dg.bfs(G.source, smdp.SOL_TUNED)
        assert np.array_equal(dg.read(smdp.RES_LEVEL), orc.bfs(G.row, G.col, G.source))


def test_large_graphs_search_the_renumbered_layouts_too(fresh):
    """2^23 arcs: the automatic layout is buckets, and candidates of every kind solve exactly."""
    g = smdp.gen_rmat(19, 16, wlo=1, whi=255, seed=4)
    with smdp.Graph(fresh, g) as dg:
        p = dg.autotune(smdp.APP_SSSP, g.source)
        assert p.layout in (smdp.LAYOUT_AUTO, smdp.LAYOUT_BUCKETS, smdp.LAYOUT_HOT)
        assert dg.sssp(g.source, smdp.SOL_TUNED).kernel_launches > 2
        assert np.array_equal(dg.read(smdp.RES_DIST), orc.dijkstra(g.row, g.col, g.w, g.source))
