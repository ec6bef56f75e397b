"""The work plan of a small-graph batch (host/batch_plan.h, compiled here with
the host compiler).  What a barrier may wait for follows from the plan: no
workgroup belongs to two teams, and a graph is solved by the whole of one, so
no barrier waits for another graph's solve (a barrier gives up after about a
second, and a path of 490000 vertices takes two)."""
import os
import shutil
import subprocess

import numpy as np
import pytest

from conftest import PKG

HERE = os.path.dirname(os.path.abspath(__file__))
V, MAX = 32768, 16  # vertices of one workgroup, workgroups of a team


@pytest.fixture(scope="module")
def driver(tmp_path_factory):
    if not shutil.which("g++"):
        pytest.skip("no host C++ compiler")
    exe = str(tmp_path_factory.mktemp("plan") / "plan")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-I" + os.path.join(PKG, "host"),
                    os.path.join(HERE, "plan", "plan_driver.cpp"), "-o", exe], check=True)
    return exe


def _plan(driver, graphs, resident=256, cluster=MAX, share=None):
    share = sum(m for _, m, _ in graphs) / max(1, resident) if share is None else share
    text = f"{resident} {share} {cluster} {len(graphs)}\n" + "".join(f"{n} {m} {int(f)}\n" for n, m, f in graphs)
    out = subprocess.run([driver], input=text, capture_output=True, text=True, check=True).stdout.split("\n")
    base = [int(x) for x in out[0].split()[1:]]
    items = [tuple(map(int, x.split()[1:])) for x in out if x.startswith("item")]
    single = [tuple(map(int, x.split()[1:])) for x in out if x.startswith("single")]
    # teams are disjoint runs of workgroups, of two or more, that are resident together
    assert base[0] == 0 and all(2 <= b - a <= MAX for a, b in zip(base, base[1:])) and base[-1] <= resident
    assert sorted([g for g, _, _ in items] + [g for g, _ in single]) == list(range(len(graphs)))
    for g, team, clustered in items:
        n, _, fit = graphs[g]
        k = base[team + 1] - base[team]
        if clustered:
            block = -(-(-(-n // k)) // 64) * 64
            assert fit and k <= cluster and block <= V and block * k >= n
    for g, lds in single:
        assert lds == int(graphs[g][2] and graphs[g][0] <= V)
    return base, items, single


def test_long_paths_share_no_workgroup(driver):
    """20 paths that need 15 workgroups each, on 256: 17 teams, three with a second path."""
    base, items, single = _plan(driver, [(490000 - 137 * i, 489999 - 137 * i, True) for i in range(20)])
    assert not single and len(base) == 18
    assert sorted(np.bincount([t for _, t, _ in items])) == [1] * 14 + [2] * 3


@pytest.mark.parametrize("resident", [0, 1, 2, 5, 16, 31, 256])
@pytest.mark.parametrize("cluster", [1, 16])
def test_random_batches(driver, resident, cluster):
    r = np.random.RandomState(resident + cluster)
    for _ in range(20):
        graphs = [(int(np.exp(r.uniform(0, 14))), int(np.exp(r.uniform(0, 17))), r.rand() < 0.8)
                  for _ in range(r.randint(1, 400))]
        _plan(driver, graphs, resident, cluster)


def test_graphs_beyond_clusters_beside_them(driver):
    """A graph for the memory solve gets workgroups of its own, or the list of a team."""
    base, items, _ = _plan(driver, [(5_000_000, 40_000_000, True)] + [(400_000, 3_000_000, True)] * 40)
    assert items[0] == (0, 0, 0) and base[1] == 16
    many = [(400_000, 3_000_000 + i, True) for i in range(40)] + [(100_000, 2_900_000, False)]
    base, items, single = _plan(driver, many, share=200_000)
    assert not single and (40, 0) in [(g, c) for g, _, c in items]


def test_edges_of_one_workgroup(driver):
    for n, k in ((V, 0), (V + 1, 2), (2 * V, 2), (2 * V + 1, 3), (16 * V, 16)):
        base, items, single = _plan(driver, [(n, 10, True)], share=10)
        assert (len(single) == 1) == (k == 0) and (k == 0 or base[1] == k), n
    _, items, single = _plan(driver, [(16 * V + 1, 10, True), (10, 0, True)], share=10)
    assert not items and sorted(single) == [(0, 0), (1, 1)]


@pytest.mark.parametrize("count,resident,team", [(400, 512, 0), (512, 512, 0), (600, 512, 0), (255, 256, 0), (128, 256, 0),
                                                 (127, 256, 2), (100, 256, 2), (30, 256, 8), (4, 256, 16)])
def test_equal_graphs_in_memory_do_not_ask_for_more_workgroups_than_there_are(driver, count, resident, team):
    base, items, single = _plan(driver, [(4000, 32000, False)] * count, resident)
    if team:
        assert len(items) == count and set(np.diff(base)) == {team}
    else:
        assert not items and len(single) == count
    _, items, _ = _plan(driver, [(1000, 1 << 14, False)] * count, resident)
    assert not items  # too small for a team


def test_graphs_above_the_mean_get_teams_in_memory(driver):
    base, items, single = _plan(driver, [(90000, 900000, False)] * 3 + [(2000, 20000, False)] * 250)
    assert sorted(g for g, _, _ in items) == [0, 1, 2] and set(np.diff(base)) == {16} and len(single) == 250
