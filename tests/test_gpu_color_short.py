"""Short layers of the tuned colouring: the run of them in one launch must hand a layer back
when a count does not fit its barrier flag, and go on after it."""
import numpy as np
import pytest
import orc
import smdp

pytestmark = pytest.mark.gpu


def _graph(n, src, dst):
    """The symmetric graph of the edges src - dst."""
    s, d = np.concatenate([src, dst]), np.concatenate([dst, src])
    order = np.argsort(s, kind="stable")
    row = np.zeros(n + 1, np.int64)
    np.add.at(row, s + 1, 1)
    return smdp.HostGraph(np.cumsum(row).astype(np.int32), d[order].astype(np.int32))


def _path(first, count):
    v = np.arange(first, first + count)
    return v[:-1], v[1:]


def _check(g, k_min, use_prio):
    prio = np.arange(g.n, dtype=np.uint32) if use_prio else None  # the order of the ids
    ref, k = orc.color_closed(g.row, g.col, None)
    assert k >= k_min
    with smdp.Context(0) as ctx:
        c, st = ctx.color(g, prio, smdp.SOL_TUNED)
    assert np.array_equal(c, ref)
    assert st.rounds == k
    assert st.q_push[0] == int((ref >= 2).sum())
    assert st.edges_relaxed >= 0


@pytest.mark.parametrize("use_prio", [False, True])
@pytest.mark.parametrize("lead", [1, 2, 40])
def test_hub_of_more_arcs_than_a_flag_holds(lead, use_prio):
    """A path, a hub of 1100000 leaves (more than 2^20 - 1 arcs in one workgroup's queue,
    met at the run's first layer and later ones), and a path after the last leaf."""
    leaves, tail = 1_100_000, 30
    hub = lead
    n = lead + 1 + leaves + tail
    leaf = np.arange(hub + 1, hub + 1 + leaves)
    p, q = _path(0, lead + 1), _path(int(leaf[-1]), tail + 1)
    _check(_graph(n, np.concatenate([p[0], np.full(leaves, hub), q[0]]), np.concatenate([p[1], leaf, q[1]])),
           lead + 2 + tail, use_prio)


@pytest.mark.parametrize("use_prio", [False, True])
def test_more_entries_than_a_flag_holds(use_prio):
    """One layer holds x, whose 2048 leaves the layer releases, and a hub whose 128000
    neighbours wait for the end of a longer path: x's arcs lie in the share of one or two
    workgroups, so one of them queues at least 1023 of the next layer's 2048 vertices."""
    leaves, wait, lead, tail = 2048, 128_000, 5, 60
    x, hub = lead, lead + 1
    late = hub + 1 + np.arange(tail)            # a path from the start, longer than the lead
    leaf = int(late[-1]) + 1 + np.arange(leaves)
    held = int(leaf[-1]) + 1 + np.arange(wait)
    n = int(held[-1]) + 1
    p = _path(0, lead)
    src = [p[0], [lead - 1, lead - 1, lead - 1], late[:-1], np.full(leaves, x), np.full(wait, hub),
           np.full(wait, late[-1])]
    dst = [p[1], [x, hub, late[0]], late[1:], leaf, held, held]
    _check(_graph(n, np.concatenate(src), np.concatenate(dst)), lead + tail, use_prio)


@pytest.mark.parametrize("width", [1, 31, 32, 33, 64, 1000, 2047, 2048, 2049])
def test_layers_of_a_width(width):
    """Layers of one width, each vertex joined to the one before and after it in its chain."""
    depth = 40
    v = np.arange(width * (depth - 1))
    _check(_graph(width * depth, v, v + width), depth, False)
