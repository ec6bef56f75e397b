"""Tree passes over slots of children: runs of children with and without children of their own that
end inside, at and past a workgroup's tile of 256 slots, with a hole (an arc into the root)."""
import numpy as np
import pytest
import orc
import smdp

pytestmark = pytest.mark.gpu


def _check(ctx, kids, root=0):
    row = np.zeros(len(kids) + 1, np.int32)
    row[1:] = np.cumsum([len(k) for k in kids])
    g = smdp.HostGraph(row, np.array([c for k in kids for c in k], np.int32))
    with smdp.Graph(ctx, g) as dg:
        for _ in range(2):  # the second run finds the first one's buffers
            dg.tree(root)
            rh, rd, _ = orc.tree(g.row, g.col, root)
            assert np.array_equal(dg.read(smdp.RES_HEIGHT), rh) and np.array_equal(dg.read(smdp.RES_DESC), rd)


@pytest.mark.parametrize("hole", [False, True])
@pytest.mark.parametrize("inner", [1, 255, 256, 257, 1023, 1024, 1025, 70000])
def test_inner_children(ctx, inner, hole):
    """The root has `inner` children with 0 to 3 leaves and one or no child that has one, and 5 leaves."""
    kids = [[]]
    r = np.random.RandomState(inner)

    def add(parent):
        kids.append([])
        kids[parent].append(len(kids) - 1)
        return len(kids) - 1

    for _ in range(inner):
        u = add(0)
        for _ in range(r.randint(0, 4)):
            add(u)
        if r.randint(0, 2) or not kids[u]:
            add(add(u))
    for _ in range(5):
        add(0)
    if hole:
        kids[1 + r.randint(0, len(kids) - 1)].append(0)
    for k in kids:
        r.shuffle(k)
    _check(ctx, kids)
