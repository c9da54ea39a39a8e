"""The single-root engine on a grid's blocks: g5_bfs_run on the diagonal ones,
whose rows need not start at vertex 0, and the memory that the hooks take."""
import ctypes

import numpy as np
import pytest

import gpugraph500_amd as g5

pytestmark = pytest.mark.gpu

PARTS = 2


@pytest.fixture(scope="module")
def blocks():
    return g5.Graph.kronecker_2d(14, PARTS, PARTS)


@pytest.mark.parametrize("how", [{}, {"codec": True}, {"topdown": True}, "profile"])
def test_root_outside_the_block(blocks, how):
    """An accepted root (below the block's rows) that is not one of its vertices
    reaches nothing."""
    b = blocks[3]
    start = g5.block_bounds(b.nglobal, PARTS, PARTS, 1, 1)[0]
    assert start >= b.n_rows > 4000
    e = g5.BFS(b)
    if how == "profile":
        e.profile(True)
        how = {}
    for root in (0, 1, 4000, b.n_rows - 1):
        assert e.run(root, **how)[0] == 1
        pred, lev = e.result()
        assert (pred == -1).all() and (lev == -1).all() and e.nedge() == 0
    with pytest.raises(g5.G5Error):
        e.run(start)


def test_root_of_the_first_block(blocks):
    b = blocks[0]
    rowptr = b.download()[0]
    a, h = g5.BFS(b), g5.BFS(b)
    a.start(0)  # a handle that the hooks have used
    a.expand()
    for root in np.flatnonzero(np.diff(rowptr))[[0, 5, -1]].tolist():
        assert a.run(root)[0] == h.run(root, topdown=True)[0] > 1
        for x, y in zip(a.result(), h.result()):
            assert np.array_equal(x, y)


def free_bytes():
    free, total = ctypes.c_int64(), ctypes.c_int64()
    g5.check(g5.lib().g5_mem_info(ctypes.byref(free), ctypes.byref(total)))
    return free.value


def test_diagonal_blocks_take_what_the_others_take():
    """The buffers of a whole search (6 bytes a vertex, 25 MB an engine here) come
    with the first one."""
    took = []
    for b in g5.Graph.kronecker_2d(23, PARTS, PARTS):
        before = free_bytes()
        engines = [g5.BFS(b) for _ in range(4)]
        took.append(before - free_bytes())
        for e in engines:
            e.free()
    assert max(took[0], took[3]) <= max(took[1], took[2]) + (16 << 20), took
