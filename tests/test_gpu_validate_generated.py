"""Validation of generated graphs, whose edges are checked once each and whose
parent edges are counted: every map gets the oracle's flags, count and depths,
and those that the same graph gets when it is uploaded."""
import numpy as np
import pytest

import gpugraph500_amd as g5
import oracle_lib as O
from test_gpu_validate import mutations, same_as_oracle

pytestmark = pytest.mark.gpu


def dfs_tree(ref, root):
    """A depth-first tree: every parent edge is there, the depths run deep."""
    pred = np.full(ref.n_rows, -1, np.int64)
    pred[root] = root
    stack = [(root, iter(ref.cols[ref.rowptr[root]:ref.rowptr[root + 1]].tolist()))]
    while stack:
        v, it = stack[-1]
        for u in it:
            if pred[u] < 0:
                pred[u] = v
                stack.append((u, iter(ref.cols[ref.rowptr[u]:ref.rowptr[u + 1]].tolist())))
                break
        else:
            stack.pop()
    return pred


# scale 1-5: rows and edges below one wave's window and step; edgefactor 1:
# windows of mostly empty rows; 200: rows of thousands of neighbours; 15 / 16:
# several shares per wave, hub rows longer than a share
@pytest.mark.parametrize("scale,ef", [(1, 1), (5, 16), (6, 1), (8, 3), (9, 200), (13, 1), (15, 16), (16, 5)])
def test_generated_graph_flags(scale, ef):
    e = O.kronecker_edges(scale, ef)
    ref = O.build_csr(e)
    if ref.nnz == 0:
        pytest.skip("no edges")
    g = g5.Graph.kronecker(scale, ef)
    up = g5.Graph.upload(ref.rowptr, ref.cols, ref.n_rows, gdeg=ref.gdeg)
    val, val_up = g5.Validator(g), g5.Validator(up)
    root = int(np.argmax(np.diff(ref.rowptr)))
    pred, lev, _ = O.bfs_bin(ref, root)
    assert same_as_oracle(e, ref, val, root, pred) == 0
    maps = [("depth-first", dfs_tree(ref, root))]
    rng = np.random.default_rng(scale)
    if (lev == 1).sum() > 1 and (lev == 2).sum() > 1:
        maps += mutations(ref, root, pred, lev, rng)
    # one vertex at a time: the last row with neighbours, the last neighbour's
    # side of an edge, a leaf that names itself
    rows = np.flatnonzero(np.diff(ref.rowptr))
    for v in (int(rows[-1]), int(rows[0]), int(rows[len(rows) // 2])):
        if v == root:
            continue
        for p in (v, -1, int(ref.cols[ref.rowptr[v + 1] - 1])):
            q = pred.copy()
            q[v] = p
            maps.append((f"parent({v}) = {p}", q))
    for name, p in maps:
        bad = same_as_oracle(e, ref, val, root, p)
        assert bad == same_as_oracle(e, ref, val_up, root, p), name
