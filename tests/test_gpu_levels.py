"""g5_bfs_run's levels on the device: levels, parents and the level count equal
the oracle's and the host-driven search's (topdown=True) on graphs that reach
the edges of its tiles, queues and buffers, with the direction switch at both
ends."""
import numpy as np
import pytest

import gpugraph500_amd as g5
import oracle_lib as O

pytestmark = pytest.mark.gpu


def path(n):
    return np.stack([np.arange(n - 1), np.arange(1, n)], 1)


def star(n):  # one vertex of many tiles' edges, then leaves of one edge
    return np.stack([np.zeros(n - 1, np.int64), np.arange(1, n)], 1)


def tree(n, k):  # k children each: frontiers of many sources with few edges
    c = np.arange(1, n)
    return np.stack([(c - 1) // k, c], 1)


def comb(n):  # hubs on a path, each with its own leaves: top-down after bottom-up and back
    hubs = np.arange(0, n, 500)
    leaves = np.setdiff1d(np.arange(n), hubs)
    return np.concatenate([np.stack([hubs[:-1], hubs[1:]], 1), np.stack([leaves // 500 * 500, leaves], 1)])


def matching(n):  # components of two
    return np.arange(n // 2 * 2).reshape(-1, 2)


def shuffled(e, seed):
    p = np.random.default_rng(seed).permutation(int(e.max()) + 1)
    return p[e]


GRAPHS = {
    "path": lambda: path(2500),
    "star64": lambda: star(64),
    "star": lambda: star(70001),
    "binary tree": lambda: tree(100000, 2),
    "unary steps": lambda: tree(5000, 1),
    "wide tree": lambda: tree(300000, 37),
    "comb": lambda: comb(40000),
    "matching": lambda: matching(3000),
    "dense": lambda: np.argwhere(np.triu(np.ones((700, 700), bool), 1)),
    "random": lambda: np.random.default_rng(3).integers(0, 150000, (400000, 2)),
    "sparse random": lambda: np.random.default_rng(4).integers(0, 200000, (140000, 2)),
}


@pytest.mark.parametrize("name", sorted(GRAPHS))
def test_levels_on_the_device(name):
    e = shuffled(GRAPHS[name]().astype(np.int64), 1)
    ref = O.build_csr(e)
    g = g5.Graph.upload(ref.rowptr, ref.cols, ref.n_rows, gdeg=ref.gdeg)
    deg = np.diff(ref.rowptr)
    rng = np.random.default_rng(2)
    roots = {int(np.argmax(deg)), int(np.flatnonzero(deg)[0]), int(rng.choice(np.flatnonzero(deg)))}
    if (deg == 0).any():
        roots.add(int(np.flatnonzero(deg == 0)[0]))
    b = g5.BFS(g)
    for root in sorted(roots):
        pred, lev, nl = O.bfs_bin(ref, root)
        b.tune()
        assert b.run(root, topdown=True)[0] == nl
        for alpha, beta in ((20, 24), (1, 1 << 40), (1 << 40, 1), (3, 3)):
            b.tune(alpha, beta)
            assert b.run(root)[0] == nl, (root, alpha, beta)
            p, lv = b.result()
            assert np.array_equal(lv, lev), (root, alpha, beta)
            assert np.array_equal(p, pred), (root, alpha, beta)
            assert b.nedge() == O.nedge(ref, lev)
        assert not b.expand() and len(b.outqueue()) == 0  # nothing left to expand


@pytest.mark.parametrize("scale,ef", [(17, 1), (17, 40), (19, 7), (20, 16)])
def test_against_the_host_driven_search(scale, ef):
    g = g5.Graph.kronecker(scale, ef)
    a, b = g5.BFS(g), g5.BFS(g)
    for root in g.select_roots(g.nglobal)[:6].tolist():
        for alpha in (20, 2, 300):
            a.tune(alpha)
            na, nb = a.run(root)[0], b.run(root, topdown=True)[0]
            assert na == nb
            (pa, la), (pb, lb) = a.result(), b.result()
            assert np.array_equal(pa, pb) and np.array_equal(la, lb), (root, alpha)
