"""The passes that sum over a lane's reached vertices (g5_msbfs_nedge and
g5_msbfs_leave) where neighbouring vertices carry different lane sets: many
small components, so that a wave meets up to 64 distinct words, degrees whose
sums pass 32 bits, and every way of splitting a wave over the leaving lanes."""
import numpy as np
import pytest

import gpugraph500_amd as g5
import oracle_lib as O
from test_gpu_continuous import checksum

pytestmark = pytest.mark.gpu


def rings(n, sizes, seed):
    """n vertices in rings of the given sizes (repeated until n is full, the
    rest edgeless), ids shuffled; gdeg up to 2^32 - 1."""
    rng = np.random.default_rng(seed)
    ids = rng.permutation(n)
    adj = [[] for _ in range(n)]
    at, i = 0, 0
    comps = []
    while at + sizes[i % len(sizes)] <= n:
        c = ids[at:at + sizes[i % len(sizes)]]
        at += len(c)
        i += 1
        comps.append(c)
        for a, b in zip(c, np.roll(c, 1)):
            if a != b:
                adj[a].append(b)
                adj[b].append(a)
    rows = [np.unique(np.array(a, np.int64)) for a in adj]
    rowptr = np.concatenate([[0], np.cumsum([len(r) for r in rows])])
    cols = np.concatenate(rows).astype(np.uint32)
    gdeg = rng.integers(1, 1 << 32, n, dtype=np.int64)
    gdeg[rng.random(n) < 0.1] = 0
    return rowptr, cols, gdeg, comps


@pytest.mark.parametrize("n,sizes,lanes", [(64, (2,), 32), (64, (3, 5), 1), (320, (7, 2, 11), 64),
                                           (4096, (50, 64, 3), 33), (70016, (1000, 1500), 64), (70016, (70000,), 5)])
def test_sums_over_small_components(n, sizes, lanes):
    rowptr, cols, gdeg, comps = rings(n, sizes, n + lanes)
    g = g5.Graph.upload(rowptr, cols, n, gdeg=gdeg)
    m = g5.MSBFS(g)
    rng = np.random.default_rng(1)
    roots = [int(comps[i % len(comps)][rng.integers(len(comps[i % len(comps)]))]) for i in range(lanes)]
    member = {int(v): i for i, c in enumerate(comps) for v in c}
    want = [int(gdeg[comps[member[r]]].astype(object).sum()) // 2 for r in roots]
    m.run(roots)
    assert m.nedge().tolist() == want

    # the same lanes in continuous mode, leaving in groups of 1, 2, 3, 5, ...
    m.open()
    m.join(roots, list(range(lanes)))
    for _ in range(40000):
        live, _ = m.step()
        if not live:
            break
    preds = [m.result(lane)[0] for lane in range(lanes)] if n <= 4096 else None
    left = list(rng.permutation(lanes))
    for k in (1, 2, 3, 5, 17, 64):
        group, left = left[:k], left[k:]
        if not group:
            break
        ne, ck = m.leave(sum(1 << int(x) for x in group))
        for x in group:
            assert int(ne[x]) == want[x], f"lane {x}"
            if preds is not None:
                assert int(ck[x]) == checksum(preds[x]), f"lane {x}"


def test_leaving_lanes_match_the_oracle():
    ref = O.build_csr(O.kronecker_edges(11))
    g = g5.Graph.upload(ref.rowptr, ref.cols, ref.n_rows, gdeg=ref.gdeg)
    m = g5.MSBFS(g)
    roots = [int(r) for r in O.select_roots(ref, 1 << 11)][:64]
    for k in (1, 2, 4, 7, 9, 16, 31, 32, 64):
        m.open()
        lanes = [(5 * i + 3) % 64 for i in range(k)]  # spread over the word
        m.join(roots[:k], lanes)
        while m.step()[0]:
            pass
        ne, ck = m.leave(sum(1 << x for x in lanes))
        for r, x in zip(roots, lanes):
            pred, lev, _ = O.bfs_bin(ref, r)
            assert int(ne[x]) == O.nedge(ref, lev) and int(ck[x]) == checksum(pred)


@pytest.mark.parametrize("scale, edgefactor, thread, split", [(11, 16, 32, 16), (16, 16, 64, 32),
                                                             (18, 16, 256, 32)])
def test_thread_bound_follows_a_smaller_wave_bound_until_it_is_set(scale, edgefactor, thread, split):
    g = g5.Graph.kronecker(scale, edgefactor)
    m = g5.MSBFS(g)
    d = m.get_tune()
    assert (d["thread_max"], d["wave_max"], d["split_max"]) == (thread, 2048, split)
    roots = [int(r) for r in g.select_roots(g.nglobal, 20)]
    m.run(roots)
    want = [m.result(lane) for lane in range(20)]

    def check():
        m.run(roots)
        for lane in range(20):
            pred, lev = m.result(lane)
            assert np.array_equal(pred, want[lane][0]) and np.array_equal(lev, want[lane][1])

    for wave in (64, 32, 300, 100):
        m.tune(wave_max=wave)
        assert m.get_tune()["thread_max"] == min(thread, wave) and m.get_tune()["wave_max"] == wave
        check()
    with pytest.raises(g5.G5Error):
        m.tune(wave_max=31)
    m.tune(thread_max=8)
    m.tune(wave_max=16)
    assert m.get_tune()["thread_max"] == 8
    check()
    with pytest.raises(g5.G5Error):
        m.tune(wave_max=7)


@pytest.mark.parametrize("sources, targets", [(3, 64), (40, 1000), (700, 3000), (2000, 40)])
def test_push_levels_keep_the_smallest_parent(sources, targets):
    """Every target has several parents at one level: the edges that find a pair
    set are looked at again, in tiles of few and of many sources."""
    rng = np.random.default_rng(sources)
    n = 1 + sources + targets
    e = [np.stack([np.zeros(sources, np.int64), 1 + np.arange(sources)], 1)]
    for _ in range(5):
        t = 1 + sources + np.arange(targets)
        e.append(np.stack([1 + rng.integers(0, sources, targets), t], 1))
    s = 1 + np.arange(sources)
    e.append(np.stack([s, 1 + sources + rng.integers(0, targets, sources)], 1))
    ref = O.build_csr(rng.permutation(n)[np.concatenate(e)])
    g = g5.Graph.upload(ref.rowptr, ref.cols, ref.n_rows, gdeg=ref.gdeg)
    m = g5.MSBFS(g)
    m.set_mode(2)
    roots = [int(r) for r in rng.choice(n, min(n, 64), replace=False)]
    for _ in range(2):
        m.run(roots)
        for lane in range(0, len(roots), 5):
            pred, lev = m.result(lane)
            opred, olev, _ = O.bfs_bin(ref, roots[lane])
            assert np.array_equal(pred, opred) and np.array_equal(lev, olev)


@pytest.mark.parametrize("shape", [dict(thread_max=0, wave_max=0), dict(thread_max=0, wave_max=1 << 20),
                                   dict(thread_max=1 << 20, wave_max=1 << 20), dict(thread_max=9, wave_max=40),
                                   dict(thread_max=9, wave_max=1 << 20), dict(thread_max=40, wave_max=40)])
def test_bins_in_one_launch_and_in_three(shape):
    """Pull levels with any of the bins empty; accounting runs them one by one."""
    ref = O.build_csr(O.kronecker_edges(12))
    g = g5.Graph.upload(ref.rowptr, ref.cols, ref.n_rows, gdeg=ref.gdeg)
    m = g5.MSBFS(g)
    m.tune(**shape)
    m.set_mode(1)
    roots = [int(r) for r in O.select_roots(ref, 1 << 12)][:40]
    want = [O.bfs_bin(ref, r)[:2] for r in roots]
    for prof in (False, True, False):
        m.profile(prof)
        m.run(roots)
        for lane in range(0, len(roots), 3):
            pred, lev = m.result(lane)
            assert np.array_equal(pred, want[lane][0]) and np.array_equal(lev, want[lane][1])


@pytest.mark.parametrize("mode", [0, 1, 2])
def test_graph_without_edges(mode):
    n = 128
    g = g5.Graph.upload(np.zeros(n + 1, np.int64), np.zeros(0, np.uint32), n, gdeg=np.zeros(n, np.int64))
    m = g5.MSBFS(g)
    m.set_mode(mode)
    for prof in (False, True):
        m.profile(prof)
        m.run([0, 5, 127])
        for lane, r in enumerate((0, 5, 127)):
            pred, lev = m.result(lane)
            assert pred[r] == r and lev[r] == 0 and (np.delete(pred, r) == -1).all()


@pytest.mark.parametrize("n", [64, 128, 1 << 12, (1 << 18) - 64, 1 << 18])
def test_thread_bin_in_quarters_of_words(n):
    """Rings and pairs over all ids: every vertex in the thread bin, up to the
    size where a wave takes whole words, partly filled words at its end."""
    rng = np.random.default_rng(n)
    v = rng.permutation(n)[:n - 21]
    e = np.stack([v, np.roll(v, 1)], 1)
    far = rng.integers(0, len(v), (n // 3, 2))
    e = np.concatenate([e, v[far[far[:, 0] != far[:, 1]]]])
    e = e[np.lexsort((e[:, 1], e[:, 0]))]
    both = np.unique(np.concatenate([e, e[:, ::-1]]), axis=0)
    both = both[both[:, 0] != both[:, 1]]
    rowptr = np.concatenate([[0], np.cumsum(np.bincount(both[:, 0], minlength=n))])
    g = g5.Graph.upload(rowptr, both[:, 1].astype(np.uint32), n, gdeg=np.diff(rowptr))
    roots = [int(v[i]) for i in rng.integers(0, len(v), 40)]
    a, b = g5.MSBFS(g), g5.MSBFS(g)
    a.set_mode(1)
    b.set_mode(2)  # push only: no pull kernels
    for _ in range(2):
        a.run(roots)
        b.run(roots)
        for lane in range(0, 40, 6):
            for x, y in zip(a.result(lane), b.result(lane)):
                assert np.array_equal(x, y)
    assert a.nedge().tolist() == b.nedge().tolist()


@pytest.mark.parametrize("n", [640, 4096, 40000])
def test_push_levels_with_and_without_a_bitmap_of_marks(n):
    """Push only: a few sources, then nearly all vertices at once (more edges
    than n / 8 after a push level), then their neighbours."""
    rng = np.random.default_rng(n)
    k = n // 2
    e = np.concatenate([np.stack([rng.integers(0, 4, k), 4 + np.arange(k)], 1),
                        np.stack([4 + rng.integers(0, k, n - 4 - k), np.arange(4 + k, n)], 1),
                        np.stack([np.arange(3), np.arange(1, 4)], 1)])
    ref = O.build_csr(rng.permutation(n)[e])
    g = g5.Graph.upload(ref.rowptr, ref.cols, ref.n_rows, gdeg=ref.gdeg)
    m = g5.MSBFS(g)
    m.set_mode(2)
    roots = [int(r) for r in rng.choice(n, 64, replace=False)]
    for _ in range(2):
        m.run(roots)
        for lane in range(0, 64, 7):
            pred, lev = m.result(lane)
            opred, olev, _ = O.bfs_bin(ref, roots[lane])
            assert np.array_equal(pred, opred) and np.array_equal(lev, olev)
