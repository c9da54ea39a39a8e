"""Which bins a pull level runs on: levels whose frontier words hold few lanes
bound the thread bin as split levels do, whatever graph they come up on, and no
result depends on it."""
import numpy as np
import pytest

import gpugraph500_amd as g5

pytestmark = pytest.mark.gpu

HITS = 6  # what a thread of the thread bin keeps


def upload(u, v, n):
    keep = u != v
    u, v = u[keep], v[keep]
    k = np.unique(np.concatenate([u * n + v, v * n + u]))
    rowptr = np.concatenate([[0], np.cumsum(np.bincount(k // n, minlength=n))])
    return g5.Graph.upload(rowptr, (k % n).astype(np.uint32), n), np.diff(rowptr)


def regular(n, d, seed):
    """Every vertex has about d neighbours, none of them near."""
    rng = np.random.default_rng(seed)
    return upload(np.tile(np.arange(n), d // 2), np.concatenate([rng.permutation(n) for _ in range(d // 2)]), n)


def ring(n, d, seed):
    """... all of them within 64 d: the search grows for a few levels only."""
    rng = np.random.default_rng(seed)
    u = np.tile(np.arange(n), d // 2)
    return upload(u, (u + rng.integers(1, 64 * d, u.size)) % n, n)


def same_maps(a, b, lanes):
    for lane in lanes:
        for x, y in zip(a.result(lane), b.result(lane)):
            assert np.array_equal(x, y), f"lane {lane}"


@pytest.mark.parametrize("make,n,d,lanes,some", [(regular, 1 << 18, 40, 64, True), (regular, (1 << 18) + 64, 48, 33, True),
                                                (regular, (1 << 18) - 64, 40, 64, False), (ring, 1 << 18, 40, 64, True)])
def test_words_of_few_lanes(make, n, d, lanes, some):
    g, deg = make(n, d, n + d)
    roots = np.random.default_rng(d).choice(n, lanes, replace=False)
    m, push = g5.MSBFS(g), g5.MSBFS(g)
    m.tune(thread_max=256, split_max=32, lane_ratio=0)
    push.set_mode(2)
    push.run(roots)
    m.profile(True)  # the bins one by one, with the neighbours that each reads
    m.run(roots)
    same_maps(m, push, range(0, lanes, 9))
    skew = max(1.0, (deg.astype(float) ** 2).sum() * (deg > 0).sum() / float(deg.sum()) ** 2)
    pairs, last, sparse = lanes, lanes, []
    for rec in m.levels():
        # (every lane is in the frontier until the level that finds nothing)
        few = lanes * rec[10] > HITS * pairs * skew and pairs * pairs > HITS * (deg > 0).sum() * last
        if rec[9] == 0 and rec[8] > 0:
            sparse.append(bool(few and n >= 1 << 18))
            short = (deg <= 32).any()
            assert (rec[5] > 0) == sparse[-1], "neighbours read by the wave bin"
            assert (rec[6] == 0) == (sparse[-1] and not short), "and by the thread bin"
        pairs, last = rec[8], pairs
    assert any(sparse) == some and not all(sparse)
    # the bins together, searches one after the other, and a server's lanes
    m.profile(False)
    for _ in range(2):
        m.run(roots)
        same_maps(m, push, range(0, lanes, 9))
    m.open()
    m.join(roots[:20], list(range(20)))
    m.step()
    m.join(roots[20:lanes], list(range(20, lanes)))
    while m.step()[0]:
        pass
    same_maps(m, push, range(0, lanes, 9))


@pytest.mark.parametrize("n,d", [(1 << 17, 56), (1 << 17, 72), (1 << 16, 130), ((1 << 17) + 128, 64)])
def test_wave_bins_of_most_vertices(n, d):
    """Below and beyond 2^23 stored neighbours: in a launch with the other bins,
    and in one of their own."""
    g, deg = regular(n, d, n + d)
    m, push = g5.MSBFS(g), g5.MSBFS(g)
    m.tune(thread_max=32, split_max=16)
    assert m.bins()[1] > m.bins()[2] and g.nnz < 1 << 24
    push.set_mode(2)
    roots = np.random.default_rng(n).choice(n, 50, replace=False)
    push.run(roots)
    for mode in (1, 0, 0):
        m.set_mode(mode)
        m.run(roots)
        same_maps(m, push, range(0, 50, 7))
        assert m.nedge().tolist() == push.nedge().tolist()


@pytest.mark.parametrize("n,left,whole", [(1 << 18, 1, False), (1 << 18, 0, True), ((1 << 18) + 64, 21, True),
                                          ((1 << 18) + 1024, 21, True), (1 << 19, 5, True)])
def test_thread_bin_in_whole_words(n, left, whole):
    """Thread bins of 2^18 vertices and more in a launch with the other bins, the
    last word full or not; `left` ids have no edge."""
    rng = np.random.default_rng(n + left)
    v = rng.permutation(n)[left:]
    far = rng.integers(0, len(v), (2, n // 3))
    # some rows for the other bins, which end at a multiple of 64
    hubs = v[rng.integers(0, 40, 20000 if n > (1 << 18) + 64 else 0)]
    g, deg = upload(np.concatenate([v, v[far[0]], hubs]),
                    np.concatenate([np.roll(v, 1), v[far[1]], v[rng.integers(0, len(v), len(hubs))]]), n)
    m, push = g5.MSBFS(g), g5.MSBFS(g)
    m.tune(wave_max=400)
    assert (m.bins()[2] >= 1 << 18) == whole
    push.set_mode(2)
    roots = [int(v[i]) for i in rng.integers(0, len(v), 40)]
    push.run(roots)
    for mode in (1, 0, 1):
        m.set_mode(mode)
        m.run(roots)
        same_maps(m, push, range(0, 40, 6))
        assert m.nedge().tolist() == push.nedge().tolist()
