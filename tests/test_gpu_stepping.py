"""Bitmaps to queues and back at the edges of tiles, waves and words, and the
level steps of the hooks and of the host-driven search on them: what a step
leaves must not depend on the form its frontier came in."""
import ctypes

import numpy as np
import pytest

import gpugraph500_amd as g5
import oracle_lib as O

pytestmark = pytest.mark.gpu

TILES = 1024  # workgroups of a pass over a bitmap, 64 words or more each


def bits_of(v, words):
    b = np.zeros(words * 64, np.uint8)
    b[v] = 1
    return np.packbits(b, bitorder="little").view(np.uint64)


@pytest.mark.parametrize("words", [1, 15, 16, 17, 63, 64, 65, 200, 64 * TILES - 1, 64 * TILES, 64 * TILES + 1,
                                   128 * TILES + 65])
@pytest.mark.parametrize("density", [0.0, 0.002, 0.6, 1.0])
def test_bitmap_and_queue(words, density):
    rng = np.random.default_rng(words)
    n = words * 64
    v = np.flatnonzero(rng.random(n) < density) if density < 1 else np.arange(n)
    if density == 0:
        v = np.array([n - 1])  # the last vertex alone
    bits = g5.DeviceArray.from_host(bits_of(v, words))
    q = g5.DeviceArray(n, np.uint32)
    cnt, lib = ctypes.c_int64(-1), g5.lib()
    assert g5.bitmap_count(bits, words) == len(v)
    g5.check(lib.g5_bitmap_to_queue(bits.ptr, words, q.ptr, ctypes.byref(cnt)))
    assert cnt.value == len(v)
    assert np.array_equal(q.to_host()[:len(v)], v)
    # back: in order, and in any order with repeats
    for ids in (v, rng.permutation(np.concatenate([v, v[:len(v) // 3 + 1]]))):
        d = g5.DeviceArray.from_host(ids.astype(np.uint32))
        back = g5.DeviceArray.from_host(np.full(words, ~np.uint64(0)))
        g5.check(lib.g5_queue_to_bitmap(d.ptr, len(ids), back.ptr, words))
        assert np.array_equal(back.to_host(), bits_of(v, words))
    # ids beyond the words are refused and counted
    ids = np.concatenate([v[:50], [n, n + 64, 2**32 - 1]]).astype(np.uint32)
    d = g5.DeviceArray.from_host(ids)
    with pytest.raises(g5.G5Error, match="3 ids beyond"):
        g5.check(lib.g5_queue_to_bitmap(d.ptr, len(ids), bits.ptr, words))
    assert np.array_equal(bits.to_host(), bits_of(v[:50], words))


def test_empty_bitmap_and_queue():
    cnt, lib = ctypes.c_int64(7), g5.lib()
    g5.check(lib.g5_bitmap_to_queue(None, 0, None, ctypes.byref(cnt)))
    assert cnt.value == 0 and g5.bitmap_count(g5.DeviceArray(1, np.uint64), 0) == 0
    bits = g5.DeviceArray.from_host(np.full(3, ~np.uint64(0)))
    g5.check(lib.g5_queue_to_bitmap(None, 0, bits.ptr, 3))
    assert not bits.to_host().any()


def graph(kind):
    if kind == "kronecker":
        ref = O.build_csr(O.kronecker_edges(13))
    else:  # hubs with leaves, hubs on a path: few sources with many edges, and the reverse
        c = np.arange(1, 9000)
        ref = O.build_csr(np.concatenate([np.stack([c // 1500 * 1500, c], 1), np.stack([c - 1, c], 1)[::7]]))
    return ref, g5.Graph.upload(ref.rowptr, ref.cols, ref.n_rows, gdeg=ref.gdeg)


@pytest.mark.parametrize("kind", ["kronecker", "hubs"])
@pytest.mark.parametrize("form", ["own", "queue", "bitmap", "bottom_up", "mixed"])
def test_a_step_does_not_depend_on_the_form_of_its_frontier(kind, form):
    ref, g = graph(kind)
    b = g5.BFS(g)
    root = int(O.select_roots(ref, ref.n_rows)[0]) if kind == "kronecker" else 1501
    opred, olev, _ = O.bfs_bin(ref, root)
    lib, words = g5.lib(), g.n_cols // 64
    for turn in range(2):  # the second search starts from what the first left
        b.start(root)
        depth = 0
        while True:
            want = np.flatnonzero(olev == depth + 1)
            bu = depth > 0 and (form == "bottom_up" or (form == "mixed" and depth % 2 == 1))
            assert (b.expand_bottom_up(g) if bu else b.expand()) == (len(want) > 0)
            assert np.array_equal(b.outqueue(), want)
            if not len(want):
                break
            if form == "queue":
                b.set_outqueue(want)
                b.set_inqueue(want)
            elif form == "own":
                b.set_outqueue()
                b.set_inqueue()
            else:
                # vertices reached before are given again, and must be dropped
                again = bits_of(np.flatnonzero((olev >= 0) & (olev <= depth + 1)), words)
                d = g5.DeviceArray.from_host(again if turn else bits_of(want, words))
                g5.check(lib.g5_bfs_set_out_bitmap(b.h, d.ptr))
                assert np.array_equal(b.outqueue(), want)
                p, nw = ctypes.c_void_p(), ctypes.c_int64()
                g5.check(lib.g5_bfs_out_bitmap(b.h, ctypes.byref(p), ctypes.byref(nw)))
                g5.check(lib.g5_bfs_set_in_bitmap(b.h, p))
            depth += 1
        pred, lev = b.result()
        assert np.array_equal(pred, opred) and np.array_equal(lev, olev)


@pytest.mark.parametrize("kind", ["kronecker", "hubs"])
@pytest.mark.parametrize("alpha, beta", [(20, 24), (1 << 40, 1), (1, 1 << 40), (2, 2)])
def test_host_driven_search(kind, alpha, beta):
    ref, g = graph(kind)
    b = g5.BFS(g)
    b.tune(alpha, beta)
    for root in (0, 1, int(ref.n_rows - 64)):
        opred, olev, _ = O.bfs_bin(ref, root)
        for kw in (dict(codec=True), dict(topdown=True), dict(codec=True, topdown=True)):
            nl, _ = b.run(root, **kw)
            pred, lev = b.result()
            assert nl == olev.max() + 1
            assert np.array_equal(pred, opred) and np.array_equal(lev, olev)
            assert not b.expand()  # nothing is left to expand
