"""Maps and bitmaps that do not lie in one allocation of the engine's GPU: in
host memory they give the same results, and a buffer that ends before them is
refused, as a copy refuses it."""
import ctypes

import numpy as np
import pytest

import gpugraph500_amd as g5
import oracle_lib as O

pytestmark = pytest.mark.gpu


class Host:
    """Host memory as the bindings take a device buffer."""

    def __init__(self, a):
        self.a = a
        self.ptr = ctypes.c_void_p(a.ctypes.data)


@pytest.fixture(scope="module")
def graph():
    ref = O.build_csr(O.kronecker_edges(13))
    root = int(O.select_roots(ref, 1 << 13)[0])
    return ref, g5.Graph.kronecker(13), root, O.bfs_bin(ref, root)


@pytest.mark.parametrize("uploaded", [False, True])
def test_validated_map_in_host_memory(graph, uploaded):
    ref, g, root, (pred, lev, _) = graph
    if uploaded:
        g = g5.Graph.upload(ref.rowptr, ref.cols, ref.n_rows, gdeg=ref.gdeg)
    v = g5.Validator(g)
    bad = pred.copy()
    bad[np.flatnonzero(lev == 2)[0]] = root
    for p in (pred, bad):
        want = v.validate(root, p, want_depth=True)
        got = v.validate_device(root, Host(p), want_depth=True)
        assert got[:2] == want[:2] and np.array_equal(got[2], want[2])


def test_validated_map_at_an_odd_address(graph):
    ref, g, root, (pred, _, _) = graph
    raw = np.zeros(pred.nbytes + 8, np.uint8)
    raw[4:4 + pred.nbytes] = pred.view(np.uint8)
    d = g5.DeviceArray.from_host(raw)
    at = Host(raw)  # only its place on the device counts
    at.ptr = ctypes.c_void_p(d.ptr.value + 4)
    assert g5.Validator(g).validate_device(root, at)[:2] == g5.Validator(g).validate(root, pred)[:2]


def test_short_buffers_are_refused(graph):
    """... and the error is gone with the call that reported it."""
    ref, g, root, (pred, _, _) = graph
    short = g5.DeviceArray.from_host(pred[:-64])
    v = g5.Validator(g)
    with pytest.raises(g5.G5Error):
        v.validate_device(root, short)
    assert v.validate_device(root, g5.DeviceArray.from_host(pred))[0] == 0
    b, lib = g5.BFS(g), g5.lib()
    bits = g5.DeviceArray.from_host(np.zeros(ref.n_rows // 128, np.uint64))
    b.start(root)
    assert lib.g5_bfs_set_out_bitmap(b.h, bits.ptr) != 0
    assert lib.g5_bfs_set_in_bitmap(b.h, bits.ptr) != 0


@pytest.mark.parametrize("where", ["device", "host"])
def test_a_search_by_bitmaps(graph, where):
    ref, g, root, (pred, lev, nlevels) = graph
    b, lib = g5.BFS(g), g5.lib()
    b.start(root)
    for depth in range(1, nlevels + 1):
        assert b.expand() == (depth < nlevels)
        bits = np.packbits(lev == depth, bitorder="little").view(np.uint64).copy()
        x = g5.DeviceArray.from_host(bits) if where == "device" else Host(bits)
        if depth % 2:
            g5.check(lib.g5_bfs_set_out_bitmap(b.h, x.ptr))
        else:
            g5.check(lib.g5_bfs_set_out_bitmap(b.h, None))
        g5.check(lib.g5_bfs_set_in_bitmap(b.h, x.ptr))
    p, l = b.result()
    assert np.array_equal(p, pred) and np.array_equal(l, lev)
