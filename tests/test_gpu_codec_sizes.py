"""The codec at the sizes where its launches change: one workgroup up to 8192
values, tiles of 64 miniblocks, two tiles per workgroup past 1024 tiles, one
more table of header hops at 128, 1024 and 8192 groups.  Streams are the
oracle encoder's word for word, values come back, and what is no stream of at
most the capacity's values is refused as before."""
import ctypes

import numpy as np
import pytest

import gpugraph500_amd as g5
import oracle_lib as O

pytestmark = pytest.mark.gpu


def kinds(n, seed):
    rng = np.random.default_rng(seed)
    yield "queue", (np.cumsum(rng.integers(1, 200, n)) - 1).astype(np.uint32)
    # widths 0..32 side by side, so that resets (raw miniblocks) sit anywhere
    width = rng.integers(0, 33, n // 128 + 1).repeat(128)[:n]
    step = rng.integers(0, 1 << 32, n, dtype=np.uint64) & ((np.uint64(1) << width.astype(np.uint64)) - np.uint64(1))
    x = np.zeros((n + 3) // 4 * 4, np.uint64)
    x[:n] = step
    yield "mixed", (np.cumsum(x.reshape(-1, 4), axis=0, dtype=np.uint64).reshape(-1)[:n] % (1 << 32)).astype(np.uint32)
    yield "same", np.full(n, 12345678, np.uint32)


@pytest.mark.parametrize("n", [1, 127, 128, 8064 + 127, 8192, 8193, 8192 + 128, 16384, 16384 + 127, 128 * 2048,
                               129 * 2048 + 1, 1024 * 2048 + 5, 1025 * 2048, 3000001])
def test_streams_and_values(n):
    for name, x in kinds(n, n):
        w = g5.s4_encode(x)
        assert np.array_equal(w, O.s4_encode(x)), (name, n)
        assert np.array_equal(g5.s4_decode(w, n), x), (name, n)
        back, nw = g5.s4_roundtrip(x)
        assert nw == len(w) and np.array_equal(back, x), (name, n)


def test_past_the_largest_grid():
    n = 1024 * 8192 + 64 * 128 + 77  # 1025 tiles: two per workgroup
    for name, x in kinds(n, 3):
        w = g5.s4_encode(x)
        assert np.array_equal(w, O.s4_encode(x)), name
        assert np.array_equal(g5.s4_decode(w, n), x), name


@pytest.mark.parametrize("n", [3000, 8192, 100000])
def test_capacity_and_alignment(n):
    """A capacity above the stream's values, and a stream on any word."""
    x = next(kinds(n, n))[1]
    w = O.s4_encode(x)
    assert np.array_equal(g5.s4_decode(w, 50 * n), x)
    L = g5.lib()
    for off in (1, 2, 3):
        din = g5.DeviceArray.from_host(np.concatenate([np.zeros(off, np.uint32), w]))
        dout = g5.DeviceArray(n + off, np.uint32)
        got = g5.c_sz()
        g5.check(L.g5_s4_decode(ctypes.c_void_p(din.ptr.value + 4 * off), len(w),
                                ctypes.c_void_p(dout.ptr.value + 4 * off), n, ctypes.byref(got)))
        assert got.value == n and np.array_equal(dout.to_host()[off:], x)


def test_few_words_of_many_miniblocks():
    """A short stream that holds more miniblocks than one workgroup takes."""
    for n in (8192 + 128, 128 * 2048 * 3 + 9):
        x = np.full(n, 7, np.uint32)
        x[4:] = x[0]
        w = O.s4_encode(x)
        assert len(w) < 8000
        assert np.array_equal(g5.s4_decode(w, n), x)
        with pytest.raises(g5.G5Error):
            g5.s4_decode(w, n - 1)
        with pytest.raises(g5.G5Error):
            g5.s4_decode(w[:len(w) // 2], n)


def varints(vals):
    """The tail's bytes of deltas `vals`, padded to words (test helper)."""
    out = bytearray()
    for v in vals:
        v = int(v)
        while v >= 128:
            out.append(v & 127)
            v >>= 7
        out.append(v | 128)
    out += bytes(-len(out) % 4)
    return np.frombuffer(bytes(out), np.uint32)


@pytest.mark.parametrize("blocks", [0, 3, 70])
def test_tails_of_any_length(blocks):
    """A stream may end in more varints than an encoder writes."""
    rng = np.random.default_rng(blocks)
    head = O.s4_encode(np.arange(128 * blocks, dtype=np.uint32) * 5)
    for k in (0, 1, 63, 64, 65, 127, 128, 1000, 20000):
        d = rng.integers(0, 1 << rng.integers(1, 32), k, dtype=np.uint64)
        w = np.concatenate([head, varints(d)]).astype(np.uint32)
        want = np.concatenate([np.arange(128 * blocks, dtype=np.uint32) * 5,
                               (np.cumsum(d, dtype=np.uint64) % (1 << 32)).astype(np.uint32)])
        assert np.array_equal(g5.s4_decode(w, len(want)), want), k
        assert np.array_equal(g5.s4_decode(w, len(want) + 1000), want), k
        if k:
            with pytest.raises(g5.G5Error) as e:
                g5.s4_decode(w, len(want) - 1)
            assert e.value.code == -4  # more values than the capacity


@pytest.mark.parametrize("n", [5000, 400000])
def test_bad_headers(n):
    x = next(kinds(n, 5))[1]
    w = O.s4_encode(x)
    for at, val in ((1, 7), (2, 7), (3, 7), (0, 127), (0, n // 128 * 128 + 128 * 2048)):
        bad = w.copy()
        bad[at] = val
        with pytest.raises(g5.G5Error) as e:
            g5.s4_decode(bad, n + 128 * 5000)
        assert e.value.code == -5
    bad = w.copy()
    bad[4] = 33 << 24
    with pytest.raises(g5.G5Error) as e:
        g5.s4_decode(bad, n)
    assert e.value.code == -5
    assert np.array_equal(g5.s4_decode(w, n), x)
