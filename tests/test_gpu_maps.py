"""Element-wise maps whose operands walk memory across the result's rows (turned through LDS in 64 x 64 tiles where that is ahead) and
maps whose rows are no whole number of aligned vectors: exact against numpy on small integers, at the edges of the tile and of the
vector, on maps small enough for the element-by-element kernel and large enough for the others."""
import ctypes

import numpy as np
import pytest

import swiftrt_amd as srt
from swiftrt_amd import native
from tests import helpers as H

pytestmark = pytest.mark.gpu
DTS = [H.F32, H.F16, H.BF16]


def ints(g, shape, dt):
    return H.encode(g.integers(-8, 9, shape), dt)


def check(got, want, dt):
    assert np.array_equal(H.to64(got.array()), H.to64(H.encode(want, dt)))


@pytest.mark.parametrize("dt", DTS)
@pytest.mark.parametrize("m,n", [(16, 16), (15, 200), (63, 65), (64, 128), (129, 17), (300, 1001)])
def test_turned_operands(dt, m, n):
    g = H.rng(m * n)
    at, bt, a, b = ints(g, (n, m), dt), ints(g, (n, m), dt), ints(g, (m, n), dt), ints(g, (n,), dt)
    A, B = H.to64(at).T, H.to64(bt).T
    T = srt.Tensor
    out = lambda: srt.Tensor(shape=[m, n], dtype=at.dtype)   # noqa: E731
    q = srt.current_queue()
    for lhs, rhs, want in [(T(at).t, T(a), A + H.to64(a)), (T(a), T(bt).t, H.to64(a) + B), (T(at).t, T(bt).t, A + B),
                           (T(at).t, T.repeating(T(b), [m, n]), A + H.to64(b)), (T(at).t, 3.0, A + 3)]:
        o = out()
        q.add(lhs, rhs, o)
        check(o, want, dt)
    o = out()
    q.neg(T(at).t, o)
    check(o, -A, dt)
    other = H.BF16 if dt == H.F32 else H.F32
    o = srt.Tensor(shape=[m, n], dtype=H.NP_STORAGE[other])
    q.copy(T(at).t, o)                                       # with conversion
    check(o, A, other)


# enough full tiles to be turned: a tile less a row or column, whole ones, several with remainders, rows of whole pieces that fill a
# third of their tiles (16-bit), long rows of a few
@pytest.mark.parametrize("dt", DTS)
@pytest.mark.parametrize("m,n", [(61, 62), (64, 64), (48, 56), (127, 190), (300, 1001), (40, 40), (16, 1028), (33, 2049)])
def test_turned_operands_of_large_maps(dt, m, n):
    g = H.rng(m * n + 1)
    batch = -(-2_100_000 // (m * n))
    at, bt, a, b = ints(g, (batch, n, m), dt), ints(g, (batch, n, m), dt), ints(g, (batch, m, n), dt), ints(g, (n,), dt)
    A, B = np.swapaxes(H.to64(at), 1, 2), np.swapaxes(H.to64(bt), 1, 2)
    T, q = srt.Tensor, srt.current_queue()
    for lhs, rhs, want in [(T(at).t, T(a), A + H.to64(a)), (T(a), T(bt).t, H.to64(a) + B), (T(at).t, T(bt).t, A + B),
                           (T(at).t, T.repeating(T(b), [batch, m, n]), A + H.to64(b)), (T(at).t, 3.0, A + 3)]:
        o = T(shape=[batch, m, n], dtype=at.dtype)
        q.add(lhs, rhs, o)
        check(o, want, dt)
    other = H.BF16 if dt == H.F32 else H.F32
    o = T(shape=[batch, m, n], dtype=H.NP_STORAGE[other])
    q.copy(T(at).t, o)                                       # with conversion
    check(o, A, other)
    frame = T(H.encode(np.full((batch, m + 3, n + 5), 5), dt))
    q.copy(T(at).t, frame[:, 1:1 + m, 3:3 + n])
    want = np.full((batch, m + 3, n + 5), 5.0)
    want[:, 1:1 + m, 3:3 + n] = A
    check(frame, want, dt)


@pytest.mark.parametrize("dt", DTS)
def test_turned_inside_a_batch_and_a_frame(dt):
    g = H.rng(3)
    x = ints(g, (3, 70, 90), dt)
    frame = srt.Tensor(H.encode(np.full((3, 100, 80), 5), dt))
    view = frame[:, 4:94, 3:73]
    srt.current_queue().copy(srt.Tensor(x).t, view)
    want = np.full((3, 100, 80), 5.0)
    want[:, 4:94, 3:73] = np.swapaxes(H.to64(x), 1, 2)
    check(frame, want, dt)


@pytest.mark.parametrize("dt", DTS)
@pytest.mark.parametrize("n", [7, 15, 16, 17, 33, 1001])
def test_ragged_rows(dt, n):
    g = H.rng(n)
    a, b = ints(g, (37, n), dt), ints(g, (n,), dt)
    frame = srt.Tensor(H.encode(np.full((37, n + 5), 5), dt))
    srt.current_queue().mul(srt.Tensor(a), srt.Tensor.repeating(srt.Tensor(b), [37, n]), frame[:, 3:3 + n])
    want = np.full((37, n + 5), 5.0)
    want[:, 3:3 + n] = H.to64(a) * H.to64(b)
    check(frame, want, dt)
    check(srt.Tensor(a) + srt.Tensor(a), 2 * H.to64(a), dt)
    flat = srt.Tensor(np.ascontiguousarray(a.reshape(-1)[1:]))
    check(flat + flat, 2 * H.to64(a).reshape(-1)[1:], dt)


# every remainder of a vector, rows from the fewest vectors that go this way; maps past the size from which ragged rows take vectors,
# past the one for long chains of arithmetic, and past the one from which a lane takes four vectors
@pytest.mark.parametrize("dt", DTS)
@pytest.mark.parametrize("n,elements", [*((n, 2_100_000) for n in (16, 17, 19, 31, 32, 33, 34, 35, 36, 37, 38, 39, 47, 1001)),
                                        (17, 6_100_000), (23, 6_100_000), (63, 800_000), (999, 41_000_000), (1001, 41_000_000)])
def test_ragged_rows_of_large_maps(dt, n, elements):
    g = H.rng(n)
    m = -(-elements // n)
    a, c, b = ints(g, (m, n), dt), ints(g, (m, n), dt), ints(g, (n,), dt)
    T, q = srt.Tensor, srt.current_queue()
    frame = T(H.encode(np.full((m, n + 5), 5), dt))
    view, row = frame[:, 3:3 + n], T.repeating(T(b), [m, n])
    want = np.full((m, n + 5), 5.0)
    want[:, 3:3 + n] = H.to64(a) * H.to64(b)
    q.mul(T(a), row, view)
    check(frame, want, dt)
    want[:, 3:3 + n] = want[:, 3:3 + n] - H.to64(c)
    q.subtract(view, T(c), view)                             # in place: a vector moved back to end inside its row reads its neighbour's
    check(frame, want, dt)
    if elements > 10_000_000:
        return
    want[:, 3:3 + n] = H.to64(H.encode(H.to64(b) - want[:, 3:3 + n], dt))
    q.subtract(row, view, view)
    check(frame, want, dt)
    dense, got = T(shape=[m, n], dtype=a.dtype), T(H.encode(np.full((m, n + 5), 5), dt))
    scaled = T(H.encode(g.standard_normal((m, n)), dt))
    q.tanh(scaled, dense)                                    # (dense: aligned vectors)
    q.tanh(scaled, got[:, 3:3 + n])
    full = got.array()
    assert np.array_equal(full[:, 3:3 + n].view(np.uint16), dense.array().view(np.uint16))
    assert np.all(H.to64(full[:, :3]) == 5) and np.all(H.to64(full[:, 3 + n:]) == 5)
    other = H.BF16 if dt == H.F32 else H.F32
    o = T(shape=[m, n], dtype=H.NP_STORAGE[other])
    q.copy(view, o)                                          # with conversion
    check(o, want[:, 3:3 + n], other)


@pytest.mark.parametrize("dt", DTS)
def test_column_major_results_are_walked_in_their_storage_order(dt):
    g = H.rng(4)
    a, b = ints(g, (65, 130), dt), ints(g, (65, 130), dt)
    col = lambda x: srt.Tensor(x, order=srt.Order.col)       # noqa: E731
    check(col(a) + col(b), H.to64(a) + H.to64(b), dt)
    check(col(a) + srt.Tensor(b), H.to64(a) + H.to64(b), dt)   # row-major into column-major


@pytest.mark.parametrize("count", [0xfffffff9, 0xffffffff])
def test_extents_just_below_32_bits(count):
    """One dense 16-bit row whose extent rounded up to whole vectors passes 2^32 (two buffers of 8.6 GB): read back at both ends and
    in the middle."""
    L, q = native.lib(), srt.current_queue()
    d, keep = native.make_descriptor(native.REAL16BF, (count,), (1,), native.ORDER_ROW)
    src, dst = q.allocate(2 * count), q.allocate(2 * count)
    element = np.array([0x3FC0], np.uint16)              # 1.5
    native.check(L.srtFillFlat(native.REAL16BF, src.pointer, ctypes.c_void_p(element.ctypes.data), count, q.stream))
    q.zero(dst, 2 * count)
    native.check(L.srtNeg(src.pointer, ctypes.byref(d), dst.pointer, ctypes.byref(d), q.stream))
    for at in (0, count // 2, count - 4096):
        got = np.zeros(4096, np.uint16)
        native.check(L.srtMemcpyAsync(ctypes.c_void_p(got.ctypes.data), ctypes.c_void_p(dst.pointer + 2 * at), 8192, native.D2H,
                                      q.stream))
        q.wait_for_completion()
        assert np.all(got == 0xBFC0), at
