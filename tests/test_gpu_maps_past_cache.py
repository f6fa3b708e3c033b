"""Maps of 256 MiB of traffic and more, whose lanes take two vectors each and store past the caches: the last vector of a row and of a block,
rows on whole lines, on whole vectors and off them, with a row under every other one, turned operands and a conversion.  The operands repeat
a pattern of 61 rows, of small integers, so every result is exact and known from the pattern."""
import numpy as np
import pytest

import swiftrt_amd as srt
from tests import helpers as H

pytestmark = pytest.mark.gpu
T = srt.Tensor
PATTERN = 61


def repeated(pattern, rows):
    return np.ascontiguousarray(np.tile(pattern, (-(-rows // PATTERN), 1))[:rows])


def bits(a):
    return a.view(np.uint32 if a.itemsize == 4 else np.uint16)


def check(got, pattern, rows):
    got, pattern = bits(got.array()).reshape(rows, -1), bits(pattern)
    whole = rows // PATTERN * PATTERN
    assert (got[:whole].reshape(-1, *pattern.shape) == pattern).all()
    assert (got[whole:] == pattern[:rows - whole]).all()


@pytest.mark.parametrize("dt", [H.F32, H.F16, H.BF16])
@pytest.mark.parametrize("n", [4096, 2056, 1001, 255])
def test_maps_past_the_cache(dt, n):
    size = 4 if dt == H.F32 else 2
    rows = (1 << 28) // (2 * size * n) + 3                     # an input and a result are just past the line
    g = H.rng(n)
    a, row = H.encode(g.integers(-8, 9, (PATTERN, n)), dt), H.encode(g.integers(-8, 9, (n,)), dt)
    x, q = T(repeated(a, rows)), srt.current_queue()
    A = H.to64(a)
    o = T(shape=[rows, n], dtype=a.dtype)
    q.add(x, T.repeating(T(row), [rows, n]), o)
    check(o, H.encode(A + H.to64(row), dt), rows)
    q.neg(x, o)
    check(o, H.encode(-A, dt), rows)
    q.add(x, x, x)                                             # in place
    check(x, H.encode(2 * A, dt), rows)
    other = H.BF16 if dt == H.F32 else H.F32
    c = T(shape=[rows, n], dtype=H.NP_STORAGE[other])
    q.copy(x, c)
    check(c, H.encode(2 * A, other), rows)


# results' rows on whole 128-byte lines and off them; extents off the tile
@pytest.mark.parametrize("dt", [H.F32, H.BF16])
@pytest.mark.parametrize("rows,off", [(8192, 0), (8256, 40), (8200, 0), (8193, 1)])
def test_turned_maps_past_the_cache(dt, rows, off):
    size = 4 if dt == H.F32 else 2
    n = (1 << 28) // (2 * size * rows) + 5 + off
    a = H.encode(H.rng(rows).integers(-8, 9, (PATTERN, rows)), dt)
    x = T(repeated(a, n))                                      # [n, rows], n the operand's rows
    o = T(shape=[rows, n], dtype=a.dtype)
    q = srt.current_queue()
    q.neg(x.t, o)
    want = np.ascontiguousarray(repeated(H.encode(-H.to64(a), dt), n).T)
    assert (bits(o.array()) == bits(want)).all()
    back = T(shape=[n, rows], dtype=a.dtype)
    q.copy(o.t, back)                                          # rows of `rows` elements: whole lines for 8192 and 8256
    check(back, H.encode(-H.to64(a), dt), n)
