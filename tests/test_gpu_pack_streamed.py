"""Copies of 75 MB and more, whose sources are read with the streaming hint: rows off every vector, inside a frame of NaNs, each layout of the
right operand, one that is just below.  Small integers, so the products are exact."""
import numpy as np
import pytest

import swiftrt_amd as srt
from tests import helpers as H
from tests.test_gpu_matmul import query_kernel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt,m,n,k", [(H.BF16, 129, 40003, 1001), (H.F32, 65, 20003, 1001), (H.F16, 130, 36001, 1001)])
@pytest.mark.parametrize("transposed", [False, True])
def test_large_copies(dt, m, n, k, transposed):
    g = H.rng(n)
    a = g.integers(-2, 3, (m, k)).astype(np.float32)
    b = np.tile(g.integers(-2, 3, (k, 97)), (1, -(-n // 97)))[:, :n].astype(np.float32)
    want = np.tile(a @ b[:, :97], (1, -(-n // 97)))[:, :n]
    w = np.ascontiguousarray(b.T) if transposed else b
    frame = np.full((w.shape[0] + 1, w.shape[1] + 3), np.nan, np.float32)
    frame[:-1, 1:-2] = w
    x = srt.Tensor(H.encode(a, dt))
    wt = srt.Tensor(H.encode(frame, dt))[:-1, 1:1 + w.shape[1]]
    with H.pinned("copied", dt, m, n, k, 1 | (4 if transposed else 8) | 16):
        got = srt.matmul(x, wt, transposed_rhs=transposed)
        assert query_kernel(x, False, wt, transposed, got) == "copied"
    assert np.array_equal(got.array(), H.encode(want, dt))


@pytest.mark.parametrize("dt,m,n,k,transposed", [(H.BF16, 129, 81003, 1001, False), (H.F32, 65, 41003, 1001, True), (H.F16, 66, 90001, 1001, True)])
def test_copies_read_with_the_hint(dt, m, n, k, transposed):
    assert 160e6 < n * k * (4 if dt == H.F32 else 2) < 270e6
    test_large_copies(dt, m, n, k, transposed)
