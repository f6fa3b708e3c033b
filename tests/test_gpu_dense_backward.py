"""srtDenseBackward: the bits of the three calls it stands for, in either order, of views, with and without a bias, at empty extents; what those refuse."""
import numpy as np
import pytest

import swiftrt_amd as srt
from swiftrt_amd import native
from swiftrt_amd.tensor import matmul_gradients
from tests import helpers as H

pytestmark = pytest.mark.gpu


def three_calls(layer, x, y, dy):
    dz = srt.Tensor(shape=y.shape, dtype=y.dtype, order=y.order)
    db = srt.Tensor(shape=[y.shape[1]], dtype=y.dtype) if layer.bias is not None else None
    srt.current_queue().activation_backward(y, dy, layer.activation, layer.coef, dz, db)
    return *matmul_gradients(dz, x, False, layer.weight, False), db


@pytest.mark.parametrize("M,K,N", [(1, 1, 1), (5, 33, 17), (64, 128, 96), (256, 784, 1000), (300, 257, 131)])
@pytest.mark.parametrize("order", [srt.Order.row, srt.Order.col])
@pytest.mark.parametrize("dt", [H.F32, H.F16, H.BF16])
def test_the_bits_of_the_three_calls(dt, order, M, K, N):
    g = H.rng(81)
    make = lambda *s: H.encode(g.standard_normal(s) / 4, dt)
    wide = srt.Tensor(make(M, K + 3), order=order)
    x = wide[:, 1:K + 1] if M % 2 else srt.Tensor(make(M, K), order=order)
    for act, bias in ((srt.ActivationType.tanh, True), (srt.ActivationType.relu, False)):
        layer = srt.Dense(srt.Tensor(make(K, N), order=order), srt.Tensor(make(N)) if bias else None, act)
        y, dy = layer(x), srt.Tensor(make(M, N), order=order)
        for got, want in zip(srt.dense_backward(layer, x, y, dy), three_calls(layer, x, y, dy)):
            assert (got is None) == (want is None)
            if want is not None:
                assert got.order == want.order and got.shape == want.shape and got.array().tobytes() == want.array().tobytes()


def test_no_rows():
    layer = srt.Dense(srt.Tensor(np.ones((8, 4), np.float32)), srt.Tensor(np.ones(4, np.float32)), srt.ActivationType.relu)
    x, y = srt.Tensor(shape=[0, 8], dtype=np.float32), srt.Tensor(shape=[0, 4], dtype=np.float32)
    dx, dw, db = srt.dense_backward(layer, x, y, y)
    assert dx.shape == (0, 8) and not dw.array().any() and not db.array().any()


def test_what_is_refused():
    layer = srt.Dense(srt.Tensor(np.ones((8, 4), np.float32)), None, srt.ActivationType.relu)
    t = lambda *s, dtype=np.float32: srt.Tensor(np.ones(s, dtype))
    with pytest.raises(ValueError):
        srt.dense_backward(layer, t(3, 8), t(3, 5), t(3, 5))
    with pytest.raises(native.SrtError):
        srt.dense_backward(layer, t(3, 8), t(3, 4), t(2, 4))
    with pytest.raises(native.NotSupportedError):
        srt.dense_backward(layer, t(3, 8, dtype=np.float16), t(3, 4), t(3, 4))
