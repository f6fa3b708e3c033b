"""The LSTM step in one launch against the three calls it stands for: integer-valued operands, whose sums are exact in any order, so
the gates and with them the results agree bit for bit; cells it does not take; results in memory that an operand uses."""
import numpy as np
import pytest

import swiftrt_amd as srt
from tests import helpers as H
from tests.test_gpu_cells import bits

pytestmark = pytest.mark.gpu
q = lambda: srt.current_queue()   # noqa: E731


def cell_inputs(dt, b, i, h, seed, bias_step=1):
    g = H.rng(seed)
    make = lambda *shape: srt.Tensor(H.encode(g.integers(-2, 3, shape) / 4.0, dt))   # noqa: E731
    bias = make(4 * h * bias_step)[::bias_step]
    return make(b, i), make(b, h), make(b, h), make(i + h, 4 * h), bias


def by_calls(x, cell, hidden, weight, bias):
    gates = srt.matmul(srt.concatenate(x, hidden, 1), weight, bias=bias)
    nc, nh = srt.Tensor(shape=cell.shape, dtype=cell.dtype), srt.Tensor(shape=cell.shape, dtype=cell.dtype)
    q().lstm_gates(gates, cell, nc, nh)
    return nc, nh


# rows either side of a tile; inputs and hidden either side of a slab, of a 16-byte piece and of a round of the waves' slabs; one
# group of columns; two tiles a unit
@pytest.mark.parametrize("dt", [H.F32, H.F16, H.BF16])
@pytest.mark.parametrize("b,i,h", [(1, 8, 8), (31, 9, 16), (32, 32, 64), (33, 31, 72), (5, 65, 40), (64, 512, 512), (70, 333, 128), (128, 257, 1024),
                                   (40, 700, 520), (3, 1024, 1000)])
def test_one_launch_is_the_three(dt, b, i, h):
    x, cell, hidden, weight, bias = cell_inputs(dt, b, i, h, b + i + h, bias_step=2 if b == 31 else 1)
    nc, nh = srt.Tensor(shape=[b, h], dtype=x.dtype), srt.Tensor(shape=[b, h], dtype=x.dtype)
    assert q().lstm_cell(x, cell, hidden, weight, bias, nc, nh)
    want_cell, want_hidden = by_calls(x, cell, hidden, weight, bias)
    assert np.array_equal(bits(nc), bits(want_cell)) and np.array_equal(bits(nh), bits(want_hidden))


def test_views_stay_inside_and_a_nan_in_its_row():
    g = H.rng(9)
    b, i, h = 37, 45, 24
    buf = np.full((b, 200), np.nan, np.float32)
    buf[:, 3:3 + i], buf[:, 60:60 + h], buf[:, 100:100 + h] = (g.integers(-2, 3, (b, n)) / 4.0 for n in (i, h, h))
    buf[5, 4] = np.nan
    weight_buf = np.full((i + h, 4 * h + 7), np.nan, np.float32)
    weight_buf[:, 2:2 + 4 * h] = g.integers(-2, 3, (i + h, 4 * h)) / 4.0
    wide, outs = srt.Tensor(buf), [srt.Tensor(np.full((b, 30), 7.0, np.float32)) for _ in range(2)]
    x, hidden, cell = wide[:, 3:3 + i], wide[:, 60:60 + h], wide[:, 100:100 + h]
    weight, bias = srt.Tensor(weight_buf)[:, 2:2 + 4 * h], srt.Tensor(np.zeros(4 * h, np.float32))
    assert q().lstm_cell(x, cell, hidden, weight, bias, *(o[:, 1:1 + h] for o in outs))
    for o, want in zip(outs, by_calls(x, cell, hidden, weight, bias)):
        got = o.array()
        assert np.array_equal(got[:, 1:1 + h], want.array(), equal_nan=True) and (got[:, [0, *range(1 + h, 30)]] == 7.0).all()
        rows = np.isnan(got).any(1)
        assert rows[5] and rows.sum() == 1


def test_cells_left_to_the_three_calls():
    for b, i, h in ((4, 16, 12), (4, 3, 16), (512, 64, 1024)):   # columns not in groups; x short of a piece; more than two tiles a unit
        x, cell, hidden, weight, bias = cell_inputs(H.F32, b, i, h, 3)
        nc, nh = srt.Tensor(shape=[b, h], dtype=np.float32), srt.Tensor(shape=[b, h], dtype=np.float32)
        assert not q().lstm_cell(x, cell, hidden, weight, bias, nc, nh)
        got = srt.LSTMCell(weight, bias)(x, cell, hidden)
        for a, w in zip(got, by_calls(x, cell, hidden, weight, bias)):
            assert np.array_equal(a.array(), w.array())
    x, cell, hidden, weight, bias = cell_inputs(H.F32, 8, 16, 16, 4)
    new = srt.Tensor(shape=[8, 16], dtype=np.float32)
    for nc, nh in ((cell, new), (new, hidden), (new, new), (new, x)):   # other workgroups still read what one would store
        assert not q().lstm_cell(x, cell, hidden, weight, bias, nc, nh)


@pytest.mark.parametrize("dt", [H.F32, H.BF16])
def test_a_cell_without_a_bias(dt):
    x, cell, hidden, weight, _ = cell_inputs(dt, 9, 24, 16, 5)
    layer = srt.LSTMCell(weight, None)
    got = layer(x, cell, hidden)
    gates = srt.matmul(srt.concatenate(x, hidden, 1), weight)
    update, add, keep, out = (layer.part(i, gates) for i in range(4))
    new_cell = cell * srt.sigmoid(keep) + srt.sigmoid(update) * srt.tanh(add)
    for a, w in zip(got, (new_cell, srt.tanh(new_cell) * srt.sigmoid(out))):
        assert np.array_equal(bits(a), bits(w))


# device us, three launches / one: a cell is taken where one is ahead, there or (under 35 us) for a program that makes the three calls
@pytest.mark.parametrize("dt,b,i,h,taken", [
    (H.BF16, 32, 1024, 1024, True), (H.BF16, 128, 1024, 1024, True), (H.BF16, 64, 512, 2048, True),         # 18.8 / 9.5, 20.9 / 22.1, 24.2 / 30.4
    (H.BF16, 128, 4096, 1024, False), (H.BF16, 8, 8192, 256, False), (H.F16, 64, 16384, 8, True),           # 27.5 / 50.7, 26.4 / 36.9, 55.9 / 21.9
    (H.F32, 128, 1024, 1024, True), (H.F32, 64, 1024, 2048, False), (H.F32, 64, 16384, 256, False)])        # 36.3 / 33.4, 41.5 / 48.5, 90.8 / 103.6
def test_cells_are_taken_where_one_launch_is_ahead(dt, b, i, h, taken):
    dtype = H.encode(np.zeros(1), dt).dtype
    make = lambda *shape: srt.Tensor(shape=shape, dtype=dtype)   # noqa: E731
    assert q().lstm_cell(make(b, i), make(b, h), make(b, h), make(i + h, 4 * h), make(4 * h), make(b, h), make(b, h)) == taken
