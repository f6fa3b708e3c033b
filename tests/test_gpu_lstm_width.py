"""The LSTM step in one launch for hidden sizes that are no whole groups of eight: the bits of the three calls, nothing read or stored outside the views."""
import numpy as np
import pytest

import swiftrt_amd as srt
from tests import helpers as H
from tests.test_gpu_cells import bits
from tests.test_gpu_lstm_cell import by_calls, cell_inputs

pytestmark = pytest.mark.gpu


# the last group of one to seven columns, the smallest width, either side of a slab, rows past a tile, k ranges of any end
@pytest.mark.parametrize("dt", [H.F32, H.F16, H.BF16])
@pytest.mark.parametrize("b,i,h", [(1, 8, 17), (5, 40, 20), (33, 31, 23), (2, 65, 44), (64, 100, 65), (9, 16, 99), (40, 721, 254), (3, 384, 1020)])
def test_one_launch_is_the_three(dt, b, i, h):
    x, cell, hidden, weight, bias = cell_inputs(dt, b, i, h, b + i + h, bias_step=2 if b == 33 else 1)
    nc, nh = srt.Tensor(shape=[b, h], dtype=x.dtype), srt.Tensor(shape=[b, h], dtype=x.dtype)
    assert srt.current_queue().lstm_cell(x, cell, hidden, weight, bias, nc, nh)
    for got, want in zip((nc, nh), by_calls(x, cell, hidden, weight, bias)):
        assert np.array_equal(bits(got), bits(want))


@pytest.mark.parametrize("dt", [H.F32, H.BF16])
def test_between_nans(dt):
    """Every operand a view with NaN on both sides of its rows, the bias too; the results views of a buffer of sevens."""
    b, i, h = 37, 45, 29
    g = H.rng(19)

    def framed(rows, columns):
        buf = np.full((rows + 2, columns + 5), np.nan, np.float32)
        buf[1:-1, 2:2 + columns] = g.integers(-2, 3, (rows, columns)) / 4.0
        return srt.Tensor(H.encode(buf, dt))[1:rows + 1, 2:2 + columns]
    x, hidden, cell, weight = framed(b, i), framed(b, h), framed(b, h), framed(i + h, 4 * h)
    row = np.full(4 * h + 9, np.nan, np.float32)
    row[4:4 + 4 * h] = g.integers(-2, 3, 4 * h) / 4.0
    bias = srt.Tensor(H.encode(row, dt))[4:4 + 4 * h]
    outs = [srt.Tensor(H.encode(np.full((b, h + 4), 7.0), dt)) for _ in range(2)]
    assert srt.current_queue().lstm_cell(x, cell, hidden, weight, bias, *(o[:, 1:1 + h] for o in outs))
    dense = [srt.Tensor(v.array()) for v in (x, cell, hidden, weight, bias)]
    for o, want in zip(outs, by_calls(*dense)):
        got = H.to64(o.array())
        assert np.array_equal(got[:, 1:1 + h], H.to64(want.array())) and (got[:, [0, *range(1 + h, h + 4)]] == 7.0).all()


# a program's step, us, one launch / three calls
@pytest.mark.parametrize("dt,b,i,h,taken", [
    (H.BF16, 6, 2975, 2079, False), (H.F16, 2, 1245, 2415, False), (H.F32, 78, 2842, 663, False),     # 75 / 37, 55 / 35, 55 / 36
    (H.F16, 1, 384, 1020, True), (H.BF16, 6, 975, 2078, True), (H.F32, 64, 512, 511, True)])          # 19 / 40; 28 / 36
def test_cells_are_taken_where_one_launch_is_ahead(dt, b, i, h, taken):
    dtype = H.encode(np.zeros(1), dt).dtype
    make = lambda *shape: srt.Tensor(shape=shape, dtype=dtype)   # noqa: E731
    assert srt.current_queue().lstm_cell(make(b, i), make(b, h), make(b, h), make(i + h, 4 * h), make(4 * h), make(b, h), make(b, h)) == taken
