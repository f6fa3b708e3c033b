"""The LSTM gate kernel against the element-wise operations it stands for (bit for bit), concatenation in one launch, and
element-wise maps either side of the size at which a lane takes four vectors."""
import numpy as np
import pytest

import swiftrt_amd as srt
from swiftrt_amd import native
from tests import helpers as H

pytestmark = pytest.mark.gpu
DTS = [H.F32, H.F16, H.BF16]


def unfused(gates, cell):
    """Recurrent.swift:255-266 as nine device operations."""
    h = cell.shape[1]
    part = [gates[:, i * h:(i + 1) * h] for i in range(4)]
    new_cell = cell * srt.sigmoid(part[2]) + srt.sigmoid(part[0]) * srt.tanh(part[1])
    return new_cell, srt.tanh(new_cell) * srt.sigmoid(part[3])


def bits(t):
    a = t.array()
    return a.view(np.uint32 if a.dtype == np.float32 else np.uint16)


# one element; an odd width; the lane-per-element form; the vector form (over 256 x 1024 elements), and too odd for it
@pytest.mark.parametrize("dt", DTS)
@pytest.mark.parametrize("b,h", [(1, 1), (3, 37), (64, 512), (512, 1024), (513, 1023)])
def test_gates_are_the_unfused_chain(dt, b, h):
    g = H.rng(b + h)
    gates = srt.Tensor(H.encode(3 * g.standard_normal((b, 4 * h)), dt))
    cell = srt.Tensor(H.encode(g.standard_normal((b, h)), dt))
    nc, nh = srt.Tensor(shape=[b, h], dtype=cell.dtype), srt.Tensor(shape=[b, h], dtype=cell.dtype)
    srt.current_queue().lstm_gates(gates, cell, nc, nh)
    want_cell, want_hidden = unfused(gates, cell)
    assert np.array_equal(bits(nc), bits(want_cell)) and np.array_equal(bits(nh), bits(want_hidden))


def test_gates_beyond_31_bits_of_lanes():
    """The odd width goes lane per element; 2^31 of them take a second launch.  One value everywhere but in the last row."""
    rows, h = 0x80000000 // 1023 + 2, 1023
    q = srt.current_queue()
    filled = lambda shape, value: srt.filled(shape, value, np.uint16)          # noqa: E731
    gates, cell = filled([rows, 4 * h], 0.5), filled([rows, h], 0.25)
    q.fill(last := srt.Tensor(shape=[1, 4 * h], dtype=np.uint16), -1.0)
    q.copy(last, gates[rows - 1:rows])
    nc, nh = srt.Tensor(shape=[rows, h], dtype=np.uint16), srt.Tensor(shape=[rows, h], dtype=np.uint16)
    q.lstm_gates(gates, cell, nc, nh)
    for at in (0, rows // 2, rows - 2, rows - 1):
        row = slice(at, at + 1)
        dense = lambda t: (o := srt.Tensor(shape=[1, t.shape[1]], dtype=np.uint16), q.copy(t[row], o))[0]   # noqa: E731
        want_cell, want_hidden = unfused(dense(gates), dense(cell))
        assert np.array_equal(bits(dense(nc)), bits(want_cell)) and np.array_equal(bits(dense(nh)), bits(want_hidden)), at


def test_gates_on_views_and_refusals():
    g = H.rng(5)
    wide = srt.Tensor(g.standard_normal((9, 200)).astype(np.float32))
    gates, cell = wide[:, 3:3 + 4 * 24], wide[:, 120:144]
    out = srt.Tensor(np.zeros((9, 60), np.float32))
    q = srt.current_queue()
    q.lstm_gates(gates, cell, out[:, 1:25], out[:, 30:54])
    want_cell, want_hidden = unfused(gates, cell)
    got = out.array()
    assert np.array_equal(got[:, 1:25], want_cell.array()) and np.array_equal(got[:, 30:54], want_hidden.array())
    assert not got[:, [0, *range(25, 30), *range(54, 60)]].any()
    with pytest.raises(native.SrtError):
        q.lstm_gates(gates, wide[:, :23], out[:, 1:24], out[:, 30:53])       # gates are not four times as wide


@pytest.mark.parametrize("dt", DTS)
def test_cells_the_gate_kernel_does_not_take(dt):
    """A weight with columns past the fourth part; one row of gates under several rows of state, or under a stack of them."""
    g = H.rng(6)
    make = lambda *shape: srt.Tensor(H.encode(g.standard_normal(shape), dt))   # noqa: E731
    h = 24
    for columns, batch, state in ((4 * h + 3, 5, (5, h)), (4 * h, 1, (5, h)), (4 * h, 5, (3, 5, h))):
        weight, bias, x, hidden, cell = make(16 + h, columns), make(columns), make(batch, 16), make(batch, h), make(*state)
        new_cell, new_hidden = srt.LSTMCell(weight, bias)(x, cell, hidden)
        fused = srt.matmul(srt.concatenate(x, hidden, 1), weight, bias=bias)
        part = [fused[:, i * h:(i + 1) * h] for i in range(4)]
        want_cell = cell * srt.sigmoid(part[2]) + srt.sigmoid(part[0]) * srt.tanh(part[1])
        assert new_cell.shape == state and np.array_equal(bits(new_cell), bits(want_cell))
        assert np.array_equal(bits(new_hidden), bits(srt.tanh(want_cell) * srt.sigmoid(part[3])))


@pytest.mark.parametrize("dt", DTS)
@pytest.mark.parametrize("shapes,axis", [(((4, 8), (4, 16)), 1), (((3, 5), (3, 7)), 1), (((5, 9), (2, 9)), 0),
                                         (((2, 3, 8), (2, 4, 8)), 1), (((1024, 3000), (1024, 3000)), 1), (((4, 0), (4, 3)), 1)])
def test_concatenate(dt, shapes, axis):
    g = H.rng(7)
    a, b = [H.encode(g.standard_normal(s), dt) for s in shapes]
    got = srt.concatenate(srt.Tensor(a), srt.Tensor(b), axis)
    assert np.array_equal(got.array(), np.concatenate([a, b], axis))
    if a.ndim == 2 and a.size:
        got = srt.concatenate(srt.Tensor(np.ascontiguousarray(a.T)).t, srt.Tensor(b), axis)   # a strided operand
        assert np.array_equal(got.array(), np.concatenate([a, b], axis))


@pytest.mark.parametrize("dt", DTS)
def test_maps_either_side_of_one_vector_per_lane(dt):
    g = H.rng(9)
    per = 4 if dt == H.F32 else 8
    edge = 80_000_000 // (256 * 2 * per * (4 if dt == H.F32 else 2)) * per     # 256 rows: just below the boundary, past it, no vectors
    for columns in (edge, edge + per, edge + 1):
        x = H.encode(g.integers(-8, 9, (256, columns)), dt)
        b = H.encode(g.integers(-8, 9, columns), dt)
        got = srt.Tensor(x) + srt.Tensor(b)
        want = H.encode(H.to64(x) + H.to64(b), dt)
        assert np.array_equal(H.to64(got.array()), H.to64(want))
