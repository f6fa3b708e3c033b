"""Which calls an LSTM cell makes, by a queue that writes them down."""
import numpy as np

import swiftrt_amd as srt
from swiftrt_amd import tensor as T


class Recorder:
    """Takes a cell's calls in HipQueue's place, as a queue that runs no cell in one launch; reads every operand as it does."""

    def __init__(self):
        self.calls = []

    def lstm_cell(self, x, cell, hidden, weight, bias, new_cell, new_hidden):
        assert all(isinstance(t, T.Tensor) for t in (x, cell, hidden, weight, bias, new_cell, new_hidden))
        self.calls.append(("lstm_cell",))
        return False

    def concatenate(self, a, b, axis, out):
        self.calls.append(("concatenate", a.shape, b.shape, axis))

    def matmul(self, lhs, transpose_lhs, rhs, transpose_rhs, result, bias=None, activation=None, coef=0.0):
        self.calls.append(("matmul", lhs.shape, rhs.shape, bias))

    def lstm_gates(self, gates, cell, new_cell, new_hidden):
        self.calls.append(("lstm_gates", gates.shape, cell.shape))


def test_a_cell_without_a_bias_makes_the_three_calls(monkeypatch):
    queue = Recorder()
    monkeypatch.setattr(T, "current_queue", lambda: queue)
    make = lambda *shape: srt.Tensor(shape=shape, dtype=np.float32)   # noqa: E731
    bias = make(32)
    for b in (bias, None):
        new_cell, new_hidden = srt.LSTMCell(make(24, 32), b)(make(4, 16), make(4, 8), make(4, 8))
        assert new_cell.shape == new_hidden.shape == (4, 8) and new_cell.dtype == np.float32
    three = lambda b: [("concatenate", (4, 16), (4, 8), 1), ("matmul", (4, 24), (24, 32), b), ("lstm_gates", (4, 32), (4, 8))]   # noqa: E731
    assert queue.calls == [("lstm_cell",)] + three(bias) + three(None)
