"""Results are born on the device: nothing is made on the host or copied there before the host asks, and what the host then
sees is what the call wrote (zeros where nothing has)."""
import numpy as np
import pytest

import swiftrt_amd as srt
from swiftrt_amd import native

pytestmark = pytest.mark.gpu


def test_a_result_has_no_host_replica_until_read():
    a = srt.Tensor(np.arange(12, dtype=np.float32).reshape(3, 4))
    c = srt.matmul(a, srt.Tensor(np.eye(4, dtype=np.float32)))
    assert c.storage._host is None
    assert np.array_equal(c.array(), np.arange(12, dtype=np.float32).reshape(3, 4))
    assert c.storage.last_copy == "d2h"


def test_a_fresh_tensor_reads_as_zeros_on_both_sides():
    z = srt.Tensor(shape=[5, 7], dtype=np.float32)
    out = z + 1.0                                        # read on the device first
    assert np.array_equal(out.array(), np.ones((5, 7), np.float32)) and np.array_equal(z.array(), np.zeros((5, 7), np.float32))


def test_a_partial_write_keeps_the_rest_of_the_buffer():
    q = srt.current_queue()
    fresh = srt.Tensor(shape=[4, 6], dtype=np.float32)   # never written as a whole: zeros around the view
    q.copy(srt.Tensor(np.ones((4, 2), np.float32)), fresh[:, 2:4])
    assert np.array_equal(fresh.array(), np.tile(np.float32([0, 0, 1, 1, 0, 0]), (4, 1)))
    held = srt.Tensor(np.full((4, 6), 3, np.float32))
    q.copy(srt.Tensor(np.ones((4, 2), np.float32)), held[:, 2:4])
    assert np.array_equal(held.array(), np.tile(np.float32([3, 3, 1, 1, 3, 3]), (4, 1)))


def test_a_refused_call_leaves_the_result_as_it_was():
    q = srt.current_queue()
    a = srt.Tensor(np.ones((4, 4), np.float32))
    out = srt.Tensor(np.full((4, 5), 2, np.float32))
    with pytest.raises(native.SrtError):
        q.matmul(a, False, a, False, out)
    assert np.array_equal(out.array(), np.full((4, 5), 2, np.float32))
    assert np.array_equal((out + 0.0).array(), np.full((4, 5), 2, np.float32))
