"""Layouts and descriptors shared between tensors: by layout and nothing else, and no more of them than the limit."""
import numpy as np

import swiftrt_amd as srt
from swiftrt_amd import tensor as T


def descriptor(t):
    t.descriptor_ref()
    d = t._descriptor[1]
    return d.type, d.rank, d.order, d.count, d.spanCount, [d.shape[i] for i in range(d.rank)], [d.strides[i] for i in range(d.rank)]


def test_descriptors_are_those_of_their_layout():
    base = srt.Tensor(np.zeros((6, 8), np.float32))
    views = [base, base.t, base[1:5, 2:8:2], srt.Tensor(shape=[6, 8], dtype=np.float16), srt.Tensor(shape=(6, 8), dtype=np.float32, order=srt.Order.col),
             srt.Tensor(shape=[np.int64(6), 8], dtype=np.uint16), srt.Tensor.repeating(srt.Tensor(shape=[8], dtype=np.float32), [6, 8])]
    for _ in range(2):
        for t in views:
            d, keep = t.descriptor()
            want = d.type, d.rank, d.order, d.count, d.spanCount, [d.shape[i] for i in range(d.rank)], [d.strides[i] for i in range(d.rank)]
            assert descriptor(t) == want
    assert srt.Tensor(shape=[6, 8], dtype=np.float32).descriptor_ref() is base.descriptor_ref()


def test_the_shared_layouts_are_bounded(monkeypatch):
    monkeypatch.setattr(T, "_LAYOUTS_MOST", 8)
    tensors = [srt.Tensor(shape=[3, n], dtype=np.float32) for n in range(1, 40)]
    made = [descriptor(t) for t in tensors]
    assert len(T._dense_layouts) <= 8 and len(T._descriptors) <= 8
    assert [descriptor(t) for t in tensors] == made and all(t.strides == (t.shape[1], 1) for t in tensors)   # what they hold stays
