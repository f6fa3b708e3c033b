"""Which of its two tiles the kernel whose waves split k (gemm_waves.h) takes for x^T . W, by the grid of a captured call; us, 32 x 32 / 64 x 64 tiles."""
import ctypes
import os

import numpy as np
import pytest

import swiftrt_amd as srt
from swiftrt_amd import native
from tests import helpers as H
from tests.test_gpu_captured_workspace import captured
from tests.test_gpu_stream import KernelNode

pytestmark = [pytest.mark.gpu, pytest.mark.skipif("debug" in os.environ.get("SWIFTRT_HIP_LIBRARY", ""),
                                                  reason="the debug build synchronises after every launch")]


@pytest.mark.parametrize("M,N,K,edge", [(512, 1280, 8104, 64), (704, 1024, 5769, 64), (1578, 384, 4776, 64), (72, 600, 4104, 32),   # 67 / 33, 44 / 23
                                        (512, 1280, 136, 32)])
def test_the_tile_of_long_k_loops(M, N, K, edge):
    g, L, q = H.rng(58), native.lib(), srt.current_queue()
    x, w = (g.integers(-1, 2, s).astype(np.float32) for s in ((K, M), (K, N)))
    xt, wt, out = srt.Tensor(H.encode(x, H.BF16)), srt.Tensor(H.encode(w, H.BF16)), srt.Tensor(shape=[M, N], dtype=np.uint16)
    with H.pinned("mfma_32x32_waves", H.BF16, M, N, K, 26 | (64 if M % 8 == 0 and N % 8 == 0 else 0)):
        q.matmul(xt, True, wt, False, out)
        assert np.array_equal(out.array(), H.encode(x.T @ w, H.BF16))   # (whole sums below 2^24: exact in any order)
        graph, run = captured(q, lambda: q.matmul(xt, True, wt, False, out))
    count, node, kernel = ctypes.c_size_t(1), ctypes.c_void_p(), KernelNode()
    assert L.hipGraphGetNodes(graph, ctypes.byref(node), ctypes.byref(count)) == 0
    assert L.hipGraphKernelNodeGetParams(node, ctypes.byref(kernel)) == 0
    tiles = -(-M // edge) * -(-N // edge)
    assert tiles <= int(np.prod(tuple(kernel.grid))) < tiles + 8   # (a walk's launch: whole eighths)
    assert L.hipGraphExecDestroy(run) == 0 and L.hipGraphDestroy(graph) == 0
