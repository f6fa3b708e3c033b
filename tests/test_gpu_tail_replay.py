"""A captured product whose plan shares left-over tiles: a replay carries the capture's epoch and would find the flags of the one before raised, so
under capture the tiles are not shared.  Every replay is exact, with the operands changed in between and the program's own calls beside it."""
import ctypes
import os

import numpy as np
import pytest

import swiftrt_amd as srt
from swiftrt_amd import native
from tests import helpers as H
from tests.test_gpu_matmul import query_kernel

pytestmark = pytest.mark.gpu


@pytest.mark.skipif("debug" in os.environ.get("SWIFTRT_HIP_LIBRARY", ""), reason="the debug build synchronises after every launch")
@pytest.mark.parametrize("M,N,K", [(520, 776, 1024), (1024, 1024, 4096)])
def test_replays_of_a_captured_tail(M, N, K):
    g, L, q = H.rng(48), native.lib(), srt.current_queue()
    w = g.integers(-2, 3, (K, N)).astype(np.float32)
    inputs = [g.integers(-2, 3, (M, K)).astype(np.float32) for _ in range(3)]
    xt, wt, out = srt.Tensor(H.encode(inputs[0], H.F16)), srt.Tensor(H.encode(w, H.F16)), srt.Tensor(shape=[M, N], dtype=np.float16)
    sources = [srt.Tensor(H.encode(v, H.F16)) for v in inputs]
    (ad, k1), (bd, k2), (od, k3) = xt.descriptor(), wt.descriptor(), out.descriptor()
    a, b, o = xt.device_read(q), wt.device_read(q), out.device_read_write(q)

    def call():
        native.check(L.srtMatmul(a, ctypes.byref(ad), 0, b, ctypes.byref(bd), 0, o, ctypes.byref(od), q.stream))
    with H.pinned("mfma_256x256_m16_k64", H.F16, M, N, K, 25 | 64):
        call()                                              # loaded before the capture
    with H.pinned("mfma_256x256_m16_k64_tail", H.F16, M, N, K, 25 | 64):
        assert query_kernel(xt, False, wt, False, out) == "mfma_256x256_m16_k64_tail"
        call()
        graph, run = ctypes.c_void_p(), ctypes.c_void_p()
        assert L.hipStreamBeginCapture(q.stream, 1) == 0
        try:
            call()
        finally:
            assert L.hipStreamEndCapture(q.stream, ctypes.byref(graph)) == 0
        assert L.hipGraphInstantiate(ctypes.byref(run), graph, None, None, ctypes.c_size_t(0)) == 0
        for source, v in zip(sources, inputs):
            want = H.encode((v.astype(np.float64) @ w).astype(np.float32), H.F16)
            for again in (lambda: L.hipGraphLaunch(run, q.stream), call):
                q.copy(source, xt)
                q.fill(out, 0.0)
                again()
                out.device_written()
                assert np.array_equal(out.array(), want)
        assert L.hipGraphExecDestroy(run) == 0 and L.hipGraphDestroy(graph) == 0
