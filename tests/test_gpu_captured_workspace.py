"""Plans with a workspace, captured into a graph: the block would be another tensor's by the time of a replay, so under capture they give way to
plans without one.  Every replay is exact, with the operands changed in between, and leaves the blocks of such a workspace's sizes alone."""
import ctypes
import os

import numpy as np
import pytest

import swiftrt_amd as srt
from swiftrt_amd import native
from tests import helpers as H
from tests.test_gpu_matmul import query_kernel

pytestmark = [pytest.mark.gpu, pytest.mark.skipif("debug" in os.environ.get("SWIFTRT_HIP_LIBRARY", ""),
                                                  reason="the debug build synchronises after every launch")]


@pytest.fixture(autouse=True)
def clean_cache():
    srt.PlanCache.clear()
    yield
    srt.PlanCache.clear()


def captured(q, call):
    """The graph of one call and its executable form."""
    L, graph, run = native.lib(), ctypes.c_void_p(), ctypes.c_void_p()
    assert L.hipStreamBeginCapture(q.stream, 1) == 0   # hipStreamCaptureModeThreadLocal; the runtime's symbols through the library that links it
    try:
        call()
    finally:
        assert L.hipStreamEndCapture(q.stream, ctypes.byref(graph)) == 0
    assert L.hipGraphInstantiate(ctypes.byref(run), graph, None, None, ctypes.c_size_t(0)) == 0
    return graph, run


# parts of k: half tiles (either layout of W), whole tiles, fp32; copies, whose second choice takes parts as well
@pytest.mark.parametrize("plan,dt,M,N,K,tb", [
    ("mfma_256x256_splitk", H.BF16, 128, 2048, 4096, False), ("mfma_256x256_splitk", H.F16, 128, 1024, 2048, True),
    ("mfma_256x256_splitk", H.BF16, 264, 520, 2048, False), ("f32_mfma_128x128_parts", H.F32, 256, 384, 2048, False),
    ("f32_mfma_128x128_parts", H.F32, 130, 260, 1024, True), ("copied", H.BF16, 128, 2048, 4160, False), ("copied", H.F32, 128, 512, 8224, False),
    ("copied", H.F32, 256, 1024, 4128, False)])
def test_replays_leave_other_tensors_alone(plan, dt, M, N, K, tb):
    g, L, q = H.rng(52), native.lib(), srt.current_queue()
    w = g.integers(-2, 3, (N, K) if tb else (K, N)).astype(np.float32)
    inputs = [g.integers(-2, 3, (M, K)).astype(np.float32) for _ in range(3)]
    wants = [H.encode((v.astype(np.float64) @ (w.T if tb else w)).astype(np.float32), dt) for v in inputs]
    xt, wt = srt.Tensor(H.encode(inputs[0], dt)), srt.Tensor(H.encode(w, dt))
    out = srt.Tensor(shape=[M, N], dtype=wants[0].dtype)
    sources = [srt.Tensor(H.encode(v, dt)) for v in inputs]
    (ad, k1), (bd, k2), (od, k3) = xt.descriptor(), wt.descriptor(), out.descriptor()
    a, b, o = xt.device_read(q), wt.device_read(q), out.device_read_write(q)

    def call():
        native.check(L.srtMatmul(a, ctypes.byref(ad), 0, b, ctypes.byref(bd), int(tb), o, ctypes.byref(od), q.stream))
    with H.pinned(plan, dt, M, N, K, 17 | (4 if tb else 8) | 64):
        assert query_kernel(xt, False, wt, tb, out) in (plan, "f32_mfma")
        call()
        assert np.array_equal(out.array(), wants[0])
        graph, run = captured(q, call)
        # what the allocator would hand the workspace's block to: tensors of its size (parts of M x N sums; the copies; the tiles' partials)
        held = [srt.Tensor(shape=[n], dtype=np.float32) for n in
                [parts * M * N for parts in (2, 4, 8, 16)] + [1 << s for s in range(16, 25)] for _ in range(2)]
        for t in held:
            q.fill(t, 7.0)
        for source, want in zip(sources, wants):
            for again in (lambda: L.hipGraphLaunch(run, q.stream), call):
                q.copy(source, xt)
                q.fill(out, 0.0)
                again()
                out.device_written()
                assert np.array_equal(out.array(), want)
        for t in held:
            assert np.all(t.array() == 7.0)
        assert L.hipGraphExecDestroy(run) == 0 and L.hipGraphDestroy(graph) == 0
