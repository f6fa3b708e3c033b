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


@pytest.mark.parametrize("dt,M,N", [(H.F32, 700, 1000), (H.BF16, 4099, 264)])
def test_captured_bias_gradient(dt, M, N):
    """Its partial rows are the fixed array's under capture: the eager call's bits, and no other tensor is written."""
    g, L, q = H.rng(53), native.lib(), srt.current_queue()
    sources = [srt.Tensor(H.encode(g.standard_normal((M, N)), dt)) for _ in range(3)]
    y, dy = srt.Tensor(H.encode(g.standard_normal((M, N)), dt)), srt.Tensor(H.encode(g.standard_normal((M, N)), dt))
    dx, db, want_dx, want_db = (srt.Tensor(shape=s, dtype=H.NP_STORAGE[dt]) for s in ([M, N], [N]) * 2)

    def call(dx, db):
        q.activation_backward(y, dy, srt.ActivationType.tanh, 0.0, dx, db)
    call(dx, db)
    graph, run = captured(q, lambda: call(dx, db))
    held = [srt.Tensor(shape=[1 << s], dtype=np.float32) for s in range(12, 23) for _ in range(2)]
    held += [srt.Tensor(shape=[chunks * N], dtype=np.float32) for chunks in range(1, 257)]   # a row of sums a chunk of 16 rows or more
    for t in held:
        q.fill(t, 7.0)
    for source in sources:
        q.copy(source, dy)
        call(want_dx, want_db)
        q.fill(dx, 0.0)
        q.fill(db, 0.0)
        assert L.hipGraphLaunch(run, q.stream) == 0
        dx.device_written()
        db.device_written()
        assert dx.array().tobytes() == want_dx.array().tobytes() and db.array().tobytes() == want_db.array().tobytes()
    for t in held:
        assert np.all(t.array() == 7.0)
    assert L.hipGraphExecDestroy(run) == 0 and L.hipGraphDestroy(graph) == 0


def test_a_captured_pullback_is_refused_with_nothing_launched():
    g, L, q = H.rng(54), native.lib(), srt.current_queue()
    t = lambda *s: srt.Tensor(H.encode(g.standard_normal(s), H.F32))
    layer = srt.Dense(t(48, 64), t(64), srt.ActivationType.relu)
    x, dy = t(32, 48), t(32, 64)
    y = layer(x)
    dx, dw, db = (srt.Tensor(shape=s, dtype=np.float32) for s in ([32, 48], [48, 64], [64]))
    for out in (dx, dw, db):
        q.fill(out, 7.0)
    for tensor in (x, dy, layer.weight):
        tensor.device_read(q)

    def call():
        with pytest.raises(native.NotSupportedError):
            q.dense_backward(x, layer.weight, y, dy, int(layer.activation), 0.0, dx, dw, db)
    graph, run = captured(q, call)
    nodes = ctypes.c_size_t()
    assert L.hipGraphGetNodes(graph, None, ctypes.byref(nodes)) == 0 and nodes.value == 0
    for out in (dx, dw, db):
        assert np.all(out.array() == 7.0)
    assert L.hipGraphExecDestroy(run) == 0 and L.hipGraphDestroy(graph) == 0
