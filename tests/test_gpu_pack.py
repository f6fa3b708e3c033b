"""Operands copied into aligned workspace (gemm_pack.hip) and results whose rows are not whole aligned 16-byte chunks.

Integer operands, exact comparison (every partial sum is representable, so the kernel and its order of summation do not
matter); operands framed by NaNs, results by a sentinel, so that a copy or a store past an edge shows."""
import ctypes
import os

import numpy as np
import pytest

import swiftrt_amd as srt
from swiftrt_amd import native
from tests import helpers as H
from tests.test_gpu_canaries import NAN_BITS, pin, run_matmul_case
from tests.test_gpu_matmul import query_kernel

pytestmark = pytest.mark.gpu

ANY = ("copied", "mfma_128x128_any", "mfma_64x64_any")   # the copies, and the kernels that stage the operands as they are


@pytest.fixture(autouse=True)
def clean_cache():
    srt.PlanCache.clear()
    yield
    srt.PlanCache.clear()


# k extents either side of a staging unit and of the rule's short ones; one and several tiles; each layout; a batch
@pytest.mark.parametrize("M,N,K,batch", [(129, 257, 129, 1), (127, 513, 257, 1), (65, 70, 1023, 1), (300, 333, 127, 1),
                                         (2049, 2047, 65, 1), (2047, 2050, 255, 1), (71, 131, 385, 5)])
@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
def test_copied_operands(tmp_path, M, N, K, batch, ta, tb):
    ran = run_matmul_case(tmp_path, H.BF16, M, N, K, batch, ta, tb, ANY, 900 + M + K, left=3, right=2, operand_sentinel=NAN_BITS)
    assert ran == list(ANY)


def test_copied_views_without_a_unit_stride_and_shared_matrices():
    g = H.rng(901)
    a = g.integers(-2, 3, (600, 900)).astype(np.float32)
    b = g.integers(-2, 3, (900, 800)).astype(np.float32)
    at, bt = srt.Tensor(H.encode(a, H.F16)), srt.Tensor(H.encode(b, H.F16))
    av, bv = at[1:599:2, 3:897:3], bt[2:896:3, 1:799:2]
    with H.pinned("copied", H.F16, 299, 399, 298, 16):
        got = srt.matmul(av, bv)
        assert query_kernel(av, False, bv, False, got) == "copied"
    want = a[1:599:2, 3:897:3].astype(np.float64) @ b[2:896:3, 1:799:2].astype(np.float64)
    assert np.array_equal(got.array(), H.encode(want.astype(np.float32), H.F16))
    # one right operand under every matrix of a batch (stride 0), odd extents
    x = g.integers(-2, 3, (6, 257, 301)).astype(np.float32)
    w = g.integers(-2, 3, (301, 515)).astype(np.float32)
    wt = srt.Tensor.repeating(srt.Tensor(H.encode(w, H.BF16)), [6, 301, 515])
    xt = srt.Tensor(H.encode(x, H.BF16))
    want = x.astype(np.float64) @ w.astype(np.float64)
    for plan in ("copied", "mfma_32x32_waves"):
        with H.pinned(plan, H.BF16, 257, 515, 301, 1 | 8 | 16, batch=6):
            got = srt.matmul(xt, wt)
            assert query_kernel(xt, False, wt, False, got) == plan
        assert np.array_equal(H.to64(got.array()), H.to64(H.encode(want.astype(np.float32), H.BF16))), plan


# aligned operands, an odd number of result columns: every kernel that stores such rows, edges of its tile in both directions
@pytest.mark.parametrize("dt", [H.BF16, H.F16])
@pytest.mark.parametrize("M,N,K,batch", [(256, 257, 256, 1), (136, 127, 384, 1), (264, 391, 512, 1), (72, 129, 256, 3)])
def test_results_with_ragged_rows(tmp_path, dt, M, N, K, batch):
    ran = set()
    for ta in (False, True):
        for bias, relu in ((False, False), (True, True), (True, False)):
            ran |= set(run_matmul_case(tmp_path, dt, M, N, K, batch, ta, True,
                                       ("mfma_256x256_m16_k64", "mfma_128x256_m16_k64", "mfma_256x128_m16_k64", "mfma_128x128_m16_k128",
                                        "mfma_128x128", "mfma_64x64"), 910 + N, with_bias=bias, relu=relu))
    assert ran == {"mfma_256x256_m16_k64", "mfma_128x256_m16_k64", "mfma_256x128_m16_k64", "mfma_128x128_m16_k128", "mfma_128x128",
                   "mfma_64x64"}


@pytest.mark.parametrize("act,coef", [("sigmoid", 0.0), ("tanh", 0.0), ("elu", 0.7), ("clippedRelu", 0.5)])
@pytest.mark.parametrize("dt", [H.BF16, H.F16])
def test_ragged_rows_under_every_activation(tmp_path, dt, act, coef):
    """The kernels' ragged and whole forms differ in how they store: the first 257 of 264 columns, bit for bit."""
    M, N, WIDE, K, code = 136, 257, 264, 512, srt.ActivationType[act]
    g = H.rng(940)
    for plan, ta in (("mfma_256x256_m16_k64", False), ("mfma_256x256_m16_k64", True), ("mfma_128x256_m16_k64", False),
                     ("mfma_256x128_m16_k64", True), ("mfma_128x128_m16_k128", False), ("mfma_128x128_m16_k128", True)):
        a = srt.Tensor(H.encode(g.standard_normal((K, M) if ta else (M, K)), dt))
        w, bias = H.encode(g.standard_normal((WIDE, K)) / 16, dt), H.encode(g.standard_normal(WIDE), dt)
        results = []
        for n in (N, WIDE):
            out, b = srt.Tensor(shape=[M, n], dtype=w.dtype), srt.Tensor(w[:n])
            pin(tmp_path, dt, M, n, K, 1, (2 if ta else 1) | 4 | 16 | (64 if n % 8 == 0 else 0), {10, 1 | (int(code) << 1)}, plan)
            assert query_kernel(a, ta, b, True, out) == plan
            srt.current_queue().matmul(a, ta, b, True, out, bias=srt.Tensor(bias[:n]), activation=code, coef=coef)
            results.append(out.array().view(np.uint16))
        assert np.array_equal(results[0], results[1][:, :N]), (plan, ta)


def test_the_choice_for_ragged_rows():
    for (M, N, K, kernel) in [(2048, 50257, 768, "mfma_256x256_m16_k64"), (512, 1001, 2048, "mfma_128x128_m16_k128"),
                              (128, 1809, 320, "mfma_32x32_waves"), (304, 630, 512, "mfma_64x64"),
                              (512, 1001, 200, "mfma_32x32_waves")]:
        a, b = srt.Tensor(shape=[M, K], dtype=np.uint16), srt.Tensor(shape=[N, K], dtype=np.uint16)
        assert query_kernel(a, False, b, True, srt.Tensor(shape=[M, N], dtype=np.uint16)) == kernel


# fp32 operands the 64-deep kernel reads only from a copy: k either side of its units, ragged rows and columns, each layout, a batch
@pytest.mark.parametrize("M,N,K,batch", [(1023, 2047, 1001, 1), (2049, 1155, 515, 1), (1500, 2050, 129, 1), (700, 1500, 1001, 2),
                                         (1200, 2000, 1004, 1)])
@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
def test_copied_fp32_operands(tmp_path, M, N, K, batch, ta, tb):
    ran = run_matmul_case(tmp_path, H.F32, M, N, K, batch, ta, tb, ("copied", "f32_mfma_64x64"), 920 + M + K, left=3, right=2,
                          operand_sentinel=NAN_BITS)
    assert ran == ["copied", "f32_mfma_64x64"]


def test_copied_fp32_views_without_a_unit_stride():
    g = H.rng(921)
    a = g.integers(-2, 3, (2100, 1100)).astype(np.float32)
    b = g.integers(-2, 3, (1100, 4100)).astype(np.float32)
    av, bv = srt.Tensor(a)[1:2051, 3:1099:2], srt.Tensor(b)[2:1098:2, 1:4097:2]
    got = srt.matmul(av, bv)
    assert query_kernel(av, False, bv, False, got) == "copied"
    want = a[1:2051, 3:1099:2].astype(np.float64) @ b[2:1098:2, 1:4097:2].astype(np.float64)
    assert np.array_equal(got.array(), want.astype(np.float32))


# device-filling and small 16-bit products, fp32: the choice is the copies, and a stream under capture gives them no workspace
@pytest.mark.parametrize("dt,M,N,K", [(H.BF16, 2049, 2051, 135), (H.F16, 2047, 2049, 257), (H.BF16, 1025, 1023, 1501),
                                      (H.F32, 1023, 2047, 1001)])
@pytest.mark.skipif("debug" in os.environ.get("SWIFTRT_HIP_LIBRARY", ""), reason="the debug build synchronises after every launch")
@pytest.mark.parametrize("ta,tb", [(False, False), (True, True)])
def test_without_workspace_the_operands_run_as_they_are(dt, M, N, K, ta, tb):
    g, L, q = H.rng(950), native.lib(), srt.current_queue()
    a = g.integers(-2, 3, (K, M) if ta else (M, K)).astype(np.float32)
    b = g.integers(-2, 3, (N, K) if tb else (K, N)).astype(np.float32)
    exact = (a.T if ta else a).astype(np.float64) @ (b.T if tb else b).astype(np.float64)
    want = H.encode(exact.astype(np.float32), dt)
    at, bt, out = srt.Tensor(H.encode(a, dt)), srt.Tensor(H.encode(b, dt)), srt.Tensor(shape=[M, N], dtype=want.dtype)
    assert query_kernel(at, ta, bt, tb, out) == "copied"
    (ad, k1), (bd, k2), (od, k3) = at.descriptor(), bt.descriptor(), out.descriptor()

    def call(stream):
        native.check(L.srtMatmul(at.device_read(q), ctypes.byref(ad), int(ta), bt.device_read(q), ctypes.byref(bd), int(tb),
                                 out.device_read_write(q), ctypes.byref(od), stream))
    for plan in ("mfma_128x128_any", "mfma_64x64_any", "f32_mfma_64x64", "f32_mfma_splitk"):   # loaded before the capture
        if (dt == H.F32) == plan.startswith("f32"):
            with H.pinned(plan, dt, M, N, K, (2 if ta else 1) | (4 if tb else 8) | 16):
                assert np.array_equal(srt.matmul(at, bt, ta, tb).array(), want), plan
    call(q.stream)                                                                 # eager: copied
    assert np.array_equal(out.array(), want)
    # hipStreamCaptureModeThreadLocal; the runtime's symbols through the library that links it
    graph, run = ctypes.c_void_p(), ctypes.c_void_p()
    assert L.hipStreamBeginCapture(q.stream, 1) == 0
    try:
        call(q.stream)
    finally:
        assert L.hipStreamEndCapture(q.stream, ctypes.byref(graph)) == 0
    assert L.hipGraphInstantiate(ctypes.byref(run), graph, None, None, ctypes.c_size_t(0)) == 0
    for _ in range(3):
        q.fill(out, 0.0)
        assert L.hipGraphLaunch(run, q.stream) == 0
        out.device_written()
        assert np.array_equal(out.array(), want)
        q.fill(out, 0.0)
        call(q.stream)                                                             # and eager between the replays
        assert np.array_equal(out.array(), want)
    assert L.hipGraphExecDestroy(run) == 0 and L.hipGraphDestroy(graph) == 0
