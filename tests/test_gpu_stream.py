"""The streaming kernel for a few rows against an n-contiguous weight (gemm_stream.hip): exact on integers, nothing outside a view, one set of bits
whichever workgroup adds the parts, every epilogue within one rounding, another kernel where k would be cut under capture."""
import ctypes
import os

import numpy as np
import pytest

import swiftrt_amd as srt
from swiftrt_amd import native
from tests import helpers as H
from tests.test_gpu_canaries import NAN_BITS, run_matmul_case

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def clean_cache():
    srt.PlanCache.clear()
    yield
    srt.PlanCache.clear()


# rows either side of a row tile; one strip, a strip's end inside a chunk, strips that take twelve, some and no parts; k of one step, inside and past a
# step, parts of two steps a wave, a k range with a last step of its own; rows at any alignment
@pytest.mark.parametrize("M,N,K,frame", [(1, 128, 32, (8, 8)), (16, 129, 33, (3, 2)), (17, 250, 63, (1, 0)), (32, 136, 95, (0, 0)), (8, 1000, 511, (3, 2)),
                                         (32, 2049, 512, (0, 0)), (3, 131, 4099, (3, 2)), (20, 1288, 3333, (0, 0)), (5, 16500, 520, (8, 8)), (31, 33001, 97, (1, 0))])
@pytest.mark.parametrize("dt", [H.BF16, H.F16])
def test_exact_inside_the_view(tmp_path, dt, M, N, K, frame):
    assert run_matmul_case(tmp_path, dt, M, N, K, 1, False, False, ("skinny",), 2100 + M + K, left=frame[0], right=frame[1], operand_sentinel=NAN_BITS,
                           with_bias=K % 2 == 0, relu=M % 2 == 0) == ["skinny"]


@pytest.mark.parametrize("M,N,K", [(8, 1536, 8000), (32, 4000, 2100), (32, 11008, 1096)])
def test_one_set_of_bits(M, N, K):
    g = H.rng(41)
    x, w = (srt.Tensor(H.encode(g.standard_normal(s), H.BF16)) for s in ((M, K), (K, N)))
    with H.pinned("skinny", H.BF16, M, N, K, 25 | 64) if K % 8 == 0 else H.pinned("skinny", H.BF16, M, N, K, 25):
        first = srt.matmul(x, w).array()
        for _ in range(40):
            assert np.array_equal(srt.matmul(x, w).array(), first)
    a, b = H.to64(x.array()), H.to64(w.array())
    assert H.elementwise_excess(H.decode(first), a @ b, np.abs(a) @ np.abs(b), H.BF16, K) <= 1.0


@pytest.mark.parametrize("act", list(srt.ActivationType))
def test_epilogues(act):
    M, N, K = 19, 777, 1100
    g = H.rng(43)
    x, w, b = (H.encode(g.standard_normal(s) / d, H.F16) for s, d in (((M, K), 8.0), ((K, N), 4.0), ((N,), 2.0)))
    with H.pinned("skinny", H.F16, M, N, K, 25, (1 | (int(act) << 1),)):
        got = H.to64(srt.Dense(srt.Tensor(w), srt.Tensor(b), act, relu_ceiling=1.5, elu_alpha=0.7)(srt.Tensor(x)).array())
    z = H.to64(x) @ H.to64(w) + H.to64(b)
    want = {"sigmoid": lambda: 1 / (1 + np.exp(-z)), "relu": lambda: np.maximum(z, 0), "tanh": lambda: np.tanh(z), "clippedRelu": lambda: np.clip(z, 0, 1.5),
            "elu": lambda: np.where(z > 0, z, 0.7 * np.expm1(z)), "identity": lambda: z}[act.name]()
    # one rounding to half (half a step: 2^-11 of the value), the sum's own error (1100 x 2^-24 x the products' magnitudes, under 40), the fast forms' 2^-14
    assert np.all(np.abs(got - want) <= (2.0 ** -11 + 2.0 ** -14) * np.abs(want) + 1100 * 2.0 ** -24 * 40)


@pytest.mark.skipif("debug" in os.environ.get("SWIFTRT_HIP_LIBRARY", ""), reason="the debug build synchronises after every launch")
def test_replays_of_a_captured_call():
    """A captured call takes no parts (a replay would find the last one's flags raised): every replay is exact, with the operands changed in between."""
    M, N, K = 8, 1024, 2056
    g, L, q = H.rng(47), native.lib(), srt.current_queue()
    w = g.integers(-2, 3, (K, N)).astype(np.float32)
    inputs = [g.integers(-2, 3, (M, K)).astype(np.float32) for _ in range(3)]
    xt, wt, out = srt.Tensor(H.encode(inputs[0], H.F16)), srt.Tensor(H.encode(w, H.F16)), srt.Tensor(shape=[M, N], dtype=np.float16)
    sources = [srt.Tensor(H.encode(v, H.F16)) for v in inputs]
    (ad, k1), (bd, k2), (od, k3) = xt.descriptor(), wt.descriptor(), out.descriptor()
    a, b, o = xt.device_read(q), wt.device_read(q), out.device_read_write(q)

    def call():
        native.check(L.srtMatmul(a, ctypes.byref(ad), 0, b, ctypes.byref(bd), 0, o, ctypes.byref(od), q.stream))
    with H.pinned("skinny", H.F16, M, N, K, 25 | 64):
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


def test_a_recorded_name_is_its_kernel():
    """The two plans of a few rows that cut k, told apart by the workspace they take: sixteen parts of M x N sums, eight of a strip's."""
    M, N, K = 32, 4096, 8192
    L, q = native.lib(), srt.current_queue()
    x, w = srt.Tensor(np.zeros((M, K), np.uint16)), srt.Tensor(np.zeros((K, N), np.uint16))
    out = srt.Tensor(shape=[M, N], dtype=np.uint16)

    def free():
        q.wait_for_completion()
        n, total = ctypes.c_size_t(), ctypes.c_size_t()
        assert L.hipMemGetInfo(ctypes.byref(n), ctypes.byref(total)) == 0
        return n.value

    def taken(plan):
        with H.pinned(plan, H.BF16, M, N, K, 25 | 64):
            q.matmul(x, False, w, False, out)   # kernels loaded, operands on the device
            q.wait_for_completion()
            native.check(L.srtDeviceEmptyCache())
            before = free()
            q.matmul(x, False, w, False, out)
            return before - free()
    assert taken("skinny") < 16 * M * N * 4 <= taken("mfma_256x256_splitk")


class KernelNode(ctypes.Structure):
    """hipKernelNodeParams."""
    _fields_ = [("block", ctypes.c_uint32 * 3), ("extra", ctypes.c_void_p), ("func", ctypes.c_void_p), ("grid", ctypes.c_uint32 * 3),
                ("params", ctypes.c_void_p), ("shared", ctypes.c_uint32)]


# k in one part already; parts, a weight past 50 MB in rows of a tile a unit: 64 columns a workgroup; parts, other weights: neither of the two
@pytest.mark.skipif("debug" in os.environ.get("SWIFTRT_HIP_LIBRARY", ""), reason="the debug build synchronises after every launch")
@pytest.mark.parametrize("M,N,K,groups", [(5, 16500, 520, 129), (8, 8712, 2880, 137), (32, 8200, 3080, 129), (8, 8184, 3080, None), (3, 12001, 2200, None),
                                          (17, 1024, 2056, None)])
def test_the_kernel_of_a_captured_call(M, N, K, groups):
    g, L, q = H.rng(48), native.lib(), srt.current_queue()
    x, w = (g.integers(-2, 3, s).astype(np.float32) for s in ((M, K), (K, N)))
    xt, wt, out = srt.Tensor(H.encode(x, H.BF16)), srt.Tensor(H.encode(w, H.BF16)), srt.Tensor(shape=[M, N], dtype=np.uint16)
    want = H.encode(x @ w, H.BF16)   # (sums below 2^24: exact in any order)
    (ad, k1), (bd, k2), (od, k3) = xt.descriptor(), wt.descriptor(), out.descriptor()
    a, b, o = xt.device_read(q), wt.device_read(q), out.device_read_write(q)

    def call():
        native.check(L.srtMatmul(a, ctypes.byref(ad), 0, b, ctypes.byref(bd), 0, o, ctypes.byref(od), q.stream))
    with H.pinned("skinny", H.BF16, M, N, K, 25 | (64 if K % 8 == 0 and N % 8 == 0 else 0)):
        call()
        out.device_written()
        assert np.array_equal(out.array(), want)
        graph, run = ctypes.c_void_p(), ctypes.c_void_p()
        assert L.hipStreamBeginCapture(q.stream, 1) == 0
        try:
            call()
        finally:
            assert L.hipStreamEndCapture(q.stream, ctypes.byref(graph)) == 0
    count, node, kernel = ctypes.c_size_t(1), ctypes.c_void_p(), KernelNode()
    assert L.hipGraphGetNodes(graph, None, ctypes.byref(count)) == 0 and count.value == 1
    assert L.hipGraphGetNodes(graph, ctypes.byref(node), ctypes.byref(count)) == 0
    assert L.hipGraphKernelNodeGetParams(node, ctypes.byref(kernel)) == 0
    if groups is None:
        assert tuple(kernel.grid)[0] not in ((N + 127) // 128, (N + 63) // 64)
    else:
        assert tuple(kernel.grid) == (groups, 1, 1)
    assert L.hipGraphInstantiate(ctypes.byref(run), graph, None, None, ctypes.c_size_t(0)) == 0
    for _ in range(3):
        q.fill(out, 0.0)
        assert L.hipGraphLaunch(run, q.stream) == 0
        out.device_written()
        assert np.array_equal(out.array(), want)
        call()
        out.device_written()
        assert np.array_equal(out.array(), want)
    assert L.hipGraphExecDestroy(run) == 0 and L.hipGraphDestroy(graph) == 0
