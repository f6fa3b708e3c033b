"""128 x 128 tiles for short k loops (gemm_short.h): exact on integers, nothing outside a view, every epilogue within one rounding."""
import numpy as np
import pytest

import swiftrt_amd as srt
from tests import helpers as H
from tests.test_gpu_canaries import NAN_BITS, run_matmul_case

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def clean_cache():
    srt.PlanCache.clear()
    yield
    srt.PlanCache.clear()


# k inside a 16-byte piece, of a slab, one past it, four slabs, and past four into ragged rows; rows and columns either side of a tile,
# of a wave's quarter of one and of a chunk; a batch; more tiles than units; one row of tiles; aligned operands
@pytest.mark.parametrize("M,N,K,batch,frame", [(128, 128, 64, 1, (0, 0)), (129, 255, 65, 1, (3, 2)), (33, 161, 13, 1, (3, 2)), (97, 31, 200, 3, (0, 0)),
                                               (300, 9, 256, 1, (3, 2)), (1500, 3001, 70, 1, (1, 0)), (20, 5003, 129, 1, (3, 2)), (260, 301, 350, 1, (0, 0)),
                                               (2048, 2080, 40, 1, (8, 8)), (700, 1088, 61, 2, (0, 0)), (130, 8, 8, 2, (3, 2))])
@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("dt", [H.BF16, H.F16])
def test_exact_inside_the_view(tmp_path, dt, M, N, K, batch, frame, ta, tb):
    plans = ("mfma_128x128_any", "mfma_128x128") if frame == (8, 8) else ("mfma_128x128_any",)
    assert run_matmul_case(tmp_path, dt, M, N, K, batch, ta, tb, plans, 1700 + M + K, left=frame[0], right=frame[1], operand_sentinel=NAN_BITS,
                           with_bias=K % 2 == 0, relu=M % 2 == 0) == list(plans)


@pytest.mark.parametrize("act", list(srt.ActivationType))
@pytest.mark.parametrize("order", [srt.Order.row, srt.Order.col])
def test_epilogues(act, order):
    """By columns the bias is one of the kernel's rows; the activation is applied to fp32 sums and rounded once."""
    M, N, K = 700, 1003, 90
    g = H.rng(77)
    x, w, b = (g.standard_normal(s) / d for s, d in (((M, K), 3.0), ((K, N), 3.0), ((N,), 2.0)))
    xt, wt, bt = srt.Tensor(H.encode(x, H.BF16), order=order), srt.Tensor(H.encode(w, H.BF16), order=order), srt.Tensor(H.encode(b, H.BF16))
    shape = (M, N, K) if order == srt.Order.row else (N, M, K)
    layout = 25 if order == srt.Order.row else 1 | 8 | 16 | 32
    with H.pinned("mfma_128x128_any", H.BF16, *shape, layout, (1 | (int(act) << 1),)):
        got = H.to64(srt.Dense(wt, bt, act, relu_ceiling=1.5, elu_alpha=0.7)(xt).array())
    z = H.to64(H.encode(x, H.BF16)) @ H.to64(H.encode(w, H.BF16)) + H.to64(H.encode(b, H.BF16))
    want = {"sigmoid": lambda: 1 / (1 + np.exp(-z)), "relu": lambda: np.maximum(z, 0), "tanh": lambda: np.tanh(z), "clippedRelu": lambda: np.clip(z, 0, 1.5),
            "elu": lambda: np.where(z > 0, z, 0.7 * np.expm1(z)), "identity": lambda: z}[act.name]()
    # one rounding to bf16 (eight significant bits: half a step is at most 2^-8 of the value), the sum's own error (90 x 2^-24 x the
    # products' magnitudes, under 40) and the fast forms' 2^-14
    assert np.all(np.abs(got - want) <= (2.0 ** -8 + 2.0 ** -14) * np.abs(want) + 90 * 2.0 ** -24 * 40)


def test_tiles_along_the_rows():
    """Results of 32 Mi and more in rows of other than whole lines: every tile once, the last ones of either side partial.  Sums of 24 products of
    -1, 0 and 1 and a bias up to 3 are exact in bf16."""
    M, N, K = 2690, 12501, 24
    g = H.rng(31)
    x, w, b = g.integers(-1, 2, (M, K)), g.integers(-1, 2, (K, N)), g.integers(-3, 4, N)
    xt, wt, bt = (srt.Tensor(H.encode(v.astype(np.float64), H.BF16)) for v in (x, w, b))
    with H.pinned("mfma_128x128_any", H.BF16, M, N, K, 25, (1 | (int(srt.ActivationType.identity) << 1),)):
        got = srt.Dense(wt, bt, srt.ActivationType.identity)(xt).array()
    want = x.astype(np.float32) @ w.astype(np.float32) + b.astype(np.float32)
    assert np.array_equal(got, (want.view(np.uint32) >> 16).astype(np.uint16))


# k loops past the short kernel's, many tiles: the register-staged 128 x 128 tiles of the same two plans, off and on the 16-byte rules
@pytest.mark.parametrize("M,N,K,frame", [(2049, 2051, 353, (0, 0)), (2050, 2049, 396, (3, 2)), (1500, 3001, 369, (1, 0)), (2040, 2056, 264, (1, 2)),
                                         (2040, 2056, 392, (8, 8))])
@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
def test_longer_k_loops_on_register_staged_tiles(tmp_path, M, N, K, frame, ta, tb):
    plans = ("mfma_128x128_any", "mfma_128x128") if frame == (8, 8) else ("mfma_128x128_any",)
    assert run_matmul_case(tmp_path, H.BF16 if M % 2 else H.F16, M, N, K, 1, ta, tb, plans, 1900 + M + K, left=frame[0], right=frame[1],
                           operand_sentinel=NAN_BITS, with_bias=K % 2 == 0, relu=M % 2 == 0) == list(plans)
