"""The forms of the tiles whose waves split k (gemm_waves.h) beyond one 32 x 32 tile a unit: several of them (four waves, tiles by
walk), 64 x 64 tiles of eight and of four waves, operands beyond one XCD's L2 -- exact on integers, nothing outside a view."""
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


# tiles either side of a unit's one, ragged in both directions; k of one slab, of one short of a round of the waves' slabs, of one
# past it and inside a 16-byte piece; a batch; one row of tiles (the walk's quotient by one)
@pytest.mark.parametrize("dt,M,N,K,batch", [
    (H.BF16, 520, 1030, 70, 1), (H.F16, 511, 545, 261, 1), (H.BF16, 70, 97, 195, 30), (H.F16, 31, 8300, 129, 1),   # 32 x 32, four waves
    (H.BF16, 1000, 1010, 530, 1), (H.F16, 130, 190, 1029, 20), (H.BF16, 65, 8200, 515, 1),                         # 64 x 64, eight waves
    (H.F16, 1100, 1090, 700, 1), (H.BF16, 2000, 700, 771, 1),                                                      # 64 x 64, four waves
    (H.BF16, 150, 900, 4100, 1),                                                                                   # 32 x 32 by walk
    (H.F32, 520, 545, 131, 1), (H.F32, 70, 97, 77, 30), (H.F32, 33, 8300, 30, 1), (H.F32, 150, 900, 2050, 1)])
@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
def test_every_form_is_exact_inside_its_view(tmp_path, dt, M, N, K, batch, ta, tb):
    plan = "f32_mfma_splitk" if dt == H.F32 else "mfma_32x32_waves"
    left, right = (3, 2) if N % 4 else (0, 0)
    assert run_matmul_case(tmp_path, dt, M, N, K, batch, ta, tb, (plan,), 1500 + M + K, left=left, right=right, operand_sentinel=NAN_BITS,
                           with_bias=M % 4 == 0) == [plan]


# a share of two columns a lane (eight waves finish a 32 x 32 tile) and of four; the last columns of a row inside a share
@pytest.mark.parametrize("act", list(srt.ActivationType))
@pytest.mark.parametrize("dt,M,N,K", [(H.BF16, 70, 97, 45), (H.F16, 520, 1030, 70), (H.BF16, 1000, 1010, 530), (H.F16, 1100, 1090, 700), (H.F32, 70, 99, 45),
                                      (H.F32, 520, 545, 131)])
def test_activations(act, dt, M, N, K):
    g = H.rng(79)
    x, w, b = (H.encode(g.standard_normal(s) / d, dt) for s, d in (((M, K), 3.0), ((K, N), 3.0), ((N,), 2.0)))
    with H.pinned("f32_mfma_splitk" if dt == H.F32 else "mfma_32x32_waves", dt, M, N, K, 25, (1 | (int(act) << 1),)):
        got = H.to64(srt.Dense(srt.Tensor(w), srt.Tensor(b), act, relu_ceiling=1.5, elu_alpha=0.7)(srt.Tensor(x)).array())
    x, w, b = H.to64(x), H.to64(w), H.to64(b)
    z = x @ w + b
    want = {"sigmoid": lambda: 1 / (1 + np.exp(-z)), "relu": lambda: np.maximum(z, 0), "tanh": lambda: np.tanh(z), "clippedRelu": lambda: np.clip(z, 0, 1.5),
            "elu": lambda: np.where(z > 0, z, 0.7 * np.expm1(z)), "identity": lambda: z}[act.name]()
    # one rounding of the result and the 16-bit types' fast forms (2^-14) or libm's few units in the last place; the sum's own error, which no
    # activation enlarges (slopes are at most 1), and fp32's exp(x) - 1
    relative = {H.BF16: 2.0 ** -8 + 2.0 ** -14, H.F16: 2.0 ** -11 + 2.0 ** -14, H.F32: 2.0 ** -21}[dt]
    assert np.all(np.abs(got - want) <= relative * np.abs(want) + (K + 1) * 2.0 ** -24 * (np.abs(x) @ np.abs(w) + np.abs(b)) + 2.0 ** -22)
