"""128 x 128 quarter tiles whose last 128-deep unit is ragged (gemm_mfma_m16q.h): exact, with NaN on every side of the operands' views."""
import pytest

import swiftrt_amd as srt
from tests import helpers as H
from tests.test_gpu_canaries import NAN_BITS, run_matmul_case

pytestmark = pytest.mark.gpu
QUARTER = "mfma_128x128_m16_k128"


@pytest.fixture(autouse=True)
def clean_cache():
    srt.PlanCache.clear()
    yield
    srt.PlanCache.clear()


# k one piece past a unit, one short of two, one past two, several units; a tile, edges either side of one, a batch whose matrices follow each other, more
# tiles than units (requests that run on into the next tile)
@pytest.mark.parametrize("M,N,K,batch", [(128, 128, 136, 1), (136, 248, 248, 1), (264, 120, 264, 3), (104, 392, 1000, 1), (2056, 2312, 392, 1), (40, 40, 520, 2)])
@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("dt", [H.BF16, H.F16])
def test_exact_between_nans(tmp_path, dt, M, N, K, batch, ta, tb):
    assert run_matmul_case(tmp_path, dt, M, N, K, batch, ta, tb, (QUARTER,), 2300 + M + K, operand_sentinel=NAN_BITS, with_bias=M % 16 == 0,
                           relu=N % 16 == 8) == [QUARTER]


# neither operand contiguous along k: any k at all
@pytest.mark.parametrize("M,N,K", [(136, 264, 129), (2048, 2304, 255), (128, 384, 385), (256, 128, 643)])
def test_any_k(tmp_path, M, N, K):
    assert run_matmul_case(tmp_path, H.BF16, M, N, K, 1, True, False, (QUARTER,), 2400 + K, operand_sentinel=NAN_BITS) == [QUARTER]
