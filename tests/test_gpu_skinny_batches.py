"""The LDS-staged kernel for few rows against an n-contiguous weight (gemm_skinny.hip, its transposing read): batches, which are what it runs up to 32
rows of -- one matrix has a kernel of its own --, at every staged row count, N and K ending inside a group of columns and a block of k, between NaNs."""
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


@pytest.mark.parametrize("M,N,K,batch", [(1, 72, 8, 5), (8, 1000, 520, 2), (9, 136, 264, 3), (16, 64, 1032, 2), (17, 2056, 136, 2), (32, 328, 72, 4),
                                         (32, 40, 4096, 2)])
@pytest.mark.parametrize("dt", [H.BF16, H.F16])
def test_exact_between_nans(tmp_path, dt, M, N, K, batch):
    assert run_matmul_case(tmp_path, dt, M, N, K, batch, False, False, ("skinny",), 2300 + M + K, left=8, right=8, operand_sentinel=NAN_BITS,
                           with_bias=M % 2 == 0, relu=K % 16 == 0) == ["skinny"]
