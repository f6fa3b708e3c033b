"""Results of 100 MB and more in long rows off whole 16-byte chunks, which the 256-wide tiles store past the caches at a short k against a k-contiguous
weight: both layouts of the left operand, rows inside a frame, odd and even pitches, a last row of tiles of a few rows, results either side of
the size.  Small integers: exact, and the frame untouched."""
import pytest

from tests import helpers as H
from tests.test_gpu_canaries import run_matmul_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt,M,N,K", [(H.BF16, 1032, 50003, 256), (H.F16, 3112, 16102, 320), (H.BF16, 3112, 16004, 64 * 15), (H.BF16, 1032, 48001, 256)])
@pytest.mark.parametrize("ta", [False, True])
def test_long_ragged_rows(tmp_path, dt, M, N, K, ta):
    plans = ("mfma_256x256_m16_k64", "mfma_256x256_m16") if M * N * K < 20e9 else ("mfma_256x256_m16_k64",)
    assert "mfma_256x256_m16_k64" in run_matmul_case(tmp_path, dt, M, N, K, 1, ta, True, plans, 960 + N + K, with_bias=not ta, relu=ta)
