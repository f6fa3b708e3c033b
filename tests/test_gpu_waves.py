"""16-bit 32 x 32 tiles whose waves split k (gemm_waves.hip): rows that start and end anywhere.

Integer operands, exact comparison (every partial sum is representable, so the kernel and its order of summation do not
matter); operands framed by NaNs, results by a sentinel, so that a load or a store past an edge shows."""
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


# one whole vector along each dimension; k either side of a slab, of a wave's slabs and of the waves' whole range, one to seven
# elements past a vector; rows either side of a tile; fewer elements than a vector (not these tiles); the staging kernel beside them
@pytest.mark.parametrize("M,N,K,batch", [(8, 8, 8, 1), (9, 15, 13, 1), (31, 33, 31, 1), (32, 32, 32, 2), (34, 30, 34, 1), (33, 35, 255, 1),
                                         (64, 37, 261, 3), (66, 95, 515, 1), (10, 129, 518, 1), (97, 12, 70, 1), (70, 41, 1039, 1),
                                         (40, 40, 7, 1), (5, 70, 100, 1)])
@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("left,right", [(0, 0), (3, 2)])
@pytest.mark.parametrize("dt", [H.BF16, H.F16])
def test_rows_of_any_extent_and_alignment(tmp_path, dt, M, N, K, batch, ta, tb, left, right):
    ran = run_matmul_case(tmp_path, dt, M, N, K, batch, ta, tb, ("mfma_32x32_waves", "mfma_64x64_any"), 800 + M + K, left=left,
                          right=right, operand_sentinel=NAN_BITS, with_bias=M % 2 == 0)
    whole_vectors = (M if ta else K) >= 8 and (K if tb else N) >= 8
    assert ran == (["mfma_32x32_waves", "mfma_64x64_any"] if whole_vectors else ["mfma_64x64_any"])


@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("dt", [H.BF16, H.F16])
def test_an_empty_sum_is_the_bias(dt, ta, tb):
    """K = 0: nothing is read, every element of the result is written."""
    M, N = 40, 72
    T = srt.Tensor
    bias = T(H.encode(np.arange(N) - 30.0, dt))
    a, b = T(shape=[0, M] if ta else [M, 0], dtype=bias.dtype), T(shape=[N, 0] if tb else [0, N], dtype=bias.dtype)
    for with_bias, want in ((False, np.zeros((M, N))), (True, np.maximum(np.tile(np.arange(N) - 30.0, (M, 1)), 0.0))):
        out = T(H.encode(np.full((M, N), 5.0), dt))
        srt.current_queue().matmul(a, ta, b, tb, out, bias=bias if with_bias else None,
                                   activation=srt.ActivationType.relu if with_bias else None)
        assert np.array_equal(H.to64(out.array()), want), with_bias
