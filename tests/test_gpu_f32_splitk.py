"""fp32 32 x 32 tiles whose waves split k: 16-byte loads of rows that start and end anywhere.

Integer operands, exact comparison (every partial sum is representable, so the kernel and its order of summation do not
matter); operands framed by NaNs, results by a sentinel, so that a load or a store past an edge shows."""
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


# one whole vector along each dimension; k either side of a slab, of a wave's slabs and of the waves' whole range; rows either
# side of a tile; fewer elements than a vector (the kernel that reads by elements)
@pytest.mark.parametrize("M,N,K,batch", [(4, 4, 4, 1), (5, 7, 6, 1), (31, 33, 15, 1), (32, 32, 16, 2), (34, 30, 17, 1),
                                         (33, 35, 255, 1), (64, 37, 257, 3), (66, 95, 259, 1), (3, 129, 515, 1), (97, 2, 70, 1),
                                         (40, 40, 3, 1)])
@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("left,right", [(0, 0), (3, 2)])
def test_rows_of_any_extent_and_alignment(tmp_path, M, N, K, batch, ta, tb, left, right):
    ran = run_matmul_case(tmp_path, H.F32, M, N, K, batch, ta, tb, ("f32_mfma_splitk",), 700 + M + K, left=left, right=right,
                          operand_sentinel=NAN_BITS, with_bias=M % 2 == 0)
    assert ran == ["f32_mfma_splitk"]
