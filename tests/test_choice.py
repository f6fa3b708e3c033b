"""The kernel chosen where two are close: problems measured on both, by the kernel query."""
import ctypes

import pytest

from swiftrt_amd import native

BF16, F16, F32 = native.REAL16BF, native.REAL16F, native.REAL32F


def query(dt, M, N, K, ta=False, tb=False, batch=1):
    def descriptor(rows, columns):
        if batch == 1:
            return native.make_descriptor(dt, (rows, columns), (columns, 1), native.ORDER_ROW)
        return native.make_descriptor(dt, (batch, rows, columns), (rows * columns, columns, 1), native.ORDER_ROW)

    (ad, k1), (bd, k2), (od, k3) = descriptor(*((K, M) if ta else (M, K))), descriptor(*((N, K) if tb else (K, N))), descriptor(M, N)
    buf, p = ctypes.create_string_buffer(64), ctypes.c_void_p(256)
    assert native.lib().srtMatmulQueryKernel(ctypes.byref(ad), int(ta), ctypes.byref(bd), int(tb), ctypes.byref(od), p, p, p, buf, 64) == 0
    return buf.value.decode()


# us, copies / 128 x 128 tiles for short k loops
@pytest.mark.parametrize("dt,M,N,K,ta,tb,plan", [
    (BF16, 12191, 5312, 216, True, True, "copied"), (BF16, 8512, 9280, 143, True, True, "copied"),           # 54 / 67, 62 / 73
    (BF16, 2963, 9728, 256, True, True, "copied"), (F16, 9712, 8251, 256, False, False, "copied"),           # 29 / 35, 81 / 104
    (BF16, 6510, 5768, 256, True, True, "mfma_128x128_any"), (F16, 6562, 8768, 192, True, False, "mfma_128x128_any"),   # 48 / 42, 47 / 44
    (BF16, 4288, 7769, 104, False, True, "mfma_128x128"), (BF16, 2772, 2023, 120, True, False, "mfma_128x128_any")])   # 62 / 28, 22 / 9.5
def test_copies_and_short_k_loops(dt, M, N, K, ta, tb, plan):
    assert query(dt, M, N, K, ta, tb) == plan


# us, 64 x 64 tiles / wave-split ones: a handful of columns and one slab; columns that fill less than half of a 128 x 128 tile
@pytest.mark.parametrize("dt,batch,M,N,K,plan", [
    (F16, 48, 856, 8, 64, "mfma_64x64"), (BF16, 56, 960, 8, 64, "mfma_64x64"), (F16, 39, 848, 8, 8, "mfma_64x64"),   # 3.8 / 4.8, 5.0 / 6.8, 4.0 / 4.9
    (F16, 40, 976, 56, 32, "mfma_64x64")])                                                                           # 5.9 / 7.4
def test_narrow_batches(dt, batch, M, N, K, plan):
    assert query(dt, M, N, K, tb=True, batch=batch) == plan


# a few rows against an n-contiguous weight; us, streaming kernel / wave-split tiles
@pytest.mark.parametrize("dt,M,N,K,plan", [
    (BF16, 8, 9776, 6216, "skinny"), (BF16, 32, 11008, 4096 + 8, "skinny"), (F16, 16, 21760, 4123, "skinny"),    # 28 / 42, 22 / 33, 35 / 56
    (BF16, 32, 7096, 1992, "mfma_32x32_waves"), (BF16, 2, 3808, 3520, "mfma_32x32_waves"), (F16, 8, 17008, 960, "mfma_32x32_waves"),   # 12.8 / 8.7, 11.3 / 8.1, 11.0 / 8.9
    (BF16, 16, 19072, 1088, "skinny"), (BF16, 4, 3584, 10752, "skinny"),                                         # weights from memory: 12.6 / 15.4, 17 / 41
    (F16, 1, 6976, 3712, "mfma_32x32_waves"), (BF16, 2, 6784, 3784, "mfma_32x32_waves"),                          # out of the caches 13.2 / 9.9, 13.0 / 10.4
    (BF16, 8, 15784, 1792, "mfma_32x32_waves"), (BF16, 1, 15384, 2039, "mfma_32x32_waves")])                     # off whole lines: 16.2 / 11.4, 17.1 / 12.1
def test_a_few_rows(dt, M, N, K, plan):
    assert query(dt, M, N, K) == plan


# large weights in rows off whole lines, and the same in whole lines; us, streaming kernel / the other
@pytest.mark.parametrize("M,N,K,plan", [
    (8, 18072, 8128, "mfma_256x256_splitk"), (4, 14424, 12544, "mfma_256x256_splitk"), (8, 18048, 8128, "skinny"),          # 72 / 64, 75 / 63
    (8, 37432, 4024, "mfma_128x256_m16"), (32, 50888, 944, "mfma_128x256_m16"), (16, 50880, 944, "skinny"),                 # 84 / 61, 28 / 21
    (32, 91408, 1032, "mfma_128x256_m16"), (9, 129936, 392, "skinny"), (16, 41472, 3664, "skinny"),                         # 54 / 43, 32 / 43
    (32, 124344, 1984, "mfma_128x256_m16_k64"), (16, 124344, 1984, "skinny"), (8, 70008, 1608, "skinny")])                  # 118 / 94; three rounds of strips for two
def test_a_few_rows_off_whole_lines(M, N, K, plan):
    assert query(BF16, M, N, K) == plan


# a ragged last 128-deep unit, and tiles whose waves split k where quarter or half tiles would be padded; us, the plan before / this one
@pytest.mark.parametrize("dt,M,N,K,ta,tb,plan", [
    (BF16, 2048, 2048, 2008, True, False, "mfma_128x128_m16_k128"), (BF16, 1600, 2112, 1600, False, True, "mfma_128x128_m16_k128"),   # 43.8 / 20.9, 20.8 / 15.2
    (F16, 700, 3000, 400, False, False, "mfma_128x128_m16_k128"), (BF16, 2908, 624, 160, False, False, "mfma_128x256_m16"),          # 11.3 / 8.7; 7.8 (10.1 in quarters)
    (BF16, 1344, 760, 3008, False, False, "mfma_32x32_waves"), (F16, 1000, 1000, 1024, False, True, "mfma_32x32_waves"),            # 35.3 / 16.1
    (BF16, 1024, 1780, 448, True, True, "mfma_32x32_waves"), (F16, 2560, 674, 320, True, True, "mfma_32x32_waves"),                  # quarters 11.0 / 8.0, 10.8 / 8.2
    (BF16, 1688, 840, 7360, False, False, "mfma_128x128_m16_k128"), (F16, 1193, 1193, 5672, False, True, "mfma_128x128_m16_k128")])   # 50.6 (60.4 in wave-split tiles), 44.6 (56.4)
def test_depths_off_the_units(dt, M, N, K, ta, tb, plan):
    assert query(dt, M, N, K, ta, tb) == plan


# batches of few quarter tiles with a ragged last unit; us, these / the other
@pytest.mark.parametrize("dt,batch,M,N,K,tb", [
    (BF16, 9, 448, 704, 400, True), (F16, 42, 128, 544, 1416, False), (BF16, 3, 848, 832, 1672, True), (F16, 28, 769, 128, 1944, False)])   # 10.0 / 13.3, 29 / 29 (45 / 62 on new operands), 23 / 31, 33 / 40
def test_ragged_batches(dt, batch, M, N, K, tb):
    assert query(dt, M, N, K, tb=tb, batch=batch) == "mfma_128x128_m16_k128"
