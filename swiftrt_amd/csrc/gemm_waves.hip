// 16-bit matmul in tiles whose waves split k (gemm_waves.h): which tile a problem runs on, and what its time is taken to be.
#include "gemm_waves.h"

namespace srt {
namespace {

// Estimates in microseconds (256 units), fitted to 1900 random problems of 1-64 matrices, 1-8192 x 32-16384 x 32-8192, all layouts; a
// tile reads 128 K (32 x 32) or 256 K (64 x 64) bytes, an operand whose rows are off the 16-byte boundaries costs a sixth more, a third along m / n:
//   32 x 32   one tile a unit 3.4 + its bytes at 97 a ns; several 3.3 + each 0.26 + its bytes at 70
//   64 x 64   4.6 + bytes at 77; 4.4 + each 1.8 + bytes at 65.  (Several a unit, refitted to 400 problems of two slabs and more: with 2.9 and 59,
//             15 % low, k loops of three to eight slabs ran on them that 32 x 32 tiles finish sooner, us: 1280 x 784 x 312 x . W^T 8.6 / 6.0, 256 x 8320 x 320
//             13.4 / 9.8, 973 x 1088 x 174 7.2 / 5.6)
// Half of the estimates are within 6 %, 19 of 20 within 25 %; the better of the two by them is within 2 % of the better one on average.
double traffic(const GemmProblem& p) {
  const bool a_kc = p.sak == 1, b_kc = p.sbn != 1;
  auto off = [](const void* base, long long ld, long long batch) { return ((ld | batch) & 7) != 0 || (reinterpret_cast<uintptr_t>(base) & 15u) != 0; };
  double q = 1.0;
  if (off(p.A, a_kc ? p.sam : p.sak, p.sab)) q += a_kc ? 0.17 : 0.3;
  if (off(p.B, b_kc ? p.sbn : p.sbk, p.sbb)) q += b_kc ? 0.17 : 0.3;
  return q * (double)p.K;
}
double per_unit(const GemmProblem& p, int edge) {
  return (double)((p.M + edge - 1) / edge) * (double)((p.N + edge - 1) / edge) * (double)p.batch / compute_units();
}
double small_us(const GemmProblem& p) {
  const double tiles = per_unit(p, 32);
  double kb = 0.128 * traffic(p);
  // x^T . W past a short k: 64-byte pieces of both operands (32 x 32 / 64 x 64 tiles, us: 512 x 1280 x 8101 67 / 33, 704 x 1024 x 5769 44 / 23, 1578 x 384 x
  // 5776 51 / 28; 106 problems between 2048 and 8192 deep 1.1x)
  if (p.K >= 2048 && p.sak != 1 && p.sbn == 1 && p.M > 32 && p.N > 32) kb *= 1.5;
  return tiles <= 1.0 ? 3.4 + kb / 97.0 : 3.3 + tiles * (0.26 + kb / 70.0);
}
double large_us(const GemmProblem& p) {
  double tiles = per_unit(p, 64);
  const double kb = 0.256 * traffic(p);
  // long k loops: the first tiles past one a unit cost nearly a round (104 x 9152 x 4736 x^T . W^T, 286 tiles, 40 us; 229 problems measure 1.25 times the
  // estimate without this, 1.08 with it)
  if (p.K >= 2048 && tiles > 1.0 && tiles < 1.45) tiles = 1.45;
  return tiles <= 1.0 ? 4.6 + kb / 77.0 : 4.4 + tiles * (1.77 + kb / 65.0);
}

}  // namespace

bool waves_supported(const GemmProblem& p) {
  return (p.dtype == srtReal16BF || p.dtype == srtReal16F) && waves::fits(p);
}

double waves_us(const GemmProblem& p) {
  const double small = small_us(p), large = large_us(p);
  return small < large ? small : large;
}

hipError_t launch_waves(const GemmProblem& p, hipStream_t stream) {
  const bool bf16 = p.dtype == srtReal16BF;
  if (small_us(p) <= large_us(p) || waves::make_walk(p.M, p.N, p.batch, 64).tiles == 0)
    return bf16 ? waves::launch_layout<BF16, 1>(p, stream) : waves::launch_layout<F16, 1>(p, stream);
  return bf16 ? waves::launch_layout<BF16, 2>(p, stream) : waves::launch_layout<F16, 2>(p, stream);
}

}  // namespace srt
