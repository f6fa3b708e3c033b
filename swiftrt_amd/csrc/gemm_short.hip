// 16-bit problems with short k loops on 128 x 128 tiles (gemm_short.h): where they run, and the launch.
#include "gemm_short.h"

namespace srt {

// Up to four slabs, or five and a half into rows off the 16-byte chunks, which the alternatives store by elements (a copy of the operands
// and the ring kernels' long epilogues, or 64 x 64 and 128 x 128 register-staged tiles).  Of 500 random problems, us, theirs / here:
// 4096 x 3701 x 32 x . W 32.2 / 12.9, 2772 x 2023 x 120 x^T . W 21.8 / 9.5, 1152 x 4864 x 78 13.3 / 7.7, 1088 x 8987 x 256 25.1 / 15.2, 8 x 832 x 839 x
// 264 24.8 / 13.7, 2368 x 4333 x 32 x . W^T 26.5 / 10.1, 4288 x 7769 x 104 62.3 / 28.3; past that they meet: 1031 x 12864 x 320 21.1 / 21.7,
// 3048 x 14608 x 346 63.5 / 66.7.
bool short_supported(const GemmProblem& p) {
  return !p.row_padding && shortk::fits(p) && (p.K <= 256 || (p.K <= 352 && p.N % 8 != 0));
}

// 4.6 + its slabs one after the other at 0.85, or a unit's tiles at 1.26 + 0.73 a slab; rms 10 % over the same problems.
double short_us(const GemmProblem& p) {
  const double tiles = (double)((p.M + 127) / 128) * (double)((p.N + 127) / 128) * (double)p.batch / compute_units();
  const double slabs = (p.K + 63) / 64, alone = 0.85 * slabs, shared = tiles * (1.26 + 0.73 * slabs);
  return 4.6 + (alone > shared ? alone : shared);
}

hipError_t launch_short(const GemmProblem& p, hipStream_t stream) {
  return p.dtype == srtReal16BF ? shortk::launch<BF16>(p, stream) : shortk::launch<F16>(p, stream);
}

}  // namespace srt
