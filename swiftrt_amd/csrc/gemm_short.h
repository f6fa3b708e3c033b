// 128 x 128 tiles of 16-bit problems with short k loops: the result's bytes are the work.
//
// A k loop of one to four 64-deep slabs is over before a ring of prefetched stages has filled, and a kernel that takes a whole
// compute unit has nothing else to run while its tile is stored: 64 x 512 x 512 x 64 x . W^T took 12.5 us for 42 MB.  Here a
// workgroup needs 33 KB of LDS and under 100 registers (one slab; 172 for more), so four (two or three) share a unit, and in a grid of
// several rounds one's stores run beside another's loads.  A grid of one round, as that one of four workgroups a unit, loads first and
// stores last: what it gained (12.5 -> 9.5 us) it gained with its operands in the caches.
//
//   bound   the result's stores, then the operands' loads (each XCD's L2 holds what its neighbouring tiles share: the walk of
//           gemm_waves.h)
//   slab    64 k of 128 rows and 128 columns, a quarter of each per wave (Stage of gemm_waves.h: any alignment, a masked last slab);
//           the next one is requested before this one is multiplied
//   wave    64 x 64 of the result, 2 x 2 tiles of 32 x 32, transposed: a lane owns four consecutive columns of a row
//   store   through LDS ([128 rows][16 chunks of 16 bytes], chunk c of row r at c ^ (r & 15)): 16 bytes a lane, whole rows of a tile
//   bias    in LDS from the start, so that the epilogue waits for no load
#pragma once
#include <type_traits>

#include "gemm_waves.h"

namespace srt {
namespace shortk {

constexpr int EDGE = 128, OPERAND = 4 * 4096, BIAS = 2 * OPERAND, LDS_BYTES = BIAS + EDGE * 4;

// ONE: a single slab, whose registers are free for the sums once it is in LDS: four workgroups a unit instead of two or three.
template <typename T, bool A_KC, bool B_KC, bool ONE>
__global__ __launch_bounds__(256, ONE ? 4 : 2) void gemm_short_kernel(GemmProblem p, waves::Walk walk) {
  using S = typename T::storage;
  using StageA = waves::Stage<T, A_KC, 1, A_KC || B_KC>;
  using StageB = waves::Stage<T, B_KC, 1, A_KC || B_KC>;
  constexpr int DEPTH = StageA::DEPTH, LOADS = StageA::LOADS;
  __shared__ __attribute__((aligned(1024))) unsigned char short_lds[LDS_BYTES];
  const uint32_t lds_a = (uint32_t)(uintptr_t)(SRT_LDS unsigned char*)short_lds, lds_b = lds_a + OPERAND;

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t id = (blockIdx.x & 7) * walk.chunk + (blockIdx.x >> 3);
  if (id >= walk.tiles) return;
  const uint32_t line = waves::quotient(id, walk.fast, walk.fast_rcp), fast = id - line * walk.fast;
  const uint32_t bz = waves::quotient(line, walk.slow, walk.slow_rcp), slow = line - bz * walk.slow;
  const int m0 = (int)(walk.fast_is_m ? fast : slow) * EDGE, n0 = (int)(walk.fast_is_m ? slow : fast) * EDGE;

  StageA sa;
  StageB sb;
  sa.init((const S*)p.A + (long long)bz * p.sab, lane, m0 + 32 * wave, p.M, A_KC ? p.sam : p.sak, p.K);
  sb.init((const S*)p.B + (long long)bz * p.sbb, lane, n0 + 32 * wave, p.N, B_KC ? p.sbn : p.sbk, p.K);
  const uint32_t my_a = lds_a + (uint32_t)(wave * 4096), my_b = lds_b + (uint32_t)(wave * 4096);

  waves::u32x4_t ra[LOADS], rb[LOADS];
  sa.load(ra, 0);
  sb.load(rb, 0);
  if (p.bias && tid < EDGE) {
    const int at = p.bias_per_row ? min(m0 + tid, p.M - 1) : min(n0 + tid, p.N - 1);
    *reinterpret_cast<SRT_LDS float*>(lds_a + (uint32_t)(BIAS + tid * 4)) = T::to_float(((const S*)p.bias)[(long long)at * p.sbias]);
  }

  const int wm = wave >> 1, wn = wave & 1;
  waves::f32x16_t acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.0f;

  const int slabs = ONE ? 1 : (p.K + DEPTH - 1) / DEPTH;
  for (int s = 0; s < slabs; ++s) {
    sa.store(ra, s * DEPTH, my_a);
    sb.store(rb, s * DEPTH, my_b);
    __syncthreads();
    if (!ONE && s + 1 < slabs) {
      sa.load(ra, (s + 1) * DEPTH);
      sb.load(rb, (s + 1) * DEPTH);
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      waves::u32x4_t fa[2], fb[2];
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        fa[t] = sa.read(lds_a + (uint32_t)((2 * wm + t) * 4096), 0, q);
        fb[t] = sb.read(lds_b + (uint32_t)((2 * wn + t) * 4096), 0, q);
      }
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = waves::mfma<T>(fb[j], fa[i], 0, acc[i][j]);
    }
    __syncthreads();
  }

  // accumulator register 4 g + e of tile (i, j): row 64 wm + 32 i + lane % 32, column 64 wn + 32 j + 8 g + 4 (lane / 32) + e
  const int r = lane & 31, h = lane >> 5;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int row = 64 * wm + 32 * i + r;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      float v[16];
#pragma unroll
      for (int e = 0; e < 16; ++e) v[e] = acc[i][j][e];
      if (p.bias) {
        if (p.bias_per_row) {
          const float b = *reinterpret_cast<const SRT_LDS float*>(lds_a + (uint32_t)(BIAS + row * 4));
#pragma unroll
          for (int e = 0; e < 16; ++e) v[e] += b;
        } else {
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            const waves::f32x4_t b = *reinterpret_cast<const SRT_LDS waves::f32x4_t*>(lds_a + (uint32_t)(BIAS + (64 * wn + 32 * j + 8 * g + 4 * h) * 4));
#pragma unroll
            for (int e = 0; e < 4; ++e) v[4 * g + e] += b[e];
          }
        }
      }
      if (p.activation != srtActivationIdentity) {
        auto each = [&](auto f) {
#pragma unroll
          for (int e = 0; e < 16; ++e) v[e] = f(v[e]);
        };
        switch (p.activation) {
          case srtActivationRelu: each([](float x) { return x > 0.0f ? x : 0.0f; }); break;
          case srtActivationSigmoid: each([](float x) { return activation16_ct<(int)srtActivationSigmoid>(0.0f, x); }); break;
          case srtActivationTanh: each([](float x) { return activation16_ct<(int)srtActivationTanh>(0.0f, x); }); break;
          default: each([&](float x) { return apply_activation_16(p.activation, p.coef, x); }); break;
        }
      }
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const uint32_t chunk = (uint32_t)(8 * wn + 4 * j + g);
        const waves::u32x2_t w = {T::template pack2<true>(v[4 * g], v[4 * g + 1]), T::template pack2<true>(v[4 * g + 2], v[4 * g + 3])};
        *reinterpret_cast<SRT_LDS waves::u32x2_t*>(lds_a + (uint32_t)(row * 256) + ((chunk ^ (uint32_t)(row & 15)) << 4) + (uint32_t)(8 * h)) = w;
      }
    }
  }
  __syncthreads();
  S* C = (S*)p.C + (long long)bz * p.scb;
  const int c = tid & 15, n = n0 + 8 * c;
  // rows of whole cache lines go past the caches, up to what those would hold of them in part (64 x 512 x 512 x 64 x . W^T 11.3 -> 10.8 us,
  // x 128 14.8 -> 12.6); lines that two tiles share must meet in L2 (1064-column rows lost a third)
  const bool stream = ((p.N | (int)p.scm | (int)p.scb) & 63) == 0 && (reinterpret_cast<uintptr_t>(p.C) & 127u) == 0 &&
                      (long long)p.M * p.N * p.batch <= (64LL << 20);
#pragma unroll
  for (int it = 0; it < 8; ++it) {
    const int row = 16 * it + (tid >> 4), m = m0 + row;
    if (m >= p.M || n >= p.N) continue;
    const waves::u32x4_t w = *reinterpret_cast<const SRT_LDS waves::u32x4_t*>(lds_a + (uint32_t)(row * 256 + ((c ^ (row & 15)) << 4)));
    S* dst = C + (long long)m * p.scm + n;
    if (stream) {
      __builtin_nontemporal_store(w, reinterpret_cast<waves::u32x4_t*>(dst));
    } else if (n + 8 <= p.N) {
      __builtin_memcpy(dst, &w, 16);
    } else {
#pragma unroll
      for (int e = 0; e < 7; ++e)
        if (n + e < p.N) dst[e] = (S)(w[e >> 1] >> (16 * (e & 1)));
    }
  }
}

// Unit strides along k or along m / n, as the wave-split tiles; the result's rows contiguous.
inline bool fits(const GemmProblem& p) {
  return (p.dtype == srtReal16BF || p.dtype == srtReal16F) && waves::reads(p) && p.scn == 1 && waves::make_walk(p.M, p.N, p.batch, EDGE).tiles != 0;
}

// Whether tiles that follow each other lie along the result's rows: where two of them share a line (rows of other than whole lines) and a
// column of tiles is long, the second half of a line otherwise comes a column later, when L2 has written the first half out.  us, down
// the columns / along the rows, bf16: 8192 x 9001 x 40 67.7 / 40.4, 8192 x 9001 x 64 x . W^T 68.3 / 39.9, 8192 x 12003 x 256 157 / 117, 7001 x 7400 x 33 40.7 /
// 27.6, 6100 x 9001 x 150 62.9 / 56.2, 4200 x 9001 x 40 25.2 / 22.6, 4 x 3000 x 3333 x 64 27.5 / 25.1, 6 x 3501 x 3502 x 64 54.2 / 39.6.  Fewer
// results stay in L2 either way, and down the columns neighbours do not write one line at a time: 3072 x 9001 x 150 31.6 / 33.7, 4000 x 4999 x
// 130 21.8 / 23.3, 2048 x 2049 x 40 7.5 / 8.2.  (Rows of whole lines share none: 8192^2 x 64 30.2 / 32.0, though 3712 x 16384 x 64 39.8 / 27.4.)
inline bool along_rows(const GemmProblem& p) {
  const bool whole_lines = ((p.N | (int)p.scm | (int)p.scb) & 63) == 0 && (reinterpret_cast<uintptr_t>(p.C) & 127u) == 0;
  return !whole_lines && p.M > 20 * EDGE && (long long)p.M * p.N * p.batch >= (32LL << 20);
}

template <typename T>
hipError_t launch(const GemmProblem& p, hipStream_t stream) {
  const waves::Walk walk = waves::make_walk(p.M, p.N, p.batch, EDGE, along_rows(p));
  const dim3 grid(8 * walk.chunk), block(256);
  const bool a_kc = p.sak == 1, b_kc = p.sbn != 1;
  auto layout = [&](auto one) {
    constexpr bool ONE = decltype(one)::value;
    if (a_kc && b_kc) hipLaunchKernelGGL((gemm_short_kernel<T, true, true, ONE>), grid, block, 0, stream, p, walk);
    else if (a_kc) hipLaunchKernelGGL((gemm_short_kernel<T, true, false, ONE>), grid, block, 0, stream, p, walk);
    else if (b_kc) hipLaunchKernelGGL((gemm_short_kernel<T, false, true, ONE>), grid, block, 0, stream, p, walk);
    else hipLaunchKernelGGL((gemm_short_kernel<T, false, false, ONE>), grid, block, 0, stream, p, walk);
  };
  if (p.K <= 64) layout(std::true_type{});
  else layout(std::false_type{});
  return launch_status(stream);
}

}  // namespace shortk
}  // namespace srt
