// Result tiles of 32 x 32, or 64 x 64 as 2 x 2 of them, whose waves split k: problems of few tiles, and operands off the
// 16-byte rules.  16-bit types (gemm_waves.hip) and fp32 (gemm_f32.hip).
//
// The direct-to-LDS kernels want a device's worth of 128 x 128 tiles or more; a problem of a few of them leaves units idle
// while each tile walks its whole k range.  Small tiles and a k range cut four or eight ways within the workgroup need neither a
// workspace nor a second launch.
//
//   bound   latency for one tile per unit: a round trip to memory, the k loop, the sums; beyond that the operand traffic of small
//           tiles from L2 (a 32 x 32 tile reads 64 rows of K; measured 97 bytes/ns a unit for one tile, 70 for several)
//   slab    128 bytes of k (64, or 32 of fp32) of a tile's rows per operand: whole lines of a k-contiguous operand.  A wave takes
//           the slabs w, w + waves, ..., requests the next one as soon as the last has left its registers for LDS and multiplies
//           meanwhile; its LDS is its own, so the k loop has no barrier.  (Two or three slabs in flight measured the same or
//           worse: more registers, fewer workgroups a unit.)
//   rows    start and end anywhere: the loads need element alignment only; a piece that would cross the end of a k row is loaded from
//           that row's last 16 bytes and shifted into place when it is stored to LDS, one that would cross K see Stage.
//           (Launch-sized problems fetch their code as they run: shifting a last slab's eight pieces took 0.7 us of 3.9)
//   layout  k-contiguous operand [rows][128 bytes], chunk c of row r at c ^ ((r >> 1) & 7): a fragment is one ds_read_b128;
//           mn-contiguous [k][mn]: two ds_read_b64_tr_b16, or four dwords of fp32
//   sums    fp32; the partial tiles meet in LDS and are added pairwise, in a fixed order
//   waves   eight while a unit has one tile, four when it has several (two to five workgroups then share a unit and
//           one's sums hide behind another's k loop): 32 x 256^3 x . W^T 11.7 us with eight, 7.4 with four
//   walk    an XCD's L2 holds the rows and columns of the tiles it has in flight when those are neighbours: 320 x 3759 x 3648
//           x . W 96 us in grid order, 45 by walk; 148 x 896 x 4672 12.3 and 10.0
//   measured (us, bf16: the kernels chosen before / now)   x . W 512 x 256 x 2560 16.7 / 6.5, 648 x 344 x 3032 40.9 / 10.4, 2816 x 384 x 1888
//           23.4 / 16.6, 1001^3 19.4 / 10.8; x^T . W 148 x 896 x 4672 16.7 / 12.2, 2024 x 472 x 704 13.0 / 7.5; x . W^T 16 x 744 x 84 x 704
//           12.1 / 10.0.  fp32 (8 waves, 16 k slabs, one pair at a time before) 512^3 6.1 / 5.6, 648 x 344 x 3032 26.9 / 22.4,
//           320 x 3759 x 3648 159 / 98
#pragma once
#include "gemm_common.h"
#include "walk.h"

namespace srt {
namespace waves {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
typedef short s16x4_t __attribute__((ext_vector_type(4)));
#define SRT_LDS __attribute__((address_space(3)))

// Number of multiplications of a fragment pair and the q-th of them: one of 16 k for a 16-bit type; fp32's 8 k take four (component q
// of a fragment is k 8 s + q in lanes 0-31 and 8 s + 4 + q in the others, the two k of a two-deep instruction).  `a` gives the
// rows of the instruction's result, `b` its columns.
template <typename T>
constexpr int kMfmas = sizeof(typename T::storage) == 2 ? 1 : 4;
template <typename T>
__device__ __forceinline__ f32x16_t mfma(u32x4_t a, u32x4_t b, int q, f32x16_t c) {
  if constexpr (T::dtype == srtReal16BF)
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
  else if constexpr (T::dtype == srtReal16F)
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x2f32(__builtin_bit_cast(f32x4_t, a)[q], __builtin_bit_cast(f32x4_t, b)[q], c, 0, 0, 0);
}

// v's elements s .. moved to the front, zeros behind them (s at least a vector's elements: all zeros)
template <int ES>
__device__ __forceinline__ u32x4_t shifted(u32x4_t v, int s) {
  if constexpr (ES == 2) {
    if (s & 4) v = u32x4_t{v[2], v[3], 0u, 0u};
    if (s & 2) v = u32x4_t{v[1], v[2], v[3], 0u};
    if (s & 1) v = u32x4_t{(v[0] >> 16) | (v[1] << 16), (v[1] >> 16) | (v[2] << 16), (v[2] >> 16) | (v[3] << 16), v[3] >> 16};
    if (s >= 8) v = u32x4_t{0u, 0u, 0u, 0u};
  } else {
    if (s & 1) v = u32x4_t{v[1], v[2], v[3], 0u};
    if (s & 2) v = u32x4_t{v[2], v[3], 0u, 0u};
    if (s >= 4) v = u32x4_t{0u, 0u, 0u, 0u};
  }
  return v;
}

// A slab: 128 bytes of k of 32 TILES rows (columns) of one operand, 16 bytes a lane and load.
// The last slab ends with K.  Its k are in pieces of 16 bytes, as a k-contiguous operand is loaded; the piece that would cross
// K, and those past it, are the row's last 16 bytes instead, with zeros for the k that have had their turn: no element changes its
// place in the piece, so the same zeros serve every row.  An mn-contiguous operand follows that order of k where the other one is
// k-contiguous (CHUNKED); otherwise its k rows past K repeat the last one, as zeros.
template <typename T, bool KC, int TILES, bool CHUNKED>
struct Stage {
  using S = typename T::storage;
  static constexpr int ES = (int)sizeof(S), EPC = 16 / ES;
  static constexpr int DEPTH = 128 / ES;                  // k of a slab
  static constexpr int LOADS = 4 * TILES, BYTES = 4096 * TILES;
  static constexpr int PER_ROW = KC ? 8 : 2 * TILES * ES;   // pieces of an LDS row ([rows][k] or [k][columns])
  static constexpr int ROWS = 64 / PER_ROW;                 // LDS rows a load fills
  static constexpr int PITCH = PER_ROW * 16;
  static constexpr uint32_t TOGGLE = KC ? 64 : (ES == 4 && TILES == 2) ? 128 : 0;   // swizzle of the odd loads

  const S* ptr[KC ? LOADS : 1];   // KC: the rows' start; MN: the piece's place in k row 0
  int k;                          // the piece's place in a slab
  int over;                       // MN: elements the piece was moved back to end inside its row
  uint32_t to, from;              // LDS offsets: where the first piece goes, where the lane's first fragment is
  uint32_t ld;
  int K;
  bool edge;                      // MN, workgroup-uniform: some piece crosses the rows' end

  // extent: M or N (MN: at least EPC; KC: K at least EPC)
  __device__ __forceinline__ void init(const S* base, int lane, int mn0, int extent, long long stride, int K_) {
    ld = (uint32_t)stride;   // (fits: below 2^31; the products below are one instruction each)
    K = K_;
    const int c = lane % PER_ROW, r = lane / PER_ROW;
    edge = !KC && mn0 + 32 * TILES > extent;
    if constexpr (KC) {
      k = c * EPC;
      over = 0;
      // (a row past the extent repeats the last one: it feeds results that are not stored)
#pragma unroll
      for (int i = 0; i < LOADS; ++i) ptr[i] = base + (uint64_t)(uint32_t)min(mn0 + r + 8 * i, extent - 1) * ld;
      to = (uint32_t)(r * 128 + ((c ^ (r >> 1)) << 4));   // chunk c of row r at c ^ ((r >> 1) & 7)
      const int fr = lane & 31, h = lane >> 5;
      from = (uint32_t)(fr * 128 + ((h ^ ((fr >> 1) & 7)) << 4));
    } else {
      k = r;
      const int mn = mn0 + c * EPC, at = min(mn, extent - EPC);
      over = mn - at;
      ptr[0] = base + at;
      if constexpr (ES == 2) {
        // chunk c of k row r at c, or c ^ 4 in every other pair of rows when a row is 128 bytes
        to = (uint32_t)(r * PITCH + ((TILES == 2 ? c ^ (((r >> 1) & 1) << 2) : c) << 4));
        // 16 lanes read a 4 (k) x 16 (mn) block, lane e * 4 + q of them 4 mn of k row e, and receive its transpose
        const int g = lane >> 4, e = (lane >> 2) & 3, q = lane & 3;
        const int kr = 8 * (g >> 1) + e, ch = 2 * (g & 1) + (q >> 1);
        from = (uint32_t)(kr * PITCH + ((TILES == 2 ? ch ^ (((kr >> 1) & 1) << 2) : ch) << 4) + (q & 1) * 8);
      } else {
        // a fragment's two half waves read k rows 4 apart: neighbours in LDS (128-byte rows), or with their halves
        // exchanged (256-byte rows), so that they meet different banks
        const int fr = lane & 31, h = lane >> 5;
        if constexpr (TILES == 1) {
          to = (uint32_t)((2 * (r & 3) + (r >> 2)) * PITCH + (c << 4));
          from = (uint32_t)(h * PITCH + fr * 4);
        } else {
          to = (uint32_t)(r * PITCH + (c << 4));
          from = (uint32_t)(4 * h * PITCH + ((fr * 4) ^ (h * 128)));
        }
      }
    }
  }
  __device__ __forceinline__ u32x4_t piece(const S* q) const {
    u32x4_t v;
    __builtin_memcpy(&v, q, 16);
    return v;
  }
  // MN, last slab: where the piece of load i is in k, and whether it counts
  __device__ __forceinline__ int last_row(int k0, int i, bool* counts) const {
    const int kk = k + ROWS * i;
    const int first = k0 + (CHUNKED ? kk & ~(EPC - 1) : kk);
    const int at = CHUNKED ? min(first, K - EPC) + (kk & (EPC - 1)) : min(first, K - 1);
    *counts = CHUNKED ? at >= first : first < K;
    return at;
  }
  // the slab that starts at k0 < K
  __device__ __forceinline__ void load(u32x4_t (&v)[LOADS], int k0) const {
    if constexpr (KC) {
      const int at = min(k0 + k, K - EPC);
#pragma unroll
      for (int i = 0; i < LOADS; ++i) v[i] = piece(ptr[i] + at);
    } else if (k0 + DEPTH <= K) {
      const S* q = ptr[0] + (uint64_t)(uint32_t)(k0 + k) * ld;
#pragma unroll
      for (int i = 0; i < LOADS; ++i) v[i] = piece(q + (uint64_t)(ROWS * i) * ld);
    } else {
#pragma unroll
      for (int i = 0; i < LOADS; ++i) {
        bool counts;
        v[i] = piece(ptr[0] + (uint64_t)(uint32_t)last_row(k0, i, &counts) * ld);
      }
    }
  }
  __device__ __forceinline__ void store(u32x4_t (&v)[LOADS], int k0, uint32_t lds) const {
    if constexpr (KC) {
      if (k0 + DEPTH > K) {
        const int had = k0 + k - (K - EPC);   // elements of the piece that have had their turn (a whole piece's or more: all)
        u32x4_t mask;
#pragma unroll
        for (int d = 0; d < 4; ++d)
          mask[d] = ES == 4 ? (d >= had ? ~0u : 0u) : (2 * d >= had ? ~0u : 2 * d + 1 >= had ? 0xffff0000u : 0u);
#pragma unroll
        for (int i = 0; i < LOADS; ++i) v[i] &= mask;
      }
    } else {
      if (edge) {
#pragma unroll
        for (int i = 0; i < LOADS; ++i) v[i] = shifted<ES>(v[i], over);
      }
      if (k0 + DEPTH > K) {
#pragma unroll
        for (int i = 0; i < LOADS; ++i) {
          bool counts;
          (void)last_row(k0, i, &counts);
          if (!counts) v[i] = u32x4_t{0u, 0u, 0u, 0u};
        }
      }
    }
#pragma unroll
    for (int i = 0; i < LOADS; ++i)
      *reinterpret_cast<SRT_LDS u32x4_t*>(lds + ((i & 1) ? to ^ TOGGLE : to) + (uint32_t)(i * 1024)) = v[i];
  }
  // fragment s (of four) of the slab's tile t
  __device__ __forceinline__ u32x4_t read(uint32_t lds, int t, int s) const {
    if constexpr (KC) {
      return *reinterpret_cast<const SRT_LDS u32x4_t*>(lds + (uint32_t)(t * 4096) + (from ^ (uint32_t)(s * 32)));
    } else if constexpr (ES == 2) {
      const uint32_t a = lds + (t ? from ^ 64u : from) + (uint32_t)(s * 16 * PITCH);
      const u32x2_t lo = __builtin_bit_cast(u32x2_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16(reinterpret_cast<SRT_LDS s16x4_t*>(a)));
      const u32x2_t hi =
          __builtin_bit_cast(u32x2_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16(reinterpret_cast<SRT_LDS s16x4_t*>(a + 4 * PITCH)));
      return u32x4_t{lo[0], lo[1], hi[0], hi[1]};
    } else {
      constexpr int STEP = TILES == 1 ? 2 * PITCH : PITCH;   // one k further
      const uint32_t a = lds + (t ? from ^ 128u : from) + (uint32_t)(s * 8 * PITCH);
      return u32x4_t{*reinterpret_cast<const SRT_LDS uint32_t*>(a), *reinterpret_cast<const SRT_LDS uint32_t*>(a + STEP),
                     *reinterpret_cast<const SRT_LDS uint32_t*>(a + 2 * STEP), *reinterpret_cast<const SRT_LDS uint32_t*>(a + 3 * STEP)};
    }
  }
};

__device__ __forceinline__ uint32_t quotient(uint32_t n, uint32_t d, uint32_t rcp) { return rcp ? __umulhi(n, rcp) : d == 1 ? n : n / d; }

// WALK: workgroups take tiles by `walk`; otherwise the grid is (columns, rows, matrices) of tiles.
template <typename T, bool A_KC, bool B_KC, int TILES, int WAVES, bool WALK>
__global__ __launch_bounds__(64 * WAVES) void gemm_waves_kernel(GemmProblem p, Walk walk) {
  using S = typename T::storage;
  using StageA = Stage<T, A_KC, TILES, A_KC || B_KC>;
  using StageB = Stage<T, B_KC, TILES, A_KC || B_KC>;
  constexpr int DEPTH = StageA::DEPTH, LOADS = StageA::LOADS, EDGE = 32 * TILES;
  constexpr int SLAB = StageA::BYTES + StageB::BYTES;       // a wave's share of LDS
  // fp32: two chains of sums a wave, eight or sixteen a result, each 16 ceil(ceil(K / 32) / WAVES) products long
  constexpr int CHAINS = sizeof(S) == 4 ? 2 : 1;
  extern __shared__ __attribute__((aligned(1024))) unsigned char waves_lds[];
  const uint32_t lds = (uint32_t)(uintptr_t)(SRT_LDS unsigned char*)waves_lds;

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int m0 = blockIdx.y * EDGE, n0 = blockIdx.x * EDGE, bz = blockIdx.z;
  if constexpr (WALK) {
    const uint32_t id = (blockIdx.x & 7) * walk.chunk + (blockIdx.x >> 3);
    if (id >= walk.tiles) return;
    const uint32_t line = quotient(id, walk.fast, walk.fast_rcp), fast = id - line * walk.fast;
    const uint32_t matrix = quotient(line, walk.slow, walk.slow_rcp), slow = line - matrix * walk.slow;
    m0 = (int)(walk.fast_is_m ? fast : slow) * EDGE;
    n0 = (int)(walk.fast_is_m ? slow : fast) * EDGE;
    bz = (int)matrix;
  }
  const uint32_t lds_a = lds + (uint32_t)(wave * SLAB), lds_b = lds_a + StageA::BYTES;

  StageA sa;
  StageB sb;
  sa.init((const S*)p.A + (long long)bz * p.sab, lane, m0, p.M, A_KC ? p.sam : p.sak, p.K);
  sb.init((const S*)p.B + (long long)bz * p.sbb, lane, n0, p.N, B_KC ? p.sbn : p.sbk, p.K);

  // The accumulators hold the tile's transpose (B's fragment goes first): a lane owns row l % 32 and four consecutive columns per
  // four registers.
  f32x16_t acc[TILES][TILES], more[TILES][TILES];
#pragma unroll
  for (int i = 0; i < TILES; ++i)
#pragma unroll
    for (int j = 0; j < TILES; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = more[i][j][v] = 0.0f;

  u32x4_t ra[LOADS], rb[LOADS];
  auto request = [&](int slab) {
    sa.load(ra, slab * DEPTH);
    sb.load(rb, slab * DEPTH);
  };
  auto place = [&](int slab) {
    sa.store(ra, slab * DEPTH, lds_a);
    sb.store(rb, slab * DEPTH, lds_b);
  };
  auto multiply = [&]() {
    // the slab is written and read by this wave only: LDS operations of one wave execute in order (the next slab's writes
    // behind this one's reads, too), so a wave-level fence (for the compiler) is all that is needed
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    // the fragments are read AHEAD steps before they are multiplied, as far as registers go (left to itself the compiler reads, waits and multiplies
    // step by step, an LDS latency each)
    constexpr int AHEAD = TILES == 1 && sizeof(S) == 2 ? 4 : 1;
    u32x4_t fa[4][TILES], fb[4][TILES];
    auto fetch = [&](int s) {
#pragma unroll
      for (int t = 0; t < TILES; ++t) {
        fa[s][t] = sa.read(lds_a, t, s);
        fb[s][t] = sb.read(lds_b, t, s);
      }
    };
#pragma unroll
    for (int s = 0; s < AHEAD; ++s) fetch(s);
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      if (s + AHEAD < 4) fetch(s + AHEAD);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int q = 0; q < kMfmas<T>; ++q)
#pragma unroll
        for (int i = 0; i < TILES; ++i)
#pragma unroll
          for (int j = 0; j < TILES; ++j) {
            f32x16_t& sum = CHAINS == 2 && (s & 1) ? more[i][j] : acc[i][j];
            sum = mfma<T>(fb[s][j], fa[s][i], q, sum);
          }
      if (AHEAD < 4) __builtin_amdgcn_sched_barrier(0);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  };

  // this wave's slabs: wave, wave + WAVES, ...
  const int slabs = (p.K + DEPTH - 1) / DEPTH;
  int s = wave;
  if (s < slabs) request(s);
  for (; s < slabs; s += WAVES) {
    place(s);
    // a slab's registers are free once it is in LDS: they take the wave's next slab before this one is multiplied
    if (s + WAVES < slabs) request(s + WAVES);
    multiply();
  }

  if constexpr (CHAINS == 2) {
#pragma unroll
    for (int i = 0; i < TILES; ++i)
#pragma unroll
      for (int j = 0; j < TILES; ++j) acc[i][j] += more[i][j];
  }
  // the waves' partial tiles meet in LDS ([wave][tile][32 rows][8 chunks of 4 columns], chunk c of row r at c ^ ((r >> 1) & 7))
  // and are added pairwise, in a fixed order
  __syncthreads();
  constexpr int TILE = 4096, PART = TILES * TILES * TILE;
  {
    const int r = lane & 31, h = lane >> 5;
    const uint32_t at = lds + (uint32_t)(wave * PART + r * 128 + ((h ^ ((r >> 1) & 7)) << 4));
#pragma unroll
    for (int i = 0; i < TILES; ++i)
#pragma unroll
      for (int j = 0; j < TILES; ++j)
#pragma unroll
        for (int g = 0; g < 4; ++g)
          *reinterpret_cast<SRT_LDS f32x4_t*>((at ^ (uint32_t)(g * 32)) + (uint32_t)((i * TILES + j) * TILE)) =
              f32x4_t{acc[i][j][4 * g], acc[i][j][4 * g + 1], acc[i][j][4 * g + 2], acc[i][j][4 * g + 3]};
  }
  __syncthreads();

  Epilogue<T> ep(p);
  S* C = (S*)p.C + (long long)bz * p.scb;
  // every lane has a share, two consecutive columns where eight waves finish one 32 x 32 tile: four columns of half the lanes were 0.2-0.4 us
  // more under libm's activations (fp32 7 x 64 x 72 x 64 x . W^T, tanh: 4.4 and 3.9)
  constexpr int COLS = EDGE * EDGE / 4 < 64 * WAVES ? 2 : 4, PIECES = EDGE / COLS;   // pieces of COLS columns in a row of the tile
  static_assert(EDGE * PIECES % (64 * WAVES) == 0, "whole rounds of the lanes");
  typedef float piece_t __attribute__((ext_vector_type(COLS)));
#pragma unroll
  for (int id = 0; id < EDGE * PIECES; id += 64 * WAVES) {
    const int q = id + tid;
    const int row = q / PIECES, c = q % PIECES * COLS, r = row & 31;
    const int m = m0 + row, n = n0 + c;
    if (m >= p.M || n >= p.N) continue;
    const uint32_t at = lds + (uint32_t)(((row >> 5) * TILES + (c >> 5)) * TILE + r * 128 + ((((c >> 2) & 7) ^ ((r >> 1) & 7)) << 4) + (c & 3) * 4);
    piece_t part[WAVES];
#pragma unroll
    for (int w = 0; w < WAVES; ++w) part[w] = *reinterpret_cast<const SRT_LDS piece_t*>(at + (uint32_t)(w * PART));
#pragma unroll
    for (int step = 1; step < WAVES; step *= 2)
#pragma unroll
      for (int w = 0; w < WAVES; w += 2 * step) part[w] += part[w + step];
    float out[COLS];
#pragma unroll
    for (int e = 0; e < COLS; ++e) out[e] = part[0][e];
    ep.finish_run(out, [&](int e, int* mm, int* nn) {
      *mm = m;
      *nn = n + e;
      return n + e < p.N;
    });
    S* dst = C + (long long)m * p.scm + (long long)n * p.scn;
    if (p.scn == 1 && n + COLS <= p.N) {   // one store, at whatever alignment the row has
      if constexpr (sizeof(S) == 2) {
        uint32_t w[COLS / 2];
#pragma unroll
        for (int e = 0; e < COLS; e += 2) w[e / 2] = T::template pack2<true>(out[e], out[e + 1]);
        __builtin_memcpy(dst, w, sizeof(w));
      } else {
        __builtin_memcpy(dst, out, sizeof(out));
      }
    } else {
#pragma unroll
      for (int e = 0; e < COLS; ++e)
        if (n + e < p.N) dst[(long long)e * p.scn] = T::from_float(out[e]);
    }
  }
}

// The launch: order of the tiles and number of waves by their count (above).
template <typename T, bool A_KC, bool B_KC, int TILES>
hipError_t launch(const GemmProblem& p, hipStream_t stream) {
  constexpr int EDGE = 32 * TILES, WAVE_LDS = TILES * 8192 > TILES * TILES * 4096 ? TILES * 8192 : TILES * TILES * 4096;
  const Walk walk = make_walk(p.M, p.N, p.batch, EDGE);
  auto go = [&](auto kernel, int waves, bool by_walk, std::atomic<uint32_t>& configured) {
    const int lds_bytes = waves * WAVE_LDS;
    if (hipError_t e = ensure_lds_limit(reinterpret_cast<const void*>(kernel), lds_bytes, configured); e != hipSuccess) return e;
    const dim3 grid = by_walk ? dim3(8 * walk.chunk) : dim3((p.N + EDGE - 1) / EDGE, (p.M + EDGE - 1) / EDGE, p.batch);
    hipLaunchKernelGGL(kernel, grid, dim3(64 * waves), lds_bytes, stream, p, walk);
    return launch_status(stream);
  };
  static std::atomic<uint32_t> configured[4];
  const bool several = walk.tiles > (uint32_t)compute_units();
  if constexpr (TILES == 1) {
    // operands of one XCD's L2 or less reach every unit in any order: the walk's arithmetic is 0.2 us for nothing
    const long long bytes = ((long long)p.M + p.N) * p.K * p.batch * (long long)sizeof(typename T::storage);
    const bool any_order = bytes <= (4LL << 20);
    if (!walk.tiles || (!several && any_order)) return go(gemm_waves_kernel<T, A_KC, B_KC, 1, 8, false>, 8, false, configured[0]);
    // (several tiles a unit and a k loop of two slabs: 2 x 720 x 344 x 48 4.16 us by walk, 3.43; longer ones share enough for it to pay,
    // 384 x 1052 x 1234 7.0 and 8.7)
    if (any_order && p.K <= 128) return go(gemm_waves_kernel<T, A_KC, B_KC, 1, 4, false>, 4, false, configured[3]);
  }
  if (several) return go(gemm_waves_kernel<T, A_KC, B_KC, TILES, 4, true>, 4, true, configured[1]);
  return go(gemm_waves_kernel<T, A_KC, B_KC, TILES, 8, true>, 8, true, configured[2]);
}
template <typename T, int TILES>
hipError_t launch_layout(const GemmProblem& p, hipStream_t stream) {
  const bool a_kc = p.sak == 1, b_kc = p.sbn != 1;
  if (a_kc && b_kc) return launch<T, true, true, TILES>(p, stream);
  if (a_kc) return launch<T, true, false, TILES>(p, stream);
  if (b_kc) return launch<T, false, true, TILES>(p, stream);
  return launch<T, false, false, TILES>(p, stream);
}

// Both operands have a unit stride, with at least one whole vector along it, and a pitch below 2^31; there is something to sum.
inline bool reads(const GemmProblem& p) {
  const int per = p.dtype == srtReal32F ? 4 : 8;
  if (p.K < 1) return false;
  if (p.sak == 1 ? p.K < per : (p.sam != 1 || p.M < per)) return false;
  if (p.sbn == 1 ? p.N < per : (p.sbk != 1 || p.K < per)) return false;
  const long long lda = p.sak == 1 ? p.sam : p.sak, ldb = p.sbn == 1 ? p.sbk : p.sbn;
  if (lda < 0 || lda > 0x7fffffffLL || ldb < 0 || ldb > 0x7fffffffLL) return false;
  return (p.M + 31) / 32 <= 65535 && p.batch <= 65535;
}
// And some grid holds the 32 x 32 tiles: the walk's, or (columns, rows, matrices) of them with eight waves each.
inline bool fits(const GemmProblem& p) {
  if (!reads(p)) return false;
  return make_walk(p.M, p.N, p.batch, 32).tiles != 0 || ((uint64_t)p.N + 31) / 32 * 512 <= kMostThreads;
}

}  // namespace waves
}  // namespace srt
