// 16-bit matmul in 32 x 32 tiles whose eight waves split k: problems of few tiles.
//
// The direct-to-LDS kernels want a device's worth of 128 x 128 tiles; a problem of a few of them leaves units idle while each
// tile walks its whole k range, and operands off the 16-byte rules are copied first or staged element by element on the way.
// Small tiles and a k range cut eight ways within the workgroup need neither a workspace nor a second launch.
//
//   bound   latency: a round trip to memory per batch of slabs, then the operand traffic of small tiles (64 x K elements per
//           workgroup, at about 40 bytes/ns a unit) through L2
//   slab    32 k of 32 rows (columns) per operand and wave: 2 KiB, two 16-byte loads a lane; two slabs are requested at once and
//           multiplied as they arrive; a wave owns a contiguous eighth of K and its own LDS, so the k loop has no barrier
//   rows    start and end anywhere: the loads need element alignment only, and a piece that would cross a row's end is loaded
//           from the row's last eight elements and shifted into place when it is stored to LDS
//   layout  k-contiguous operand [32 rows][32 k], pitch 80 bytes: the MFMA operand (lane l: row l % 32, k = 8 (l / 32) .. + 7) is
//           one ds_read_b128; mn-contiguous [32 k][32 mn], 64 bytes per k row: two ds_read_b64_tr_b16, whose four k rows
//           per half wave are 256 contiguous bytes
//   sums    fp32; the eight partial tiles meet in LDS and are added pairwise, in a fixed order
//   measured (before / now, us, bf16, where this is the choice; before: 64 x 64 tiles, by 16-byte loads or any) x . W^T 136 x 448 x 576 8.4 /
//           3.8, 128 x 287 x 3376 27.8 / 7.5, 152 x 257 x 1529 21.6 / 6.2; x^T . W 128 x 440 x 656 18.5 / 3.9, 193 x 1535 x 2241 212 / 18;
//           x . W 32 x 2304 x 1469 31 / 5.2, 192 x 1537 x 2241 85 / 21, 128 x 113 x 8001 342 / 26
//   LDS     of the cycles it is busy, 24 % are bank conflicts with a k-contiguous operand (22 % with one of the two), none without
#include "gemm_common.h"

namespace srt {
namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
typedef short s16x4_t __attribute__((ext_vector_type(4)));
#define SRT_LDS __attribute__((address_space(3)))

constexpr int WAVES = 8, SLABS = 2, SK = 32;   // SK: k of a slab

template <typename T>
__device__ __forceinline__ f32x16_t mfma(u32x4_t a, u32x4_t b, f32x16_t c) {
  if constexpr (T::dtype == srtReal16BF)
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b), c, 0, 0, 0);
}

// v's eight elements s .. 7 moved to the front, zeros behind them (s >= 8: all zeros)
__device__ __forceinline__ u32x4_t shifted(u32x4_t v, int s) {
  if (s & 4) v = u32x4_t{v[2], v[3], 0u, 0u};
  if (s & 2) v = u32x4_t{v[1], v[2], v[3], 0u};
  if (s & 1) v = u32x4_t{(v[0] >> 16) | (v[1] << 16), (v[1] >> 16) | (v[2] << 16), (v[2] >> 16) | (v[3] << 16), v[3] >> 16};
  if (s >= 8) v = u32x4_t{0u, 0u, 0u, 0u};
  return v;
}

template <bool KC>
struct Stage {
  static constexpr int PITCH = KC ? 80 : 64;    // bytes of a slab's row in LDS
  static constexpr int BYTES = 32 * PITCH;
  const uint16_t* row[2];   // KC: the row's start; MN: the piece's place in k row 0
  int k[2];                 // the piece's place in a slab
  int over[2];              // MN: elements the piece was moved back to end inside its row
  uint32_t to[2], from;     // LDS offsets: where the pieces go, where the lane's operand is
  long long ld;
  int K, last_k;            // last_k: the largest k (MN) or piece start (KC) this wave may read
  bool edge;                // MN, workgroup-uniform: some piece crosses the rows' end

  // extent: M or N (MN: at least 8); k_end: where this wave's k range ends (KC: K at least 8)
  __device__ __forceinline__ void init(const uint16_t* base, int lane, int mn0, int extent, long long stride, int K_, int k_end) {
    ld = stride;
    K = K_;
    last_k = min(k_end, K_) - (KC ? 8 : 1);
    edge = !KC && mn0 + 32 > extent;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int f = lane + 64 * i;
      if (KC) {
        const int mn = f >> 2;
        k[i] = (f & 3) * 8;
        over[i] = 0;
        // (a row past the extent repeats the last one: it feeds results that are not stored)
        row[i] = base + (long long)min(mn0 + mn, extent - 1) * stride;
        to[i] = (uint32_t)(mn * PITCH + (f & 3) * 16);
      } else {
        const int mn = (f & 3) * 8;
        k[i] = f >> 2;
        const int at = min(mn0 + mn, extent - 8);
        over[i] = mn0 + mn - at;
        row[i] = base + at;
        to[i] = (uint32_t)(k[i] * PITCH + (f & 3) * 16);
      }
    }
    if (KC) {
      from = (uint32_t)((lane & 31) * PITCH + (lane >> 5) * 16);
    } else {
      // 16 lanes read a 4 (k) x 16 (mn) block, lane e * 4 + q of them 4 mn of k row e, and receive its transpose
      const int g = lane >> 4, e = (lane >> 2) & 3, q = lane & 3;
      from = (uint32_t)((8 * (g >> 1) + e) * PITCH + (16 * (g & 1) + 4 * q) * 2);
    }
  }
  __device__ __forceinline__ u32x4_t load(int i, int k0) const {
    const int at = min(k0 + k[i], last_k);
    u32x4_t v;
    __builtin_memcpy(&v, row[i] + (KC ? (long long)at : (long long)at * ld), 16);
    return v;
  }
  __device__ __forceinline__ void store(int i, int k0, u32x4_t v, uint32_t lds) const {
    if (KC) {
      if (k0 + SK > K) v = shifted(v, max(0, k0 + k[i] - (K - 8)));
    } else {
      if (edge) v = shifted(v, over[i]);
      if (k0 + SK > K && k0 + k[i] >= K) v = u32x4_t{0u, 0u, 0u, 0u};
    }
    *reinterpret_cast<SRT_LDS u32x4_t*>(lds + to[i]) = v;
  }
  // the operand of the MFMA of k 16 s .. 16 s + 15
  __device__ __forceinline__ u32x4_t read(uint32_t lds, int s) const {
    if constexpr (KC) {
      return *reinterpret_cast<const SRT_LDS u32x4_t*>(lds + from + s * 32);
    } else {
      const uint32_t a = lds + from + s * 16 * PITCH;
      const u32x2_t lo = __builtin_bit_cast(u32x2_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16(reinterpret_cast<SRT_LDS s16x4_t*>(a)));
      const u32x2_t hi =
          __builtin_bit_cast(u32x2_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16(reinterpret_cast<SRT_LDS s16x4_t*>(a + 4 * PITCH)));
      return u32x4_t{lo[0], lo[1], hi[0], hi[1]};
    }
  }
};

template <typename T, bool A_KC, bool B_KC>
__global__ __launch_bounds__(64 * WAVES) void gemm_waves_kernel(GemmProblem p) {
  using StageA = Stage<A_KC>;
  using StageB = Stage<B_KC>;
  constexpr int SLAB = StageA::BYTES + StageB::BYTES;   // a wave's share
  constexpr int RED = WAVES * 16 * 64 * 4;              // the waves' partial tiles, once every wave is done with its slabs
  constexpr int LDS = WAVES * SLAB > RED ? WAVES * SLAB : RED;
  __shared__ __attribute__((aligned(16))) unsigned char lds_raw[LDS];
  float(*red)[16][64] = reinterpret_cast<float(*)[16][64]>(lds_raw);

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 31, h = lane >> 5;
  const int m0 = blockIdx.y * 32, n0 = blockIdx.x * 32, bz = blockIdx.z;
  const uint32_t lds_a = (uint32_t)(uintptr_t)(SRT_LDS unsigned char*)lds_raw + (uint32_t)(wave * SLAB);
  const uint32_t lds_b = lds_a + StageA::BYTES;

  // this wave's slabs: a contiguous part of the k range
  const int slabs = (p.K + SK - 1) / SK;
  const int per_wave = (slabs + WAVES - 1) / WAVES;
  const int first = wave * per_wave;
  const int last = min(slabs, first + per_wave);   // exclusive

  StageA sa;
  StageB sb;
  sa.init((const uint16_t*)p.A + (long long)bz * p.sab, lane, m0, p.M, A_KC ? p.sam : p.sak, p.K, last * SK);
  sb.init((const uint16_t*)p.B + (long long)bz * p.sbb, lane, n0, p.N, B_KC ? p.sbn : p.sbk, p.K, last * SK);

  f32x16_t acc;
#pragma unroll
  for (int v = 0; v < 16; ++v) acc[v] = 0.0f;

  for (int s0 = first; s0 < last; s0 += SLABS) {
    u32x4_t ra[SLABS][2], rb[SLABS][2];
    // (slabs past the wave's range repeat its last piece: no branch between the loads)
#pragma unroll
    for (int s = 0; s < SLABS; ++s) {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        ra[s][i] = sa.load(i, (s0 + s) * SK);
        rb[s][i] = sb.load(i, (s0 + s) * SK);
      }
    }
#pragma unroll
    for (int s = 0; s < SLABS; ++s) {
      if (s0 + s >= last) break;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        sa.store(i, (s0 + s) * SK, ra[s][i], lds_a);
        sb.store(i, (s0 + s) * SK, rb[s][i], lds_b);
      }
      // the slab is written and read by this wave only: LDS operations of one wave execute in
      // order (the next slab's writes behind this one's reads, too), so a wave-level fence (for
      // the compiler) is all that is needed
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int q = 0; q < SK / 16; ++q) acc = mfma<T>(sa.read(lds_a, q), sb.read(lds_b, q), acc);
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
    }
  }

  __syncthreads();
#pragma unroll
  for (int v = 0; v < 16; ++v) red[wave][v][lane] = acc[v];
  __syncthreads();

  // wave w finishes accumulator registers 2 w and 2 w + 1; register v is row 8 (v / 4) + 4 h + v % 4, column r
  constexpr int R = 16 / WAVES;
  Epilogue<T> ep(p);
  const int n = n0 + r;
  if (n >= p.N) return;
  const int mb = m0 + 8 * (R * wave / 4) + 4 * h + (R * wave) % 4;
  float out[R];
#pragma unroll
  for (int i = 0; i < R; ++i) {
    float part[WAVES];
#pragma unroll
    for (int w = 0; w < WAVES; ++w) part[w] = red[w][R * wave + i][lane];
#pragma unroll
    for (int step = 1; step < WAVES; step *= 2)
#pragma unroll
      for (int w = 0; w < WAVES; w += 2 * step) part[w] += part[w + step];
    out[i] = part[0];
  }
  ep.finish_run(out, [&](int i, int* m, int* nn) {
    *m = mb + i;
    *nn = n;
    return *m < p.M;
  });
  typename T::storage* C = (typename T::storage*)p.C + (long long)bz * p.scb;
#pragma unroll
  for (int i = 0; i < R; ++i)
    if (mb + i < p.M) C[(long long)(mb + i) * p.scm + (long long)n * p.scn] = T::from_float(out[i]);
}

template <typename T>
hipError_t launch_as(const GemmProblem& p, hipStream_t stream) {
  const dim3 grid((p.N + 31) / 32, (p.M + 31) / 32, p.batch), block(64 * WAVES);
  const bool a_kc = p.sak == 1, b_kc = p.sbn != 1;
  if (a_kc && b_kc) hipLaunchKernelGGL((gemm_waves_kernel<T, true, true>), grid, block, 0, stream, p);
  else if (a_kc) hipLaunchKernelGGL((gemm_waves_kernel<T, true, false>), grid, block, 0, stream, p);
  else if (b_kc) hipLaunchKernelGGL((gemm_waves_kernel<T, false, true>), grid, block, 0, stream, p);
  else hipLaunchKernelGGL((gemm_waves_kernel<T, false, false>), grid, block, 0, stream, p);
  return launch_status(stream);
}

// Both operands have a unit stride, with at least one whole vector along it, and there is something to sum.
bool fits(const GemmProblem& p) {
  if (p.K < 1) return false;
  if (p.dtype != srtReal16BF && p.dtype != srtReal16F) return false;
  if (p.sak == 1 ? p.K < 8 : (p.sam != 1 || p.M < 8)) return false;
  if (p.sbn == 1 ? p.N < 8 : (p.sbk != 1 || p.K < 8)) return false;
  return (p.M + 31) / 32 <= 65535 && p.batch <= 65535;
}

}  // namespace

bool waves_supported(const GemmProblem& p) { return fits(p); }

// Whether these tiles are the choice, by two estimates in microseconds (256 units):
//   here     3 + rounds of a unit's tiles at 128 K bytes each: 60 bytes/ns up to 300 KB of a unit, 50 for one tile alone, 42 else;
//            0.55 a tile at least (its fill, sums and store).  Measured / estimated: 512 x 512 x 4096 10.8-14.2 / 13.5, 1024 x 1024 x
//            512 6.7 / 7.4, 1001^3 15.0 / 15.2, 1176 x 384 x 3280 22.2 / 23, 256 x 1344 x 7737 51-57 / 50, 32 x 256^3 9.3 / 9.2,
//            8 x 384 x 768 x 45 7.9 / 8.0
//   others   one round of 128 x 128 tiles, 5 + 5 per 1024 k, or split-K on a long k loop, 17 + 2.5 per 1024 k; + 5 for the copies of
//            operands off the 16-byte rules; 5 + 7 where k is in neither's units (register-staged tiles).  A lower bound:
//            more rounds cost more.  Measured / estimated: 512^3 7.2 / 7.5, 256 x 256 x 1024 9.5 / 10, 1001^3 17.7 / 14.9,
//            136 x 448 x 576 8.5-11.6 / 8.9, 1176 x 384 x 3280 34-66 / 27
// Problems the streaming kernel prefers, or long k loops it takes, stay with it (its rows of the weight arrive in whole lines: 64 x 2048 x 8192 x . W 19.6 there,
// 25.7 here; 2 x 7808 x 2304 x . W 9.9 and 12.2), and whole 128-deep units with the 128 x 128 tiles that
// read them: a matrix keeps the bits it has in a batch, where those are ahead (32 x 256^3 6.3 against 9.3).
bool waves_preferred(const GemmProblem& p) {
  if (p.row_padding || !fits(p)) return false;
  const double cus = compute_units(), k = (double)p.K / 1024.0, bytes = 128.0 * (double)p.K;
  const double tiles = (double)((p.M + 31) / 32) * (double)((p.N + 31) / 32) * (double)p.batch;
  const double rounds = __builtin_ceil(tiles / cus);
  const double rate = p.batch == 1 && rounds * bytes <= 300.0e3 ? 60.0e3 : rounds == 1.0 ? 50.0e3 : 42.0e3;
  const double tile_us = bytes / rate;
  const double here = 3.0 + rounds * (tile_us > 0.55 ? tile_us : 0.55);
  const double whole = 5.0 + 5.0 * k, cut = 17.0 + 2.5 * k;
  double others = whole < cut ? whole : cut;
  if (here >= others + 5.0 && here >= 5.0 + 7.0 * k) return false;   // (whatever the operands are)
  if (skinny_supported(p) && (skinny_preferred(p) || p.K >= 2048)) return false;
  if (mfma_config(p, 3) == 0) others += 5.0;
  else if (mfma_config(p, 14) != 0) return false;
  else if (mfma_splitk_parts(p) < 2) others = 5.0 + 7.0 * k;
  return here < others;
}

hipError_t launch_waves(const GemmProblem& p, hipStream_t stream) {
  return p.dtype == srtReal16BF ? launch_as<BF16>(p, stream) : launch_as<F16>(p, stream);
}

}  // namespace srt
