// Up to 32 rows against an n-contiguous weight, out[m, n] = sum_k x[m, k] * W[k, n], in 16-bit types: a decoding step through a Dense
// layer's own weight layout.
//
//   bound   reading W once.  A compute unit has about a hundred cache lines on their way at a time whatever asks for them (waves, loads in
//           flight, direct-to-LDS or not): 25-30 bytes a ns from memory, so every unit has to read, and 64 columns a workgroup over the
//           whole k range left 84 of 256 without work (N = 11008) or 192 (N = 4096).
//   split   strips of 128 columns, k in as many parts as give each unit one workgroup (stream_parts); 256 bytes of a k row a workgroup read 44 bytes
//           a ns a unit out of the caches where 128 read 32
//   W       straight to registers, no LDS: a lane's 16 bytes are 8 columns of one k row, rows 8 g + i of a step of 32 k for lane group g, so that
//           eight loads hold, column by column, the 8 consecutive k an MFMA operand wants: 32 v_perm_b32 put them in place.  Column
//           j of a lane is column 8 c + j of the strip: the j-th MFMA multiplies every eighth column, and a lane ends up with eight neighbouring results of a row.
//   sums    fp32; the four waves take every fourth step, their sums meet in LDS; the parts' in memory, added in the order of k by the workgroup that
//           finds all of them there (see Share), so the bits do not depend on timing
//   any     alignment of W, N and K: 16-byte loads at 2-byte boundaries; a strip's last lane moves back inside the row and computes, and stores, columns its
//           neighbour has too; the k that fill no step are one wave's, element by element of x
#include "gemm_common.h"
#include "status.h"

namespace srt {
namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));

template <typename T>
__device__ __forceinline__ f32x4_t mfma(u32x4_t a, u32x4_t b, f32x4_t c) {
  if constexpr (T::dtype == srtReal16BF)
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b), c, 0, 0, 0);
}

constexpr int STRIP = 128;    // columns of a strip: 16 lanes x 8
constexpr int BLOCK = 32;     // k of a step
constexpr int WAVES = 4;

// The parts of a strip leave their sums in memory and raise a flag; whichever finds the flags of all adds up.  Nobody waits: each stores its
// sums, waits for the acknowledgement, raises its flag, waits, and only then looks, so of two that finish together one sees the
// other, and if both do, both store the same bits.  Accesses are agent-scope (sc1); the mark is launch-unique (next_launch_epoch).
struct Share {
  float* partial;               // [strip][part][row tile][row of four][half of the columns][64 lanes][4]
  unsigned long long* flags;    // [strip][part]
  unsigned long long epoch;
  int parts;
};
constexpr int AGENT = 16;       // cache policy of a buffer access: sc1

template <typename T, int MT>
__global__ __launch_bounds__(64 * WAVES, 2) void gemm_stream_kernel(GemmProblem p, Share share) {
  using S = typename T::storage;
  constexpr int DEPTH = 2;   // steps in flight a wave (three or four: the same)
  __shared__ f32x4_t meet[WAVES * MT * 8 * 64];   // [wave][row tile][row of four][half of the columns][lane]
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int g = lane >> 4, c = lane & 15;
  const int strip = (int)blockIdx.x, part = (int)blockIdx.y;
  const int n = min(strip * STRIP + 8 * c, p.N - 8);   // the lane's eight columns
  const int blocks = (p.K + BLOCK - 1) / BLOCK, full = p.K / BLOCK;
  const int first = (int)((long long)blocks * part / share.parts), last = (int)((long long)blocks * (part + 1) / share.parts);

  const S* W = (const S*)p.B;
  const S* X = (const S*)p.A;
  const uint32_t w_lane = (uint32_t)(8 * g) * (uint32_t)p.sbk + (uint32_t)n;   // elements
  uint32_t x_lane[MT];   // (rows past M repeat the last one: they feed results that are not stored)
#pragma unroll
  for (int t = 0; t < MT; ++t) x_lane[t] = (uint32_t)min(16 * t + c, p.M - 1) * (uint32_t)p.sam + (uint32_t)(8 * g);

  // bias on its way from the start: read behind the parts' meeting it was a microsecond of latency (32 x 11008 x 4096 + bias + relu 22.9 -> 22.3 us)
  float bias[8], row_bias[MT];
#pragma unroll
  for (int q = 0; q < 8; ++q) bias[q] = p.bias && !p.bias_per_row ? T::to_float(((const S*)p.bias)[(long long)(n + q) * p.sbias]) : 0.0f;
#pragma unroll
  for (int t = 0; t < MT; ++t)
    row_bias[t] = p.bias && p.bias_per_row ? T::to_float(((const S*)p.bias)[(long long)min(16 * t + 4 * g + wave, p.M - 1) * p.sbias]) : 0.0f;

  struct Step {
    u32x4_t w[8];
    u32x4_t x[MT];
  };
  auto load = [&](int block, Step& s) __attribute__((always_inline)) {
    typedef u32x4_t unaligned_t __attribute__((aligned(2)));
    const S* wk = W + (long long)block * (BLOCK * p.sbk);
#pragma unroll
    for (int i = 0; i < 8; ++i)
      s.w[i] = __builtin_nontemporal_load(reinterpret_cast<const unaligned_t*>(wk + (long long)i * p.sbk + w_lane));
    const S* xk = X + block * BLOCK;
#pragma unroll
    for (int t = 0; t < MT; ++t) __builtin_memcpy(&s.x[t], xk + x_lane[t], 16);
  };

  f32x4_t acc[MT][8];
#pragma unroll
  for (int t = 0; t < MT; ++t)
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[t][j] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
  auto multiply = [&](const Step& s) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      u32x4_t f;
#pragma unroll
      for (int d = 0; d < 4; ++d)
        f[d] = __builtin_amdgcn_perm(s.w[2 * d + 1][j >> 1], s.w[2 * d][j >> 1], (j & 1) ? 0x07060302u : 0x05040100u);
#pragma unroll
      for (int t = 0; t < MT; ++t) acc[t][j] = mfma<T>(s.x[t], f, acc[t][j]);
    }
  };

  // steps first + wave, + 4, ...; the fences keep the loads of later steps ahead of a step's wait
  const int whole = min(last, full) - first;
  const int count = whole > wave ? (whole - wave + WAVES - 1) / WAVES : 0;
  auto block_at = [&](int j) { return first + wave + WAVES * j; };
  Step s[DEPTH];
  if (count >= DEPTH) {
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) {
      load(block_at(d), s[d]);
      __builtin_amdgcn_sched_barrier(0);
    }
    int j = 0;
    for (; j + 2 * DEPTH <= count; j += DEPTH) {
#pragma unroll
      for (int d = 0; d < DEPTH; ++d) {
        multiply(s[d]);
        __builtin_amdgcn_sched_barrier(0);
        load(block_at(j + DEPTH + d), s[d]);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    const int rest = count - j - DEPTH;
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) {
      multiply(s[d]);
      __builtin_amdgcn_sched_barrier(0);
      if (d < rest) load(block_at(j + DEPTH + d), s[d]);
    }
#pragma unroll
    for (int d = 0; d < DEPTH - 1; ++d)
      if (d < rest) multiply(s[d]);
  } else {
#pragma unroll
    for (int d = 0; d < DEPTH - 1; ++d)
      if (d < count) load(block_at(d), s[d]);
#pragma unroll
    for (int d = 0; d < DEPTH - 1; ++d)
      if (d < count) multiply(s[d]);
  }
  if (last > full && wave == (full - first) % WAVES) {   // the k that fill no step
    Step t;
    const int k0 = full * BLOCK + 8 * g;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      __builtin_memcpy(&t.w[i], W + (long long)min(k0 + i, p.K - 1) * p.sbk + n, 16);
      if (k0 + i >= p.K) t.w[i] = u32x4_t{0u, 0u, 0u, 0u};
    }
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      const S* row = X + (uint32_t)min(16 * m + c, p.M - 1) * (uint32_t)p.sam;
      uint32_t e[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) e[i] = k0 + i < p.K ? (uint32_t)row[k0 + i] : 0u;
      t.x[m] = u32x4_t{e[0] | (e[1] << 16), e[2] | (e[3] << 16), e[4] | (e[5] << 16), e[6] | (e[7] << 16)};
    }
    multiply(t);
  }

  // the waves' sums meet; wave w finishes rows 16 t + 4 g + w
#pragma unroll
  for (int t = 0; t < MT; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int h = 0; h < 2; ++h)
        meet[(((wave * MT + t) * 4 + r) * 2 + h) * 64 + lane] = f32x4_t{acc[t][4 * h][r], acc[t][4 * h + 1][r], acc[t][4 * h + 2][r], acc[t][4 * h + 3][r]};
  __syncthreads();
  float sum[MT][8];
#pragma unroll
  for (int t = 0; t < MT; ++t)
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      f32x4_t v[WAVES];
#pragma unroll
      for (int w = 0; w < WAVES; ++w) v[w] = meet[(((w * MT + t) * 4 + wave) * 2 + h) * 64 + lane];
#pragma unroll
      for (int q = 0; q < 4; ++q) sum[t][4 * h + q] = (v[0][q] + v[1][q]) + (v[2][q] + v[3][q]);
    }

  if (share.parts > 1) {
    constexpr int BYTES = MT * 8192;   // of a part's sums; the row tiles are 8192 apart, the rows of four 2048, the halves of the columns 1024
    const __amdgpu_buffer_rsrc_t mem = __builtin_amdgcn_make_buffer_rsrc(share.partial + (size_t)strip * share.parts * (BYTES / 4), 0,
                                                                         share.parts * BYTES, 0x00020000);
    const int at = wave * 2048 + lane * 16;
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const f32x4_t v = {sum[t][4 * h], sum[t][4 * h + 1], sum[t][4 * h + 2], sum[t][4 * h + 3]};
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_t, v), mem, part * BYTES + at + t * 8192 + h * 1024, 0, AGENT);
      }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();   // (every wave has read its share of `meet`, too)
    int* const verdict = reinterpret_cast<int*>(meet);
    if (wave == 0) {
      unsigned long long* flags = share.flags + (size_t)strip * share.parts;
      if (lane == 0) __hip_atomic_store(flags + part, share.epoch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      bool up = true;
      if (lane < share.parts) up = __hip_atomic_load(flags + lane, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == share.epoch;
      const bool all = __builtin_amdgcn_ballot_w64(!up) == 0;
      if (lane == 0) *verdict = all ? 1 : 0;
    }
    __syncthreads();
    if (!*verdict) return;
    for (int k = 0; k < share.parts; k += 4) {   // four parts' sums requested at a time
      u32x4_t v[4][MT][2];
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
          for (int h = 0; h < 2; ++h)
            v[u][t][h] = __builtin_amdgcn_raw_buffer_load_b128(mem, min(k + u, share.parts - 1) * BYTES + at + t * 8192 + h * 1024, 0, AGENT);
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        if (k + u >= share.parts) break;
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
          for (int q = 0; q < 8; ++q) {
            const float f = __builtin_bit_cast(f32x4_t, v[u][t][q >> 2])[q & 3];
            sum[t][q] = k + u == 0 ? f : sum[t][q] + f;
          }
      }
    }
  }

  Epilogue<T> ep(p);
  ep.bias = nullptr;
  S* C = (S*)p.C;
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    const int m = 16 * t + 4 * g + wave;
#pragma unroll
    for (int q = 0; q < 8; ++q) sum[t][q] += p.bias_per_row ? row_bias[t] : bias[q];
    ep.finish_run(sum[t], [](int, int*, int*) { return false; });
    if (m >= p.M) continue;
    u32x4_t out;
#pragma unroll
    for (int d = 0; d < 4; ++d) out[d] = T::template pack2<true>(sum[t][2 * d], sum[t][2 * d + 1]);
    __builtin_memcpy(C + (long long)m * p.scm + n, &out, 16);
  }
}

// Parts of the k range: one workgroup a unit.  us by parts: 32 x 11008 x 4096 (86 strips) 33.0, 22.3, 28.2, 24.5, 23.2 for 1-5 (three: two units have
// two workgroups and read half as fast for each), 8 x 9776 x 6216 (77) 50, 31.7, 28.1, 36.3, 8 x 4096 x 8192 (32) 51 for 1, 30 for 2, 19.4
// for 4, 16.7 for 8, 20.3 for 10.  A part is two steps a wave at least.
int stream_parts(const GemmProblem& p) {
  const int strips = (p.N + STRIP - 1) / STRIP, blocks = (p.K + BLOCK - 1) / BLOCK;
  int parts = compute_units() / strips;
  if (parts > 12) parts = 12;
  if (parts > blocks / (2 * WAVES)) parts = blocks / (2 * WAVES);
  return parts < 1 ? 1 : parts;
}

template <typename T, int MT>
hipError_t launch_rows(const GemmProblem& p, hipStream_t stream, bool whole) {
  const int strips = (p.N + STRIP - 1) / STRIP;
  Share share{};
  share.parts = whole ? 1 : stream_parts(p);
  void* workspace = nullptr;
  if (share.parts > 1) {
    const size_t flag_bytes = ((size_t)strips * share.parts * sizeof(unsigned long long) + 255) / 256 * 256;
    const size_t bytes = flag_bytes + (size_t)strips * share.parts * MT * 8192;
    if (hipError_t e = take_workspace(&workspace, bytes, stream); e != hipSuccess) return e;
    share.flags = reinterpret_cast<unsigned long long*>(workspace);
    share.partial = reinterpret_cast<float*>(static_cast<char*>(workspace) + flag_bytes);
    share.epoch = next_launch_epoch();
  }
  hipLaunchKernelGGL((gemm_stream_kernel<T, MT>), dim3(strips, share.parts), dim3(64 * WAVES), 0, stream, p, share);
  const hipError_t e = launch_status(stream);
  if (workspace) (void)srtDeviceFree(workspace);   // stream-ordered: reused only by work queued after the kernel
  return e;
}

}  // namespace

bool stream_supported(const GemmProblem& p) {
  if (p.dtype != srtReal16BF && p.dtype != srtReal16F) return false;
  if (p.batch != 1 || p.M < 1 || p.M > 32 || p.N < STRIP || p.K < BLOCK || p.row_padding) return false;
  if (p.sak != 1 || p.sbn != 1 || p.scn != 1 || p.sam < 0 || p.scm < 0 || p.sbk < p.N) return false;
  // the lanes' 32-bit offsets: a row of x or eight rows of W each
  return 32LL * p.sam + p.K < (1LL << 31) && 32LL * p.sbk + p.N < (1LL << 31);
}

// Microseconds, fitted to the same 2100 problems (rms 13 %): what a unit reads of W and x at 39 bytes a ns, or W from memory at 5.9 TB/s, behind a launch
// and, in parts, the parts' meeting.
double stream_us(const GemmProblem& p) {
  const int strips = (p.N + STRIP - 1) / STRIP, parts = stream_parts(p), cus = compute_units();
  const double a_unit = 0.256 * p.K * (1.0 + (p.sbk % 8 != 0 ? 0.42 : 0.0) + (p.sam % 8 != 0 ? 0.15 : 0.0)) * (p.M > 16 ? 1.25 : 1.0) / parts / 39.0 *
                        ((strips * parts + cus - 1) / cus);
  const double memory = 2.0 * p.N * p.K / 5.9e6;
  return (parts > 1 ? 7.0 : 3.3) + (p.M > 16 ? 0.7 : 0.0) + (a_unit > memory ? a_unit : memory);
}

hipError_t launch_stream(const GemmProblem& p, hipStream_t stream, bool whole) {
  const bool bf16 = p.dtype == srtReal16BF;
  if (p.M <= 16) return bf16 ? launch_rows<BF16, 1>(p, stream, whole) : launch_rows<F16, 1>(p, stream, whole);
  return bf16 ? launch_rows<BF16, 2>(p, stream, whole) : launch_rows<F16, 2>(p, stream, whole);
}

}  // namespace srt
