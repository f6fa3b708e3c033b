// Operands that miss the matrix-core kernels' 16-byte rules, copied once into aligned, zero-padded workspace.
//
// An odd extent or pitch, a base off a 16-byte boundary, or a view without a unit stride keeps an operand away from the
// direct-to-LDS kernels: what is left stages through registers with loads at 2-byte alignment (under half the aligned rate)
// or element by element, and transposes mn-contiguous operands on the way.  2048 x 50257 x 768 x . W ran at 180 TFLOP/s that
// way.  A copy moves each operand once -- bytes that grow with M K + K N where the product's work grows with M N K -- and
// leaves rows on 128-byte lines and the k extent in whole staging units (zeros up to there), so the product itself runs on
// the kernel its shape deserves.
//
//   bound     memory: every element read and written once; both operands in one launch (a launch is about 3 us here)
//   layout    the operand keeps its orientation (rows along its unit stride; a view without one takes its smaller stride as
//             the row), rows padded to a multiple of 64 elements, zero behind the extent; k is padded to the unit of the
//             kernel that will read it (pack_depth), as zero columns or zero rows
//   lanes     one 16-byte chunk of the copy each, two per lane a workgroup apart (four / two, the whole product, us: 512 x 11007 x 4096 88.5 /
//             87.4, 8191^3 794 / 786, the rest within a percent)
#include "gemm_common.h"
#include "status.h"

namespace srt {
namespace {

constexpr int kChunksPerLane = 2;
// Copies that fit the last-level cache (256 MiB) better if their sources stay out of it read the sources with the streaming hint, so that the product
// finds the copies there.  What the hint is worth, by megabytes of copies, in passes that follow each other over three sets of operands / in the first
// pass over new ones, 410 random problems: single matrices 50-75 0.983 / 0.992, 75-100 0.992 / 1.013, 100-130 1.01 / 1.025, 130-160 1.00 / 1.046,
// 160-200 1.01 / 1.07, 200-270 1.04 / 1.065, 270-300 1.01 / 1.01, beyond 0.99 / 0.985; batches 75-130 0.957 / 0.987, 130-160 0.97 / 1.02, 160-200 0.98 / 1.025,
// 200-270 1.01 / 1.02: two rows share lines that the hint drops, most where batches have short ones (40 x 1920 x 384 x 767 x . W^T, 142 MB, 120 us
// without it, 160).  2048 x 50257 x 768 (77 MB) 190 / 191 us, the first pass over new operands 214 / 203; x . W^T 2048 x 768 x 50257 (283 MB) 484 / 425.
constexpr size_t kStreamedFrom = 75000000, kStreamedBatchFrom = 160000000, kStreamedTo = 290000000;
// The copies of a call take at most this much, in blocks of a power of two: the allocator keeps a freed block for the next call of
// its size, so calls of many odd shapes share a dozen blocks instead of leaving one each (two operands that the 256 x 256 kernels'
// 32-bit offsets reach are 4 GiB; larger ones run as they are).
constexpr size_t kCopiesMost = (size_t)4 << 30;

struct PackJob {
  const void* src;
  void* dst;
  long long ld, inner, batch;   // element strides of the source: between rows, along a row, between matrices
  uint32_t rows, rows_out;      // rows of a matrix that exist / that are written
  uint32_t cols, chunks;        // elements of a row that exist; 16-byte chunks of a row of the copy
  uint32_t total;               // chunks of the copy (0: nothing to do)
};

template <int ES>
struct Element;
template <>
struct Element<2> { using type = uint16_t; };
template <>
struct Element<4> { using type = uint32_t; };

template <int ES, bool STREAM>
__global__ __launch_bounds__(256) void pack_kernel(PackJob a, PackJob b, uint32_t blocks_a) {
  using E = typename Element<ES>::type;
  constexpr uint32_t PER = 16 / ES;   // elements of a chunk
  const bool first = blockIdx.x < blocks_a;
  const PackJob& j = first ? a : b;
  const uint32_t base = (first ? blockIdx.x : blockIdx.x - blocks_a) * (256 * kChunksPerLane) + threadIdx.x;
#pragma unroll
  for (int u = 0; u < kChunksPerLane; ++u) {
    const uint32_t id = base + (uint32_t)u * 256;
    if (id >= j.total) break;
    const uint32_t line = id / j.chunks, c = id - line * j.chunks;
    const uint32_t bz = line / j.rows_out, row = line - bz * j.rows_out;
    union { E e[PER]; uint4 v; } x;
    x.v = uint4{0u, 0u, 0u, 0u};
    const uint32_t col = c * PER;
    if (row < j.rows && col < j.cols) {
      const E* src = (const E*)j.src + (long long)bz * j.batch + (long long)row * j.ld + (long long)col * j.inner;
      const uint32_t n = j.cols - col;
      if (j.inner == 1 && n >= PER) {
        if constexpr (STREAM) {
          typedef uint32_t words_t __attribute__((ext_vector_type(4), aligned(2)));   // (from any element's address)
          const words_t w = __builtin_nontemporal_load(reinterpret_cast<const words_t*>(src));
          __builtin_memcpy(&x, &w, 16);
        } else {
          __builtin_memcpy(&x, src, 16);
        }
      } else {
#pragma unroll
        for (uint32_t e = 0; e < PER; ++e)
          if (e < n) x.e[e] = src[(long long)e * j.inner];
      }
    }
    ((uint4*)j.dst)[id] = x.v;
  }
}

inline bool aligned16(const void* ptr) { return (reinterpret_cast<uintptr_t>(ptr) & 15u) == 0; }
inline long long round_up(long long v, long long unit) { return (v + unit - 1) / unit * unit; }

// The k extent of the copies: whole 128-deep units where one round of 128 x 128 tiles holds the problem, else whole 64-deep
// ones; short k loops (no such kernel) in whole 64-deep units too, which the register-staged kernels read.
int pack_depth(const GemmProblem& p) {
  if (p.dtype == srtReal32F) return p.K <= 128 ? 128 : (int)round_up(p.K, 64);   // gemm_f32_ring.h: whole 64-deep units, two at least
  const long long t128 = (long long)((p.M + 127) / 128) * ((p.N + 127) / 128) * p.batch;
  const bool quarter = t128 <= compute_units() && p.K > 128;
  const long long k = round_up(p.K, quarter ? 128 : 64);
  return (int)(quarter && k < 256 ? 256 : k);
}

// One operand as the copies' problem wants it: element (mn, k) at base[mn * s_mn + k * s_k].  Fills the job and the new
// strides; a job without chunks leaves the operand where it is.
struct Operand {
  const void* base;
  long long s_mn, s_k, s_batch;
};
size_t plan_operand(Operand* o, int extent, int K, int depth, int batch, int es, PackJob* job) {
  *job = PackJob{};
  const int per = 16 / es;
  const bool fits = aligned16(o->base) && depth == K && o->s_batch % per == 0;
  if (fits && o->s_k == 1 && (o->s_mn % per == 0 || extent == 1)) return 0;
  if (fits && o->s_mn == 1 && extent % per == 0 && o->s_k % per == 0) return 0;
  const bool along_k = o->s_k == 1 || (o->s_mn != 1 && o->s_k <= o->s_mn);
  const int matrices = o->s_batch == 0 ? 1 : batch;   // one copy of a matrix that every batch shares
  const long long pitch = along_k ? depth : round_up(extent, 64);
  job->src = o->base;
  job->ld = along_k ? o->s_mn : o->s_k;
  job->inner = along_k ? o->s_k : o->s_mn;
  job->batch = o->s_batch;
  job->rows = (uint32_t)(along_k ? extent : K);
  job->rows_out = (uint32_t)(along_k ? extent : depth);
  job->cols = (uint32_t)(along_k ? K : extent);
  job->chunks = (uint32_t)(pitch / per);
  const long long elements = (long long)matrices * job->rows_out * pitch;
  if (elements / per > 0x7fffffffLL) return ~(size_t)0;
  job->total = (uint32_t)(elements / per);
  o->s_mn = along_k ? pitch : 1;
  o->s_k = along_k ? 1 : pitch;
  o->s_batch = o->s_batch == 0 ? 0 : (long long)job->rows_out * pitch;
  return (size_t)elements * es;
}

struct PackPlan {
  GemmProblem q;      // the problem over the copies, once their addresses are filled in
  PackJob a, b;
  size_t bytes_a, bytes_b;
  size_t at_b() const { return (bytes_a + 255) / 256 * 256; }   // B's copy follows A's
  size_t workspace() const {
    size_t block = 256;
    while (block < at_b() + bytes_b) block *= 2;
    return block;
  }
};
bool plan_pack(const GemmProblem& p, PackPlan* t) {
  if (p.dtype != srtReal16BF && p.dtype != srtReal16F && p.dtype != srtReal32F) return false;
  if (p.scn != 1 || p.scm < 0 || p.K < 1 || p.batch > 65535) return false;
  if (p.sam < 0 || p.sak < 0 || p.sab < 0 || p.sbk < 0 || p.sbn < 0 || p.sbb < 0) return false;
  const int depth = pack_depth(p), es = p.dtype == srtReal32F ? 4 : 2;
  Operand a{p.A, p.sam, p.sak, p.sab}, b{p.B, p.sbn, p.sbk, p.sbb};
  t->bytes_a = plan_operand(&a, p.M, p.K, depth, p.batch, es, &t->a);
  t->bytes_b = plan_operand(&b, p.N, p.K, depth, p.batch, es, &t->b);
  if (t->bytes_a == ~(size_t)0 || t->bytes_b == ~(size_t)0) return false;
  t->q = p;
  t->q.K = depth;
  t->q.sam = a.s_mn; t->q.sak = a.s_k; t->q.sab = a.s_batch;
  t->q.sbn = b.s_mn; t->q.sbk = b.s_k; t->q.sbb = b.s_batch;
  t->q.row_padding = 1;
  if (t->bytes_a) t->q.A = nullptr;   // (workspace: aligned)
  if (t->bytes_b) t->q.B = nullptr;
  return t->bytes_a + t->bytes_b != 0 && t->workspace() <= kCopiesMost;
}

}  // namespace

bool pack_supported(const GemmProblem& p) {
  PackPlan t;
  return !p.row_padding && plan_pack(p, &t) && (p.dtype != srtReal32F || f32_ring_fits(t.q));
}

double packed_us(const GemmProblem& p) {
  PackPlan t;
  if (p.dtype != srtReal32F || p.row_padding || !plan_pack(p, &t) || !f32_ring_fits(t.q)) return 0.0;
  return 5.0 + (double)(t.bytes_a + t.bytes_b) / 3.0e6 + (double)p.batch * p.M * p.N * 4.0 / 8.0e6 + f32_ring_us(t.q);
}

// Whether copying 16-bit operands pays (fp32: f32_any_choice in gemm_f32.hip): always once the problem fills the device with
// 128 x 128 tiles; below that by two estimates in microseconds.
//   as it is   4 + its 64-deep stages at 1.0 (both operands contiguous along k), 2.5 (B along n) or 5 (A along m, or views
//              without a unit stride), once per 512 tiles of 64 x 64
//   copied     8 for the extra launch and the wait between the two, the copies' bytes at 6 TB/s, and a round of 128 x 128
//              tiles (5 + 5 per 1024 k)
// measured (as it is / copied): 1001^3 x . W^T 20.2 / 20.3, x . W 67.6 / 20.3, x^T . W 105.6 / 20.6; 300 x 500 x 700 12.8 / 16.2,
// 34.1 / 16.4, 70.6 / 16.6; 129 x 513 x 257 x . W^T 9.1 / 14.0, x^T . W 24.7 / 14.2; 32 x 255^3 x . W^T 14.2 / 20.4, x . W 32.5 / 20.3;
// 8 x 14336 x 4095 x . W^T 73 / 61; 2047 x 2049 x 2047 64.5 / 41.3, 193 / 41.5, 298 / 42.7; 4095 x 4097 x 4099 343 / 160, 725 / 163,
// 1520 / 177; 2048 x 50257 x 768 x . W 880 / 186 (34 of them the copy of W).
bool pack_preferred(const GemmProblem& p) {
  PackPlan t;
  if (p.dtype == srtReal32F || p.row_padding || !plan_pack(p, &t)) return false;
  auto tiles = [&](int s) { return (double)((p.M + s - 1) / s) * ((p.N + s - 1) / s) * p.batch; };
  const double cus = compute_units();
  if (tiles(128) >= cus) return true;
  const double per_stage = p.sak == 1 ? (p.sbk == 1 ? 1.0 : 2.5) : 5.0;
  const double as_is = 4.0 + (p.K + 63) / 64 * per_stage * __builtin_ceil(tiles(64) / (2 * cus));
  const double copied = 8.0 + 2.0 * (double)(t.bytes_a + t.bytes_b) / 6.0e6 + 5.0 + 5.0 * t.q.K / 1024.0;
  return copied < as_is;
}

hipError_t launch_packed(const GemmProblem& p, hipStream_t stream) {
  PackPlan t;
  if (!plan_pack(p, &t)) return hipErrorInvalidValue;
  void* workspace = nullptr;
  if (hipError_t e = take_workspace(&workspace, t.workspace(), stream); e != hipSuccess) return e;
  if (t.bytes_a) t.q.A = t.a.dst = workspace;
  if (t.bytes_b) t.q.B = t.b.dst = (char*)workspace + t.at_b();
  auto blocks = [](const PackJob& j) { return (j.total + 256 * kChunksPerLane - 1) / (256 * kChunksPerLane); };
  const dim3 grid(blocks(t.a) + blocks(t.b));
  auto launch = [&](auto kernel) { hipLaunchKernelGGL(kernel, grid, dim3(256), 0, stream, t.a, t.b, blocks(t.a)); };
  const size_t copies = t.bytes_a + t.bytes_b;
  const bool streamed = copies >= (p.batch == 1 ? kStreamedFrom : kStreamedBatchFrom) && copies < kStreamedTo;
  if (p.dtype == srtReal32F) streamed ? launch(pack_kernel<4, true>) : launch(pack_kernel<4, false>);
  else streamed ? launch(pack_kernel<2, true>) : launch(pack_kernel<2, false>);
  hipError_t e = launch_status(stream);
  if (e == hipSuccess) e = launch_heuristic(t.q, stream);
  (void)srtDeviceFree(workspace);   // stream-ordered: reused only by work queued after the kernels above
  return e;
}

}  // namespace srt
