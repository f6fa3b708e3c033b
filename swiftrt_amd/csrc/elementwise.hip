// Element-wise neighbours of the matmul path on the device: add / sub / mul / div / max / min
// (tensor-tensor and tensor-element), neg, exp, sigmoid, tanh, copy with type conversion, fill.
// They let the recurrent cells (tanh(matmul + bias), the LSTM gate arithmetic) and the unfused
// Dense neighbours run without a host round trip.
//
// All of them are bandwidth-bound maps, so there is ONE kernel: operands are described by a
// collapsed strided index space (broadcast = stride 0), a lane moves V consecutive elements of the
// innermost dimension as one 16-byte (or 8-byte) access when layout and alignment allow (V = 1
// otherwise), arithmetic is fp32 and the result is rounded once to the element type -- the
// reference's CPU definitions evaluated in E.Value (Sources/SwiftRTCore/platform/cpu/functions/
// CpuMath.swift: add :646-662, mul :1235-1256, max :1189-1209 `a >= b ? a : b`, sigmoid
// :1369-1377 `1 / (1 + exp(-x))`, ...).  This file is compiled with floating-point contraction
// off so the four basic operations match a C restatement bit for bit.
#include <cstring>
#include <type_traits>
#include <utility>

#include "gemm_common.h"
#include "lstm_gates.h"
#include "status.h"

namespace srt {
namespace ew {

constexpr int MAX_RANK = 4;   // after collapsing adjacent dimensions
constexpr int kVectorsPerLane = 4;   // (two: sigmoid 32.2 -> 30.7 us, bias-broadcast add 33.3 -> 36.8, the rest unchanged)
// Up to this much traffic a lane takes one vector, without the streaming hint: a small map is a launch and a memory round trip,
// four vectors one after the other are four round trips on a quarter of the lanes, and its bytes were most likely just written
// and stay in the caches for whatever reads them next.  One each / four each, us: add bf16 2048^2 (25 MB) 5.4 / 8.3, bias add bf16 1000
// x 4096 (16 MB) 4.3 / 7.2, sigmoid f32 2048 x 2000 (33 MB) 6.8 / 8.7, bias add and tanh bf16 4096^2 (67 MB) 12.2 / 13.9 and 11.9 /
// 13.2, add bf16 4096^2 (100 MB) 18.5 / 17.9, cast bf16 4096^2 to f32 (100 MB) 19.8 / 18.0, add f32 4096^2 (201 MB) 36.9 / 33.2.
constexpr unsigned long long kOneVectorBytes = 80000000;
// From the last-level cache's 256 MiB of traffic two vectors a lane, and the results stored with the streaming hint: nothing of them would be
// there for the next reader, and what the hint leaves out is their way through L2.  Four a lane and plain stores / two and the hint, us: tanh
// bf16 8192^2 (268 MB) 50.1 / 44.0, f32 94.4 / 84.9, add 71.8 / 63.9 and 142 / 132, bias add f32 4096 x 11008 (361 MB) 67.5 / 59.7, bias add and
// tanh of its sum f32 8192^2 178 / 172; below the line the sum stays for its reader (bf16 8192 x 4096, 134 MB each, 46.6 / 49.6).
constexpr unsigned long long kCachedBytes = 256ull << 20;
constexpr int kVectorsPerLanePast = 2;
// (Ragged rows too, at any length: 216 maps of rows of 17 to 5003 elements, 290 and 600 MB, 1.07x in the mean, bf16 rows of 17 1.00, of 255 1.13; behind
// by more than 2 % only f32 rows of 129 in 600 MB, 4 %.)  The kernel tells such a map by its vectors a lane.
static_assert(kVectorsPerLanePast != 1 && kVectorsPerLanePast != kVectorsPerLane);

// ---- operations -----------------------------------------------------------------------------
struct Add { static constexpr bool binary = true; static __device__ __forceinline__ float apply(float a, float b) { return a + b; } };
struct Sub { static constexpr bool binary = true; static __device__ __forceinline__ float apply(float a, float b) { return a - b; } };
struct Mul { static constexpr bool binary = true; static __device__ __forceinline__ float apply(float a, float b) { return a * b; } };
struct Div { static constexpr bool binary = true; static __device__ __forceinline__ float apply(float a, float b) { return a / b; } };
struct Max { static constexpr bool binary = true; static __device__ __forceinline__ float apply(float a, float b) { return a >= b ? a : b; } };
struct Min { static constexpr bool binary = true; static __device__ __forceinline__ float apply(float a, float b) { return a <= b ? a : b; } };
struct Neg { static constexpr bool binary = false; static __device__ __forceinline__ float apply(float a, float) { return -a; } };
struct Exp { static constexpr bool binary = false; static __device__ __forceinline__ float apply(float a, float) { return expf(a); } };
struct Sigmoid { static constexpr bool binary = false; static __device__ __forceinline__ float apply(float a, float) { return 1.0f / (1.0f + expf(-a)); } };
struct Tanh { static constexpr bool binary = false; static __device__ __forceinline__ float apply(float a, float) { return tanhf(a); } };
// For 16-bit results the hardware exponential (a few fp32 ulps) is exact enough by a wide margin:
// its error is 2^-13 of a half / 2^-16 of a bfloat16 rounding step.  fp32 results keep libm.
struct ExpFast { static constexpr bool binary = false; static __device__ __forceinline__ float apply(float a, float) { return __expf(a); } };
struct SigmoidFast {
  static constexpr bool binary = false;
  static __device__ __forceinline__ float apply(float a, float) { return __fdividef(1.0f, 1.0f + __expf(-a)); }
};
struct TanhFast {
  static constexpr bool binary = false;
  // a quotient of two short polynomials, exact to a fraction of a 16-bit rounding step and uniformly so down to
  // the smallest arguments (see activation16_ct)
  static __device__ __forceinline__ float apply(float a, float) { return srt::activation16_ct<srtActivationTanh>(0.0f, a); }
};
struct Copy { static constexpr bool binary = false; static __device__ __forceinline__ float apply(float a, float) { return a; } };

enum OpCode { kAdd, kSub, kMul, kDiv, kMax, kMin, kNeg, kExp, kSigmoid, kTanh, kCopy };

// ---- the index space --------------------------------------------------------------------------
struct Map {
  int rank;                      // 1..MAX_RANK, innermost dimension last
  uint32_t shape[MAX_RANK];      // innermost extent counted in vectors of V elements
  long long sa[MAX_RANK], sb[MAX_RANK], so[MAX_RANK];   // element strides (innermost: per element)
  unsigned long long total;      // number of vectors
  const void* a;
  const void* b;                 // null for unary operations and for tensor-element forms
  void* o;
  float element;                 // the scalar of tensor-element forms (and of fill)
  int b_is_element;
  int fill;                      // no input at all: out = element
  int b_reused;                  // the second operand is broadcast along some dimension: its lines are read again and again
  uint32_t inner_elements;       // extent of the innermost dimension in elements
};

// Operations of many instructions an element.
template <typename Op>
constexpr bool long_chain() {
  return std::is_same_v<Op, Exp> || std::is_same_v<Op, ExpFast> || std::is_same_v<Op, Sigmoid> || std::is_same_v<Op, SigmoidFast> ||
         std::is_same_v<Op, Tanh> || std::is_same_v<Op, TanhFast>;
}

template <typename T, int V>
struct alignas(V * sizeof(typename T::storage)) Pack {
  typename T::storage v[V];
};

// One vector of an input operand.  STREAM: with the non-temporal hint -- an element-wise operand
// is read once, and without the hint its lines stay in L2 until evicted (the same hint raised a
// bare streaming read of this device from 5.7 to 6.2 TB/s).  A broadcast operand (a bias row under
// every row of the other operand) is the opposite case: its few lines are wanted in the caches.
// ANYWHERE: from any element's address (global memory takes 16 bytes at element alignment).
template <typename T, int V, bool STREAM, bool ANYWHERE = false>
__device__ __forceinline__ Pack<T, V> load_pack(const typename T::storage* p) {
  using S = typename T::storage;
  constexpr int BYTES = V * (int)sizeof(S);
  if constexpr (BYTES >= 8) {
    typedef uint32_t whole_t __attribute__((ext_vector_type(BYTES / 4)));
    typedef uint32_t loose_t __attribute__((ext_vector_type(BYTES / 4), aligned(sizeof(S))));
    using words_t = std::conditional_t<ANYWHERE, loose_t, whole_t>;
    const words_t w = STREAM ? __builtin_nontemporal_load(reinterpret_cast<const words_t*>(p))
                             : *reinterpret_cast<const words_t*>(p);
    return __builtin_bit_cast(Pack<T, V>, w);
  } else {
    return *reinterpret_cast<const Pack<T, V>*>(p);
  }
}
// One vector of results; STREAM and ANYWHERE as above.
template <typename T, int V, bool STREAM, bool ANYWHERE>
__device__ __forceinline__ void store_pack(typename T::storage* p, const Pack<T, V>& v) {
  using S = typename T::storage;
  constexpr int BYTES = V * (int)sizeof(S);
  if constexpr (STREAM && BYTES >= 8) {
    typedef uint32_t whole_t __attribute__((ext_vector_type(BYTES / 4)));
    typedef uint32_t loose_t __attribute__((ext_vector_type(BYTES / 4), aligned(sizeof(S))));
    using words_t = std::conditional_t<ANYWHERE, loose_t, whole_t>;
    __builtin_nontemporal_store(__builtin_bit_cast(whole_t, v), reinterpret_cast<words_t*>(p));
  } else if constexpr (ANYWHERE) {
    __builtin_memcpy(p, &v, sizeof(v));
  } else {
    *reinterpret_cast<Pack<T, V>*>(p) = v;
  }
}

// V results of an operation, rounded to the element type.
template <typename TO, typename Op, int V>
__device__ __forceinline__ Pack<TO, V> apply_pack(const float (&fa)[V], const float (&fb)[V]) {
  Pack<TO, V> po;
  if constexpr (V > 1 && TO::dtype == srtReal16BF) {
    float r[V];
#pragma unroll
    for (int i = 0; i < V; ++i) r[i] = Op::apply(fa[i], fb[i]);
    uint32_t w[V / 2];
    encode_bf16<V>(r, w);
    po = __builtin_bit_cast(Pack<TO, V>, w);
  } else {
#pragma unroll
    for (int i = 0; i < V; ++i) po.v[i] = TO::from_float(Op::apply(fa[i], fb[i]));
  }
  return po;
}

// `v` moved to the front by `over` elements (0 .. V - 1); what follows them is left over.
template <int V>
__device__ __forceinline__ void shift_front(float (&v)[V], uint32_t over) {
#pragma unroll
  for (int s = V / 2; s > 0; s /= 2)
    if (over & s) {
#pragma unroll
      for (int i = 0; i + s < V; ++i) v[i] = v[i + s];
    }
}

// The first V - over elements of `v`.
template <typename T, int V>
__device__ __forceinline__ void store_front(typename T::storage* p, const Pack<T, V>& v, uint32_t over) {
#pragma unroll
  for (int i = 0; i < V - 1; ++i)
    if (i + over < (uint32_t)V) p[i] = v.v[i];
}

// RAGGED: rows that are no whole number of aligned vectors (odd extents, pitches or bases), read at element alignment.  The last,
// partial vector of a row is read whole, from the row's last V elements, moved to the front (what it read of its neighbour's elements,
// which that lane may be overwriting, falls off), and its `V - over` results are stored one by one.  (Read by elements too, one after
// the other, it held a launch up by 0.2 us an element: bias add bf16 1040 x 63 4.6 us, element by element throughout 3.6.)
// Rows of fewer than 1000 elements (RAGGED 1) are read without the streaming hint, because a line that two waves share is wanted twice
// (bias add f32 2^24 elements in rows of 255 36 -> 28 us); longer ones (RAGGED 2) with it (5001 x 7001 f32 add 64 us, without 79).
template <typename TI, typename TO, typename Op, int V, bool B_CACHED, int PER_LANE, int RAGGED = 0>
__device__ __forceinline__ void map_block(const Map& m, uint32_t block) {
  using SI = typename TI::storage;
  using SO = typename TO::storage;
  const SI* a = (const SI*)m.a;
  const SI* b = (const SI*)m.b;
  SO* o = (SO*)m.o;
  const int inner = m.rank - 1;
  // PER_LANE vectors per lane, a block apart, one after the other: few registers (36), eight waves per SIMD.  On
  // this device the memory parallelism of a streaming kernel comes from the waves: the same kernel with all
  // four vectors' loads issued before the first use needs 92 registers (five waves) and ran 15-20 % slower,
  // and four consecutive rows per lane with a row-broadcast operand loaded once were no faster either.
  const unsigned long long base = (unsigned long long)block * (256 * PER_LANE) + threadIdx.x;
#pragma unroll
  for (int u = 0; u < PER_LANE; ++u) {
    const unsigned long long id = base + (unsigned long long)u * 256;
    if (id >= m.total) break;
    // decompose the vector id over the collapsed dimensions
    uint32_t rest = (uint32_t)id, over = 0;   // over: elements the vector was moved back to end inside its row
    long long oa = 0, ob = 0, oo = 0;
#pragma unroll
    for (int d = MAX_RANK - 1; d >= 0; --d) {
      if (d > inner) continue;
      uint32_t idx;
      if (d == 0) {
        idx = rest;
      } else {
        const uint32_t q = rest / m.shape[d];
        idx = rest - q * m.shape[d];
        rest = q;
      }
      const long long scale = (d == inner) ? V : 1;
      if (RAGGED && d == inner && m.inner_elements - idx * V < (uint32_t)V) over = V - (m.inner_elements - idx * V);
      oa += (long long)idx * m.sa[d] * scale;
      ob += (long long)idx * m.sb[d] * scale;
      oo += (long long)idx * m.so[d] * scale;
    }
    if (RAGGED && over) {   // (an inner stride is 0 or 1 here)
      oa -= (long long)over * m.sa[inner];
      ob -= (long long)over * m.sb[inner];
    }
    float fa[V], fb[V];
    if (m.fill) {
#pragma unroll
      for (int i = 0; i < V; ++i) fa[i] = m.element;
    } else if (V > 1 && m.sa[inner] == 1) {
      const Pack<TI, V> pa = load_pack<TI, V, PER_LANE != 1 && RAGGED != 1, RAGGED != 0>(a + oa);
#pragma unroll
      for (int i = 0; i < V; ++i) fa[i] = TI::to_float(pa.v[i]);
    } else {
      // V == 1, or a broadcast along the innermost dimension
#pragma unroll
      for (int i = 0; i < V; ++i) fa[i] = TI::to_float(a[oa + (long long)i * m.sa[inner]]);
    }
    if (m.b_is_element) {
#pragma unroll
      for (int i = 0; i < V; ++i) fb[i] = m.element;
    } else if (b == nullptr) {
#pragma unroll
      for (int i = 0; i < V; ++i) fb[i] = 0.0f;
    } else if (V > 1 && m.sb[inner] == 1) {
      const Pack<TI, V> pb = load_pack<TI, V, !B_CACHED && PER_LANE != 1 && RAGGED != 1, RAGGED != 0>(b + ob);
#pragma unroll
      for (int i = 0; i < V; ++i) fb[i] = TI::to_float(pb.v[i]);
    } else {
#pragma unroll
      for (int i = 0; i < V; ++i) fb[i] = TI::to_float(b[ob + (long long)i * m.sb[inner]]);
    }
    if (RAGGED && over) {
      shift_front<V>(fa, over);
      if (Op::binary) shift_front<V>(fb, over);
    }
    const Pack<TO, V> po = apply_pack<TO, Op, V>(fa, fb);
    if (RAGGED && over) store_front<TO, V>(o + oo, po, over);
    else store_pack<TO, V, PER_LANE == kVectorsPerLanePast, RAGGED != 0>(o + oo, po);
  }
}

template <typename TI, typename TO, typename Op, int V, bool B_CACHED = false, int PER_LANE = kVectorsPerLane, int RAGGED = 0>
__global__ __launch_bounds__(256) void map_kernel(Map m) {
  map_block<TI, TO, Op, V, B_CACHED, PER_LANE, RAGGED>(m, blockIdx.x);
}

// Two copies in one launch (the halves of a concatenation).
template <typename T, int V>
__global__ __launch_bounds__(256) void copy_pair_kernel(Map m0, Map m1, uint32_t blocks0) {
  if (blockIdx.x < blocks0) map_block<T, T, Copy, V, false, 1>(m0, blockIdx.x);
  else map_block<T, T, Copy, V, false, 1>(m1, blockIdx.x - blocks0);
}

// ---- operands that walk memory across the result's rows --------------------------------------------
// An input whose unit stride lies along another dimension than the result's (`x.t` against a row-major result) made the kernel above
// read one element per line and lane: 4096^2 bf16 66 us, 1.0 TB/s.  Here a workgroup takes 64 x 64 elements of the two dimensions: it
// reads such an operand along its own rows (16 bytes per lane), turns it in LDS and writes the result along the result's rows;
// an operand that needs no turning is read where the result is written.
//   bound   memory, both sides in whole 128-byte (16-bit) or 256-byte (fp32) row segments
//   LDS     [64 rows of the result's dimension][64 + pad]: pad 2 (16-bit) and 1 (fp32) put the eight (four) elements a lane gathers on
//           different banks; its neighbours' still meet (40 % of the LDS cycles are conflicts in 16 bits, 50 % in fp32, 4096^2), which the
//           wait for memory hides (bf16 67 MB at 5.2 TB/s, fp32 134 MB at 4.7)
constexpr int TURN = 64;

struct TurnMap {
  Map m;
  int across;                       // the dimension of the operands' unit stride (the result's is the innermost one)
  int turn_a, turn_b;               // which operands are turned
  uint32_t tiles_inner, tiles_across;
};

//   STREAM  the turned operand's reads carry the streaming hint once the map is past kOneVectorBytes: f32 4096^2 32.5 -> 28.5 us, but
//           bf16 4096^2 13.0 -> 15.3
//   PAST    the results' stores as well, from kCachedBytes and with every row of the result on whole 128-byte lines: f32 4096 x 11008 81.4 -> 71.7
//           us, 8192^2 112 -> 97, bf16 55.7 -> 50.4; rows off the lines, which two workgroups fill in parts, lose (bf16 16384 x 8200 123 -> 156)
template <typename TI, typename TO, typename Op, bool STREAM, bool PAST>
__global__ __launch_bounds__(256) void turn_kernel(TurnMap t) {
  using SI = typename TI::storage;
  using SO = typename TO::storage;
  constexpr int VI = 16 / sizeof(SI);                                  // elements of a 16-byte read
  constexpr int V = 16 / (sizeof(SI) > sizeof(SO) ? sizeof(SI) : sizeof(SO));   // elements a lane writes at once
  constexpr int PITCH = TURN + (sizeof(SI) == 2 ? 2 : 1);
  __shared__ SI lds[Op::binary ? 2 : 1][TURN * PITCH];
  const Map& m = t.m;
  const int inner = m.rank - 1;
  // workgroup -> tile of the two dimensions, index of the others
  uint32_t rest = blockIdx.x;
  const uint32_t ti = rest % t.tiles_inner;
  rest /= t.tiles_inner;
  const uint32_t ta = (rest + ti) % t.tiles_across;   // along a diagonal: neighbours of a power-of-two pitch share no channel (4096^2 bf16 15.0 -> 12.9 us)
  rest /= t.tiles_across;
  long long oa = 0, ob = 0, oo = 0;
#pragma unroll
  for (int d = MAX_RANK - 2; d >= 0; --d) {
    if (d >= inner || d == t.across) continue;
    const uint32_t q = rest / m.shape[d], idx = rest - q * m.shape[d];
    rest = q;
    oa += (long long)idx * m.sa[d];
    ob += (long long)idx * m.sb[d];
    oo += (long long)idx * m.so[d];
  }
  const uint32_t i0 = ti * TURN, a0 = ta * TURN;
  const uint32_t ni = min((uint32_t)TURN, m.shape[inner] - i0), na = min((uint32_t)TURN, m.shape[t.across] - a0);
  const SI* a = (const SI*)m.a + oa + (long long)i0 * m.sa[inner] + (long long)a0 * m.sa[t.across];
  const SI* b = m.b ? (const SI*)m.b + ob + (long long)i0 * m.sb[inner] + (long long)a0 * m.sb[t.across] : nullptr;
  SO* o = (SO*)m.o + oo + i0 + (long long)a0 * m.so[t.across];
  const int tid = threadIdx.x;

  auto turn_in = [&](const SI* src, long long row_stride, SI* to) {
    constexpr int CH = TURN / VI;   // reads per row
#pragma unroll
    for (int u = 0; u < TURN * CH / 256; ++u) {
      const uint32_t id = tid + u * 256, row = id / CH, col = (id % CH) * VI;
      if (row < ni && col < na) {
        const SI* p = src + (long long)row * row_stride + col;
        Pack<TI, VI> x;
        if (col + VI <= na) {
          x = load_pack<TI, VI, STREAM, true>(p);
        } else {
#pragma unroll
          for (int e = 0; e < VI; ++e) x.v[e] = p[min((uint32_t)e, na - 1 - col)];
        }
#pragma unroll
        for (int e = 0; e < VI; ++e) to[row * PITCH + col + e] = x.v[e];
      }
    }
  };
  if (t.turn_a) turn_in(a, m.sa[inner], lds[0]);
  if (Op::binary && t.turn_b) turn_in(b, m.sb[inner], lds[Op::binary ? 1 : 0]);
  __syncthreads();

  constexpr int CO = TURN / V;      // writes per row of the result
#pragma unroll
  for (int u = 0; u < TURN * CO / 256; ++u) {
    const uint32_t id = tid + u * 256, row = id / CO, col = (id % CO) * V;   // row: along `across`, col: along the result's rows
    if (row >= na || col >= ni) continue;
    float fa[V], fb[V];
    auto gather = [&](bool turned, const SI* from, const SI* direct, long long s_inner, long long s_across, float (&f)[V]) {
      if (!turned && s_inner == 1 && col + V <= ni) {
        const Pack<TI, V> x = load_pack<TI, V, false, true>(direct + (long long)row * s_across + col);
#pragma unroll
        for (int e = 0; e < V; ++e) f[e] = TI::to_float(x.v[e]);
        return;
      }
#pragma unroll
      for (int e = 0; e < V; ++e) {
        const uint32_t c = min(col + e, ni - 1);
        f[e] = TI::to_float(turned ? from[c * PITCH + row] : direct[(long long)c * s_inner + (long long)row * s_across]);
      }
    };
    gather(t.turn_a, lds[0], a, m.sa[inner], m.sa[t.across], fa);
    if (m.b_is_element) {
#pragma unroll
      for (int e = 0; e < V; ++e) fb[e] = m.element;
    } else if (Op::binary && b) {
      gather(t.turn_b, lds[Op::binary ? 1 : 0], b, m.sb[inner], m.sb[t.across], fb);
    } else {
#pragma unroll
      for (int e = 0; e < V; ++e) fb[e] = 0.0f;
    }
    const Pack<TO, V> po = apply_pack<TO, Op, V>(fa, fb);
    SO* dst = o + (long long)row * m.so[t.across] + col;
    if (col + V <= ni) {
      store_pack<TO, V, PAST, !PAST>(dst, po);
    } else {
#pragma unroll
      for (int e = 0; e < V; ++e)
        if (col + e < ni) dst[e] = po.v[e];
    }
  }
}

// Whether operands are turned: a unit stride along another dimension than the innermost, tiles that are full enough, and enough of them.
// The kernel above, whose lanes share the lines they read, is ahead of tiles on small maps (a quarter of the workgroups, and one trip
// to memory after another) and on narrow ones.  Turned / not, us: x.t bf16 256 x 256 3.3 / 3.1, 2^20 3.5 / 4.1 (64 x 64 matrices), 2^24 12.8 / 43, but
// 65536 of 16 x 16 89 / 35, 3970 of 65 x 65 56 / 48 with an addend; f32 2^18 4.3 / 3.3, 2^20 (96 x 96) 5.2 / 4.6, 2^24 39 / 55, 16384 of 32 x
// 32 40 / 36, 508400 rows of 33 with an addend 74 / 42; rows of 4096 2^20 3.4 / 6.2 (bf16, 256 of them), rows of 2^20 62 / 632 (f32, 32).
template <typename TI, typename TO, typename Op>
bool plan_turn(const Map& m, TurnMap* t) {
  const int inner = m.rank - 1;
  if (m.fill || m.rank < 2 || m.so[inner] != 1 || m.shape[inner] < 16) return false;
  auto unit_dim = [&](const void* p, const long long* s) {
    if (!p || s[inner] == 0 || s[inner] == 1) return -1;
    for (int d = 0; d < inner; ++d)
      if (s[d] == 1 && m.shape[d] >= 16) return d;
    return -1;
  };
  const int da = unit_dim(m.a, m.sa), db = Op::binary && !m.b_is_element ? unit_dim(m.b, m.sb) : -1;
  if (da < 0 && db < 0) return false;
  t->m = m;
  t->across = da >= 0 ? da : db;
  t->turn_a = da >= 0;
  t->turn_b = db >= 0 && db == t->across;
  t->tiles_inner = (m.shape[inner] + TURN - 1) / TURN;
  t->tiles_across = (m.shape[t->across] + TURN - 1) / TURN;
  constexpr bool halves = sizeof(typename TI::storage) == 2 && sizeof(typename TO::storage) == 2;
  const double fill = (double)m.shape[inner] * m.shape[t->across] / ((double)t->tiles_inner * t->tiles_across * TURN * TURN);
  // long rows of the result: its neighbours along the operands' rows come a whole row later, when their lines may have left the caches
  if (m.shape[inner] >= 256) return m.total >= 750000 && fill >= (halves || m.total >= 12000000 ? 0.2 : 0.3);
  if (m.total < 2000000) return false;
  const bool whole = m.shape[inner] % 8 == 0 && m.shape[t->across] % 8 == 0;   // rows of whole 16-byte pieces, either way
  const bool all_turned = t->turn_a && (!m.b || t->turn_b);
  return fill >= (!halves ? 0.55 : whole && (all_turned || m.total >= 4000000) ? 0.25 : all_turned ? 0.5 : 0.6);
}

template <typename TI, typename TO, typename Op, int V, bool B_CACHED, int PER_LANE, int RAGGED>
hipError_t launch_lanes(const Map& m, hipStream_t stream) {
  const unsigned long long blocks = (m.total + 256 * PER_LANE - 1) / (256 * PER_LANE);
  if (blocks == 0) return hipSuccess;
  if (blocks > 0x7fffffffull) return hipErrorInvalidValue;
  hipLaunchKernelGGL((map_kernel<TI, TO, Op, V, B_CACHED, PER_LANE, RAGGED>), dim3((unsigned)blocks), dim3(256), 0, stream, m);
  return launch_status(stream);
}

template <typename TI, typename TO, typename Op, int V, int RAGGED>
hipError_t launch_v(const Map& m, hipStream_t stream) {
  unsigned long long vector_bytes = V * sizeof(typename TO::storage);
  if (!m.fill) vector_bytes += V * sizeof(typename TI::storage) * (m.b && !m.b_reused ? 2 : 1);
  // (single elements, 2-byte accesses: from a million of them four each, bias add bf16 4095^2 34.0 us against 37.8)
  const unsigned long long bytes = m.total * vector_bytes;
  if (bytes <= (V == 1 ? kOneVectorBytes / 16 : kOneVectorBytes)) return launch_lanes<TI, TO, Op, V, false, 1, RAGGED>(m, stream);
  // (a run-time choice between the two kinds of load inside one kernel cost every operation 14 %)
  if constexpr (V > 1) {
    if (bytes >= kCachedBytes) {
      if constexpr (Op::binary) {
        if (m.b_reused) return launch_lanes<TI, TO, Op, V, true, kVectorsPerLanePast, RAGGED>(m, stream);
      }
      return launch_lanes<TI, TO, Op, V, false, kVectorsPerLanePast, RAGGED>(m, stream);
    }
    if constexpr (Op::binary) {
      if (m.b_reused) return launch_lanes<TI, TO, Op, V, true, kVectorsPerLane, RAGGED>(m, stream);
    }
  }
  return launch_lanes<TI, TO, Op, V, false, kVectorsPerLane, RAGGED>(m, stream);
}

// Vector width the layout allows: the innermost dimension must be contiguous in the result and
// contiguous or broadcast in the inputs.  *ragged: its extent, some other stride or a base pointer is no multiple of the vector.
template <typename TI, typename TO>
int vector_width(const Map& m, bool* ragged) {
  constexpr int V = 16 / (sizeof(typename TI::storage) > sizeof(typename TO::storage) ? sizeof(typename TI::storage)
                                                                                      : sizeof(typename TO::storage));
  *ragged = false;
  const int inner = m.rank - 1;
  if (m.so[inner] != 1) return 1;
  if (m.shape[inner] % V) *ragged = true;
  auto operand_ok = [&](const void* p, const long long* s, size_t esize, bool is_out) {
    if (!p) return true;
    if (s[inner] != 1 && (is_out || s[inner] != 0)) return false;
    if (s[inner] == 1) {
      if ((uintptr_t)p % (V * esize)) *ragged = true;
      for (int d = 0; d < inner; ++d)
        if (s[d] % V) *ragged = true;
    }
    return true;
  };
  if (!operand_ok(m.o, m.so, sizeof(typename TO::storage), true)) return 1;
  if (!m.fill && !operand_ok(m.a, m.sa, sizeof(typename TI::storage), false)) return 1;
  if (!m.fill && !m.b_is_element && !operand_ok(m.b, m.sb, sizeof(typename TI::storage), false)) return 1;
  return V;
}

// Whether ragged rows are worth vectors: from four vectors a row (two of eight elements on a large map) and a few hundred thousand
// elements, more where a result is a long
// chain of arithmetic (eight in a row on one lane take longer than a small launch); fp32 with two whole operands not from 80 MB to
// what the last-level cache holds, where single elements, whole lines to a wave, are ahead.  Vectors / single elements, us: add bf16 16384 x 16 rows
// of 31 4.1 / 4.3, 63 3.6 / 4.4; bias add bf16 2^16 elements 3.4 / 3.3, 2^20 3.5 / 3.8, 2^22 6.4 / 9.4, 2^24 14 / 33; tanh bf16 rows of 63 2^18
// 3.9 / 3.4, 2^20 3.9 / 3.5, 2^22 6.9 / 8.8; add f32 rows of 255 2^20 3.5 / 4.1, 2^22 9.4 / 9.7, 2^23 22 / 17, 2^24 38 / 31, 5001
// x 7001 64 / 75.
template <typename TI, typename TO, typename Op>
bool ragged_pays(const Map& m, int v) {
  const uint32_t row = m.shape[m.rank - 1];
  if (row < 4u * (uint32_t)v && (v < 8 || row < 2u * (uint32_t)v || m.total < 6000000u)) return false;
  if (m.total < (long_chain<Op>() ? 2000000u : 750000u)) return false;
  if (sizeof(typename TI::storage) == 4 && m.b && !m.b_is_element && !m.b_reused)
  {
    const unsigned long long bytes = m.total * (8 + sizeof(typename TO::storage));
    return bytes <= kOneVectorBytes || (bytes > 300000000 && row >= 1000);
  }
  return true;
}

// The map with its innermost extent counted in vectors.
inline void count_vectors(Map* m, int v) {
  const int inner = m->rank - 1;
  const uint32_t vectors = (uint32_t)(((unsigned long long)m->shape[inner] + v - 1) / v);   // (extents reach 2^32 - 1)
  m->inner_elements = m->shape[inner];
  m->total = m->total / m->shape[inner] * vectors;
  m->shape[inner] = vectors;
}

template <typename TI, typename TO, typename Op>
hipError_t launch_t(Map m, hipStream_t stream) {
  constexpr int V = 16 / (sizeof(typename TI::storage) > sizeof(typename TO::storage) ? sizeof(typename TI::storage)
                                                                                      : sizeof(typename TO::storage));
  bool ragged;
  if (vector_width<TI, TO>(m, &ragged) == V && (!ragged || ragged_pays<TI, TO, Op>(m, V))) {
    count_vectors(&m, V);
    if (!ragged) return launch_v<TI, TO, Op, V, 0>(m, stream);
    return m.inner_elements < 1000 ? launch_v<TI, TO, Op, V, 1>(m, stream) : launch_v<TI, TO, Op, V, 2>(m, stream);
  }
  TurnMap t;
  if (plan_turn<TI, TO, Op>(m, &t)) {
    const int inner = m.rank - 1;
    const unsigned long long others = m.total / m.shape[inner] / m.shape[t.across];
    const unsigned long long blocks = others * t.tiles_inner * t.tiles_across;
    if (blocks <= 0x7fffffffull) {
      const unsigned long long bytes = m.total * (sizeof(typename TO::storage) + sizeof(typename TI::storage) * (m.b && !m.b_reused ? 2 : 1));
      bool lines = (uintptr_t)m.o % 128 == 0;
      for (int d = 0; d < inner; ++d) lines = lines && m.so[d] * (long long)sizeof(typename TO::storage) % 128 == 0;
      if (bytes >= kCachedBytes && lines) hipLaunchKernelGGL((turn_kernel<TI, TO, Op, true, true>), dim3((unsigned)blocks), dim3(256), 0, stream, t);
      else if (bytes > kOneVectorBytes) hipLaunchKernelGGL((turn_kernel<TI, TO, Op, true, false>), dim3((unsigned)blocks), dim3(256), 0, stream, t);
      else hipLaunchKernelGGL((turn_kernel<TI, TO, Op, false, false>), dim3((unsigned)blocks), dim3(256), 0, stream, t);
      return launch_status(stream);
    }
  }
  return launch_v<TI, TO, Op, 1, 0>(m, stream);
}

template <typename Op>
hipError_t launch_same_type(int dtype, const Map& m, hipStream_t stream) {
  switch (dtype) {
    case srtReal32F: return launch_t<F32, F32, Op>(m, stream);
    case srtReal16F: return launch_t<F16, F16, Op>(m, stream);
    case srtReal16BF: return launch_t<BF16, BF16, Op>(m, stream);
    default: return hipErrorNotSupported;
  }
}

hipError_t launch_op(int op, int dtype, const Map& m, hipStream_t stream) {
  switch (op) {
    case kAdd: return launch_same_type<Add>(dtype, m, stream);
    case kSub: return launch_same_type<Sub>(dtype, m, stream);
    case kMul: return launch_same_type<Mul>(dtype, m, stream);
    case kDiv: return launch_same_type<Div>(dtype, m, stream);
    case kMax: return launch_same_type<Max>(dtype, m, stream);
    case kMin: return launch_same_type<Min>(dtype, m, stream);
    case kNeg: return launch_same_type<Neg>(dtype, m, stream);
    case kExp: return dtype == srtReal32F ? launch_same_type<Exp>(dtype, m, stream)
                                          : launch_same_type<ExpFast>(dtype, m, stream);
    case kSigmoid: return dtype == srtReal32F ? launch_same_type<Sigmoid>(dtype, m, stream)
                                              : launch_same_type<SigmoidFast>(dtype, m, stream);
    case kTanh: return dtype == srtReal32F ? launch_same_type<Tanh>(dtype, m, stream)
                                           : launch_same_type<TanhFast>(dtype, m, stream);
    case kCopy: return launch_same_type<Copy>(dtype, m, stream);
    default: return hipErrorNotSupported;
  }
}

hipError_t launch_convert(int itype, int otype, const Map& m, hipStream_t stream) {
  if (itype == otype) return launch_same_type<Copy>(itype, m, stream);
  if (itype == srtReal32F && otype == srtReal16BF) return launch_t<F32, BF16, Copy>(m, stream);
  if (itype == srtReal32F && otype == srtReal16F) return launch_t<F32, F16, Copy>(m, stream);
  if (itype == srtReal16BF && otype == srtReal32F) return launch_t<BF16, F32, Copy>(m, stream);
  if (itype == srtReal16F && otype == srtReal32F) return launch_t<F16, F32, Copy>(m, stream);
  if (itype == srtReal16BF && otype == srtReal16F) return launch_t<BF16, F16, Copy>(m, stream);
  if (itype == srtReal16F && otype == srtReal16BF) return launch_t<F16, BF16, Copy>(m, stream);
  return hipErrorNotSupported;
}

template <typename T>
hipError_t launch_copy_pair(Map m0, Map m1, hipStream_t stream) {
  constexpr int V = 16 / sizeof(typename T::storage);
  auto go = [&](auto width) {
    constexpr int W = decltype(width)::value;
    const unsigned long long b0 = (m0.total + 255) / 256, b1 = (m1.total + 255) / 256;
    if (b0 + b1 > 0x7fffffffull) return hipErrorInvalidValue;
    hipLaunchKernelGGL((copy_pair_kernel<T, W>), dim3((unsigned)(b0 + b1)), dim3(256), 0, stream, m0, m1, (uint32_t)b0);
    return launch_status(stream);
  };
  bool r0, r1;
  if (vector_width<T, T>(m0, &r0) == V && !r0 && vector_width<T, T>(m1, &r1) == V && !r1) {
    count_vectors(&m0, V);
    count_vectors(&m1, V);
    return go(std::integral_constant<int, V>{});
  }
  return go(std::integral_constant<int, 1>{});
}

// ---- the gate arithmetic of an LSTM cell ---------------------------------------------------------
// From gates = [input, update, forget, output] (one row of 4 H per batch row) and the cell state:
//   cell' = cell * sigmoid(forget) + sigmoid(input) * tanh(update),  hidden' = tanh(cell') * sigmoid(output)
// with every intermediate rounded to the element type, i.e. bit for bit what the nine element-wise launches it replaces give.
// Those were launches and round trips, not bytes: 64 x 512 fp32 is 0.9 MB in all and took 9 x 7 us; here it is one launch, each
// value read and written once, a lane one 16-byte vector of the H dimension (one element when the layout does not allow it).
struct GateProblem {
  uint32_t rows, columns;            // columns counted in vectors of V elements
  const void* gates;
  const void* cell;
  void* new_cell;
  void* new_hidden;
  long long part;                    // elements between the gates of one column
  long long gates_row, gates_col, cell_row, cell_col, new_cell_row, new_cell_col, new_hidden_row, new_hidden_col;
};

template <typename T, int V>
__global__ __launch_bounds__(256) void lstm_gates_kernel(GateProblem p) {
  using S = typename T::storage;
  const uint32_t id = blockIdx.x * 256 + threadIdx.x;
  if (id >= p.rows * p.columns) return;
  const uint32_t row = id / p.columns, col = (id - row * p.columns) * V;
  const S* g = (const S*)p.gates + (long long)row * p.gates_row + (long long)col * p.gates_col;
  const Pack<T, V> gi = load_pack<T, V, false>(g), gu = load_pack<T, V, false>(g + p.part),
                   gf = load_pack<T, V, false>(g + 2 * p.part), go = load_pack<T, V, false>(g + 3 * p.part);
  const Pack<T, V> c = load_pack<T, V, false>((const S*)p.cell + (long long)row * p.cell_row + (long long)col * p.cell_col);
  Pack<T, V> nc, nh;
#pragma unroll
  for (int i = 0; i < V; ++i)
    lstm_gate<T>(T::to_float(gi.v[i]), T::to_float(gu.v[i]), T::to_float(gf.v[i]), T::to_float(go.v[i]), T::to_float(c.v[i]), &nc.v[i], &nh.v[i]);
  *reinterpret_cast<Pack<T, V>*>((S*)p.new_cell + (long long)row * p.new_cell_row + (long long)col * p.new_cell_col) = nc;
  *reinterpret_cast<Pack<T, V>*>((S*)p.new_hidden + (long long)row * p.new_hidden_row + (long long)col * p.new_hidden_col) = nh;
}

template <typename T>
hipError_t launch_lstm_gates(GateProblem p, hipStream_t stream) {
  constexpr int V = 16 / sizeof(typename T::storage);
  auto go = [&](auto width) {
    constexpr int W = decltype(width)::value;
    p.columns /= W;
    // the lanes of a launch are counted in 31 bits: a larger cell goes in pieces of whole rows
    const uint32_t rows = p.rows, most = 0x7fffffffu / p.columns;
    hipError_t e = hipSuccess;
    for (uint32_t done = 0; done < rows && e == hipSuccess; done += p.rows) {
      auto at = [&](const void* base, long long row) { return (char*)base + (long long)done * row * (long long)sizeof(typename T::storage); };
      GateProblem q = p;
      q.rows = p.rows = rows - done < most ? rows - done : most;
      q.gates = at(p.gates, p.gates_row); q.cell = at(p.cell, p.cell_row);
      q.new_cell = at(p.new_cell, p.new_cell_row); q.new_hidden = at(p.new_hidden, p.new_hidden_row);
      hipLaunchKernelGGL((lstm_gates_kernel<T, W>), dim3((q.rows * q.columns + 255) / 256), dim3(256), 0, stream, q);
      e = launch_status(stream);
    }
    return e;
  };
  const bool dense = p.gates_col == 1 && p.cell_col == 1 && p.new_cell_col == 1 && p.new_hidden_col == 1;
  const bool whole = p.columns % V == 0 && p.part % V == 0 && p.gates_row % V == 0 && p.cell_row % V == 0 && p.new_cell_row % V == 0 &&
                     p.new_hidden_row % V == 0;
  const bool aligned = (((uintptr_t)p.gates | (uintptr_t)p.cell | (uintptr_t)p.new_cell | (uintptr_t)p.new_hidden) & 15u) == 0;
  // (a small cell has more to gain from lanes than from wide accesses: the transcendental chain of a lane is serial)
  const bool few = (unsigned long long)p.rows * p.columns <= 256ull * 1024;
  if (dense && whole && aligned && !few) return go(std::integral_constant<int, V>{});
  return go(std::integral_constant<int, 1>{});
}

// ---- host side: descriptors -> collapsed index space -------------------------------------------
bool float_type(srtDataType t) { return t == srtReal32F || t == srtReal16F || t == srtReal16BF; }

bool desc_ok(const srtTensorDescriptor* d) { return d && d->shape && d->strides && d->rank >= 1; }

// Reads one element of `type` from host memory as fp32 (the scalar of tensor-element forms).
float host_element(srtDataType type, const void* p) {
  if (type == srtReal32F) {
    float f;
    memcpy(&f, p, 4);
    return f;
  }
  uint16_t h;
  memcpy(&h, p, 2);
  if (type == srtReal16BF) {
    uint32_t u = (uint32_t)h << 16;
    float f;
    memcpy(&f, &u, 4);
    return f;
  }
  _Float16 x;
  memcpy(&x, &h, 2);
  return (float)x;
}

// Builds the index space of `out` with the strides of each operand, dropping extent-1
// dimensions and merging neighbours that every operand walks contiguously (or broadcasts).
// Returns srtErrorNotSupported when more than MAX_RANK dimensions remain.
srtStatus build_map(const srtTensorDescriptor* ad, const srtTensorDescriptor* bd, const srtTensorDescriptor* od,
                    Map* m, bool* empty) {
  *empty = false;
  const uint32_t rank = od->rank;
  if (rank > 8) return srtErrorNotSupported;
  if ((ad && ad->rank != rank) || (bd && bd->rank != rank)) return srtErrorInvalidValue;
  size_t shape[8];
  long long sa[8], sb[8], so[8];
  int n = 0;
  unsigned long long total = 1;
  for (uint32_t d = 0; d < rank; ++d) {
    const size_t e = od->shape[d];
    if ((ad && ad->shape[d] != e) || (bd && bd->shape[d] != e)) return srtErrorInvalidValue;
    total *= e;
    if (e == 1) continue;
    shape[n] = e;
    sa[n] = ad ? (long long)ad->strides[d] : 0;
    sb[n] = bd ? (long long)bd->strides[d] : 0;
    so[n] = (long long)od->strides[d];
    ++n;
  }
  if (total == 0) { *empty = true; return srtSuccess; }
  if (n == 0) { shape[0] = 1; sa[0] = sb[0] = 0; so[0] = 1; n = 1; }
  // the result's storage order: its smallest stride innermost (a column-major result is a row-major walk of its storage)
  for (int d = 1; d < n; ++d)
    for (int e = d; e > 0 && so[e - 1] < so[e]; --e) {
      std::swap(shape[e - 1], shape[e]);
      std::swap(sa[e - 1], sa[e]);
      std::swap(sb[e - 1], sb[e]);
      std::swap(so[e - 1], so[e]);
    }
  // merge d into d + 1 where stride[d] == shape[d + 1] * stride[d + 1] for every operand
  int w = 0;
  for (int d = 1; d < n; ++d) {
    const long long e = (long long)shape[d];
    if (sa[w] == e * sa[d] && sb[w] == e * sb[d] && so[w] == e * so[d]) {
      shape[w] *= shape[d];
      sa[w] = sa[d]; sb[w] = sb[d]; so[w] = so[d];
    } else {
      ++w;
      shape[w] = shape[d]; sa[w] = sa[d]; sb[w] = sb[d]; so[w] = so[d];
    }
  }
  n = w + 1;
  if (n > MAX_RANK) return srtErrorNotSupported;
  m->rank = n;
  for (int d = 0; d < MAX_RANK; ++d) {
    m->shape[d] = 1; m->sa[d] = m->sb[d] = m->so[d] = 0;
  }
  for (int d = 0; d < n; ++d) {
    if (shape[d] > 0xffffffffull) return srtErrorNotSupported;
    m->shape[d] = (uint32_t)shape[d];
    m->sa[d] = sa[d]; m->sb[d] = sb[d]; m->so[d] = so[d];
  }
  if (total > 0xffffffffull) return srtErrorNotSupported;   // the kernel decomposes 32-bit ids
  m->total = total;
  m->b_reused = 0;
  for (int d = 0; d < n; ++d)
    if (bd && shape[d] > 1 && sb[d] == 0) m->b_reused = 1;
  return srtSuccess;
}

srtStatus binary(int op, const void* a, const srtTensorDescriptor* ad, const void* b, const srtTensorDescriptor* bd,
                 void* out, const srtTensorDescriptor* od, srtStream stream) {
  if (!desc_ok(ad) || !desc_ok(bd) || !desc_ok(od)) return srtErrorInvalidValue;
  if (!float_type(od->type) || ad->type != od->type || bd->type != od->type) return srtErrorNotSupported;
  Map m{};
  bool empty;
  srtStatus s = build_map(ad, bd, od, &m, &empty);
  if (s != srtSuccess || empty) return s;
  if (!a || !b || !out) return srtErrorInvalidValue;
  m.a = a; m.b = b; m.o = out;
  return from_hip(launch_op(op, od->type, m, reinterpret_cast<hipStream_t>(stream)));
}

srtStatus binary_element(int op, const void* a, const srtTensorDescriptor* ad, const void* element, void* out,
                         const srtTensorDescriptor* od, srtStream stream) {
  if (!desc_ok(ad) || !desc_ok(od) || !element) return srtErrorInvalidValue;
  if (!float_type(od->type) || ad->type != od->type) return srtErrorNotSupported;
  Map m{};
  bool empty;
  srtStatus s = build_map(ad, nullptr, od, &m, &empty);
  if (s != srtSuccess || empty) return s;
  if (!a || !out) return srtErrorInvalidValue;
  m.a = a; m.o = out;
  m.b_is_element = 1;
  m.element = host_element(od->type, element);
  return from_hip(launch_op(op, od->type, m, reinterpret_cast<hipStream_t>(stream)));
}

srtStatus unary(int op, const void* a, const srtTensorDescriptor* ad, void* out, const srtTensorDescriptor* od,
                srtStream stream) {
  if (!desc_ok(ad) || !desc_ok(od)) return srtErrorInvalidValue;
  if (!float_type(od->type) || !float_type(ad->type)) return srtErrorNotSupported;
  if (op != kCopy && ad->type != od->type) return srtErrorNotSupported;
  Map m{};
  bool empty;
  srtStatus s = build_map(ad, nullptr, od, &m, &empty);
  if (s != srtSuccess || empty) return s;
  if (!a || !out) return srtErrorInvalidValue;
  m.a = a; m.o = out;
  hipStream_t hs = reinterpret_cast<hipStream_t>(stream);
  if (op == kCopy) return from_hip(launch_convert(ad->type, od->type, m, hs));
  return from_hip(launch_op(op, od->type, m, hs));
}

void flat_map(size_t count, Map* m) {
  m->rank = 1;
  for (int d = 0; d < MAX_RANK; ++d) { m->shape[d] = 1; m->sa[d] = m->sb[d] = m->so[d] = 0; }
  m->sa[0] = m->sb[0] = m->so[0] = 1;
  m->total = count;
}

// Flat forms take a count, not a descriptor.  Long buffers are cut into pieces the 32-bit innermost
// extent can hold, and a count that is not a multiple of the vector width into a vector body and a
// short element-wise tail (the buffers themselves are allocation-aligned).
template <typename F>
srtStatus flat_pieces(size_t count, size_t in_size, size_t out_size, Map m, F launch) {
  const size_t piece = (size_t)1 << 30;
  size_t done = 0;
  while (done < count) {
    size_t n = count - done < piece ? count - done : piece;
    if (n > 8 && n % 8) n -= n % 8;   // body now, tail in the next round
    Map p = m;
    flat_map(n, &p);
    p.shape[0] = (uint32_t)n;
    if (m.a) p.a = (const char*)m.a + done * in_size;
    if (m.b) p.b = (const char*)m.b + done * in_size;
    p.o = (char*)m.o + done * out_size;
    srtStatus s = from_hip(launch(p));
    if (s != srtSuccess) return s;
    done += n;
  }
  return srtSuccess;
}

size_t type_size(srtDataType t) { return t == srtReal32F ? 4 : 2; }

}  // namespace ew
}  // namespace srt

using namespace srt::ew;

extern "C" {

#define SRT_BINARY(Name, code)                                                                              \
  srtStatus srt##Name(const void* a, const srtTensorDescriptor* aDesc, const void* b,                        \
                      const srtTensorDescriptor* bDesc, void* out, const srtTensorDescriptor* oDesc,         \
                      srtStream stream) {                                                                    \
    return binary(code, a, aDesc, b, bDesc, out, oDesc, stream);                                            \
  }                                                                                                          \
  srtStatus srt##Name##TE(const void* a, const srtTensorDescriptor* aDesc, const void* element, void* out,   \
                          const srtTensorDescriptor* oDesc, srtStream stream) {                              \
    return binary_element(code, a, aDesc, element, out, oDesc, stream);                                     \
  }

SRT_BINARY(Add, kAdd)
SRT_BINARY(Sub, kSub)
SRT_BINARY(Mul, kMul)
SRT_BINARY(Div, kDiv)
SRT_BINARY(Max, kMax)
SRT_BINARY(Min, kMin)

#define SRT_UNARY(Name, code)                                                                     \
  srtStatus srt##Name(const void* a, const srtTensorDescriptor* aDesc, void* out,                  \
                      const srtTensorDescriptor* oDesc, srtStream stream) {                        \
    return unary(code, a, aDesc, out, oDesc, stream);                                             \
  }

SRT_UNARY(Neg, kNeg)
SRT_UNARY(Exp, kExp)
SRT_UNARY(Sigmoid, kSigmoid)
SRT_UNARY(Tanh, kTanh)
SRT_UNARY(Copy, kCopy)

// Dense tensor-tensor and tensor-element forms of the six binary operators: what CudaQueue calls when
// canFlatten holds (Sources/SwiftRTCore/platform/cuda/functions/CudaMath.swift:103-113).
static srtStatus binary_flat(int op, srtDataType type, const void* a, const void* b, const void* element, void* out,
                             size_t count, srtStream stream) {
  if (!float_type(type)) return srtErrorNotSupported;
  if (count == 0) return srtSuccess;
  if (!a || !out || (!b && !element)) return srtErrorInvalidValue;
  Map m{};
  m.a = a; m.b = b; m.o = out;
  if (!b) {
    m.b_is_element = 1;
    m.element = host_element(type, element);
  }
  hipStream_t hs = reinterpret_cast<hipStream_t>(stream);
  return flat_pieces(count, type_size(type), type_size(type), m,
                     [&](const Map& p) { return launch_op(op, type, p, hs); });
}

#define SRT_BINARY_FLAT(Name, code)                                                                          \
  srtStatus srt##Name##Flat(srtDataType type, const void* a, const void* b, void* out, size_t count,          \
                            srtStream stream) {                                                               \
    return binary_flat(code, type, a, b, nullptr, out, count, stream);                                       \
  }                                                                                                           \
  srtStatus srt##Name##TEFlat(const void* a, srtDataType atype, const void* element, void* out, size_t count, \
                              srtStream stream) {                                                             \
    return binary_flat(code, atype, a, nullptr, element, out, count, stream);                                \
  }

SRT_BINARY_FLAT(Add, kAdd)
SRT_BINARY_FLAT(Sub, kSub)
SRT_BINARY_FLAT(Mul, kMul)
SRT_BINARY_FLAT(Div, kDiv)
SRT_BINARY_FLAT(Max, kMax)
SRT_BINARY_FLAT(Min, kMin)

// the reference spells the comparison family's tensor-element form the other way round, with the type first
srtStatus srtMinFlatTE(srtDataType type, const void* a, const void* element, void* out, size_t count, srtStream stream) {
  return binary_flat(kMin, type, a, nullptr, element, out, count, stream);
}
srtStatus srtMaxFlatTE(srtDataType type, const void* a, const void* element, void* out, size_t count, srtStream stream) {
  return binary_flat(kMax, type, a, nullptr, element, out, count, stream);
}

srtStatus srtCopyFlat(srtDataType atype, const void* a, srtDataType otype, void* out, size_t count,
                      srtStream stream) {
  if (!float_type(atype) || !float_type(otype)) return srtErrorNotSupported;
  if (count == 0) return srtSuccess;
  if (!a || !out) return srtErrorInvalidValue;
  Map m{};
  m.a = a; m.o = out;
  hipStream_t hs = reinterpret_cast<hipStream_t>(stream);
  return flat_pieces(count, type_size(atype), type_size(otype), m,
                     [&](const Map& p) { return launch_convert(atype, otype, p, hs); });
}

srtStatus srtFillFlat(srtDataType type, void* out, const void* element, size_t count, srtStream stream) {
  if (!float_type(type)) return srtErrorNotSupported;
  if (count == 0) return srtSuccess;
  if (!out || !element) return srtErrorInvalidValue;
  Map m{};
  m.o = out;
  m.fill = 1;
  m.element = host_element(type, element);
  hipStream_t hs = reinterpret_cast<hipStream_t>(stream);
  return flat_pieces(count, type_size(type), type_size(type), m,
                     [&](const Map& p) { return launch_op(kCopy, type, p, hs); });
}


// out = a and b joined along `axis`: the two copies of a concatenation in one launch.
srtStatus srtConcat(const void* a, const srtTensorDescriptor* aDesc, const void* b, const srtTensorDescriptor* bDesc, int32_t axis,
                    void* out, const srtTensorDescriptor* oDesc, srtStream stream) {
  if (!desc_ok(aDesc) || !desc_ok(bDesc) || !desc_ok(oDesc)) return srtErrorInvalidValue;
  if (!float_type(oDesc->type) || aDesc->type != oDesc->type || bDesc->type != oDesc->type) return srtErrorNotSupported;
  const uint32_t rank = oDesc->rank;
  if (rank > 8) return srtErrorNotSupported;
  if (aDesc->rank != rank || bDesc->rank != rank || axis < 0 || (uint32_t)axis >= rank) return srtErrorInvalidValue;
  if (aDesc->shape[axis] + bDesc->shape[axis] != oDesc->shape[axis]) return srtErrorInvalidValue;
  Map m[2]{};
  bool empty[2];
  for (int i = 0; i < 2; ++i) {
    const srtTensorDescriptor* d = i ? bDesc : aDesc;
    srtTensorDescriptor part = *oDesc;   // the piece of the result that this input fills
    size_t shape[8];
    for (uint32_t k = 0; k < rank; ++k) shape[k] = k == (uint32_t)axis ? d->shape[k] : oDesc->shape[k];
    part.shape = shape;
    if (srtStatus s = build_map(d, nullptr, &part, &m[i], &empty[i]); s != srtSuccess) return s;
    if (!empty[i] && (!(i ? b : a) || !out)) return srtErrorInvalidValue;
    m[i].a = i ? b : a;
    m[i].o = (char*)out + (i ? aDesc->shape[axis] * oDesc->strides[axis] * type_size(oDesc->type) : 0);
  }
  hipStream_t hs = reinterpret_cast<hipStream_t>(stream);
  if (empty[0] && empty[1]) return srtSuccess;
  if (empty[0] || empty[1]) return srt::from_hip(launch_op(kCopy, oDesc->type, m[empty[0] ? 1 : 0], hs));
  if ((m[0].total + m[1].total) * 2 * type_size(oDesc->type) > kOneVectorBytes) {   // bytes, not launches: the plain copy's shape
    if (srtStatus s = srt::from_hip(launch_op(kCopy, oDesc->type, m[0], hs)); s != srtSuccess) return s;
    return srt::from_hip(launch_op(kCopy, oDesc->type, m[1], hs));
  }
  switch (oDesc->type) {
    case srtReal32F: return srt::from_hip(launch_copy_pair<srt::F32>(m[0], m[1], hs));
    case srtReal16F: return srt::from_hip(launch_copy_pair<srt::F16>(m[0], m[1], hs));
    default: return srt::from_hip(launch_copy_pair<srt::BF16>(m[0], m[1], hs));
  }
}

srtStatus srtLstmGates(const void* gates, const srtTensorDescriptor* gatesDesc, const void* cell, const srtTensorDescriptor* cellDesc,
                       void* newCell, const srtTensorDescriptor* newCellDesc, void* newHidden,
                       const srtTensorDescriptor* newHiddenDesc, srtStream stream) {
  const srtTensorDescriptor* all[4] = {gatesDesc, cellDesc, newCellDesc, newHiddenDesc};
  for (const srtTensorDescriptor* d : all) {
    if (!desc_ok(d)) return srtErrorInvalidValue;
    if (!float_type(d->type) || d->type != gatesDesc->type) return srtErrorNotSupported;
    if (d->rank != 2 || d->shape[0] != gatesDesc->shape[0]) return srtErrorInvalidValue;
  }
  const size_t rows = cellDesc->shape[0], columns = cellDesc->shape[1];
  if (gatesDesc->shape[1] != 4 * columns || newCellDesc->shape[1] != columns || newHiddenDesc->shape[1] != columns)
    return srtErrorInvalidValue;
  if (rows == 0 || columns == 0) return srtSuccess;
  if (rows > 0x7fffffffull || columns > 0x7fffffffull) return srtErrorNotSupported;
  if (!gates || !cell || !newCell || !newHidden) return srtErrorInvalidValue;
  GateProblem p{};
  p.rows = (uint32_t)rows; p.columns = (uint32_t)columns;
  p.gates = gates; p.cell = cell; p.new_cell = newCell; p.new_hidden = newHidden;
  p.part = (long long)(columns * gatesDesc->strides[1]);
  p.gates_row = (long long)gatesDesc->strides[0]; p.gates_col = (long long)gatesDesc->strides[1];
  p.cell_row = (long long)cellDesc->strides[0]; p.cell_col = (long long)cellDesc->strides[1];
  p.new_cell_row = (long long)newCellDesc->strides[0]; p.new_cell_col = (long long)newCellDesc->strides[1];
  p.new_hidden_row = (long long)newHiddenDesc->strides[0]; p.new_hidden_col = (long long)newHiddenDesc->strides[1];
  hipStream_t hs = reinterpret_cast<hipStream_t>(stream);
  switch (gatesDesc->type) {
    case srtReal32F: return srt::from_hip(launch_lstm_gates<srt::F32>(p, hs));
    case srtReal16F: return srt::from_hip(launch_lstm_gates<srt::F16>(p, hs));
    default: return srt::from_hip(launch_lstm_gates<srt::BF16>(p, hs));
  }
}

}  // extern "C"
