// One step of an LSTM cell in one launch: [x, h] . W + b, cut into gates, applied to the cell state.
//
// As calls of its own the step is a concatenation, a product and the gate arithmetic: three launches of 3 + 8.5 + 3 us for
// 64 x 512 in fp32, of which the product's k loop is 5, and 14 us more of a program's own time for two more results and calls.  Here
// a workgroup computes the four gates of 8 hidden columns for 32 rows -- a 32 x 32 tile of the product whose columns are four groups
// of 8, H apart -- as the wave-split tiles do (gemm_waves.h), and its epilogue is the cell.
//
//   bound   latency, as those tiles: a round trip to memory per slab of a wave, the sums, the gates
//   k       x's slabs, then h's: each range ends with its own masked slab, and W's rows go on where x's end
//   width   8, or any from 16 up (9 to 15, never measured here, are left to the three calls): a last group of fewer than 8 columns (1 x 384 x 1020
//           f16, a program's step: 39.7 us as three calls, 18.7)
//   W       n-contiguous: a lane's 16 bytes are 8 columns of one gate (fp32: 4, two lanes a gate), so a k row of the tile is 16
//           or 32 bytes in each of four lines, which the neighbouring workgroups share through L2
//   sums    fp32; bias added in fp32 and rounded to the element type, as the product's result is; then lstm_gate
//   order   an XCD takes neighbouring groups (in grid order every XCD fetched every line: 64 x 1024 x 1024 fp32 26.4 us, now 18.3)
//   measured (us, queue calls back to back, three launches / one, fp32; bf16)   8 x 256 x 256 15.6 / 6.5; 15.4 / 6.2,  64 x 512 x 512 14.8 / 9.9;
//           15.5 / 6.4,  64 x 1024 x 1024 21.2 / 18.3; 20.6 / 12.0.  A program's step through the package, 64 x 512 x 512 fp32: 37.4 / 20.0
#include <type_traits>

#include "gemm_waves.h"
#include "lstm_gates.h"
#include "status.h"
#include "views.h"

namespace srt {
namespace {

struct CellProblem {
  int rows, inputs, hidden;             // batch, I, H
  const void *x, *h, *w, *bias, *cell;
  void *new_cell, *new_hidden;
  long long x_row, h_row, w_row, bias_step, cell_row, cell_col, new_cell_row, new_hidden_row;   // elements
};

constexpr int WAVES = 8, GROUP = 8;   // hidden columns of a workgroup
__host__ __device__ constexpr int groups_of(int hidden) { return (hidden + GROUP - 1) / GROUP; }

template <typename T>
__global__ __launch_bounds__(64 * WAVES) void lstm_cell_kernel(CellProblem p) {
  using S = typename T::storage;
  using StageA = waves::Stage<T, true, 1, true>;
  using StageB = waves::Stage<T, false, 1, true>;
  constexpr int DEPTH = StageA::DEPTH, LOADS = StageA::LOADS, EPC = StageA::EPC, SLAB = StageA::BYTES + StageB::BYTES, TILE = 4096;
  extern __shared__ __attribute__((aligned(1024))) unsigned char cell_lds[];
  const uint32_t lds = (uint32_t)(uintptr_t)(SRT_LDS unsigned char*)cell_lds;

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // workgroup x runs on XCD x % 8, which takes its consecutive eighth of the groups: neighbours share W's lines
  const int per_xcd = (groups_of(p.hidden) + 7) / 8, group = (int)(blockIdx.x & 7) * per_xcd + (int)(blockIdx.x >> 3);
  if (group * GROUP >= p.hidden) return;
  const int m0 = blockIdx.y * 32, j0 = group * GROUP;
  const uint32_t lds_a = lds + (uint32_t)(wave * SLAB), lds_b = lds_a + StageA::BYTES;

  // the stages of the two k ranges: x against W's first rows, h against the rest
  const S* w = (const S*)p.w;
  const int piece = lane % StageB::PER_ROW;
  const int column = piece * EPC / GROUP * p.hidden + j0 + piece * EPC % GROUP;
  auto stages = [&](const void* a, long long a_row, const S* b, int depth, StageA* sa, StageB* sb) {
    sa->init((const S*)a, lane, m0, p.rows, a_row, depth);
    sb->init(b, lane, 0, 4 * p.hidden, p.w_row, depth);
    // a last group of fewer than 8 columns reads into the next gate's, for results that are not stored; behind the fourth gate a row ends, and a
    // piece that would cross that end is moved back inside and shifted into place
    const int at = min(column, 4 * p.hidden - EPC);
    sb->ptr[0] = b + at;
    sb->over = column - at;
    sb->edge = j0 + GROUP > p.hidden;
  };
  StageA ax, ah;
  StageB bx, bh;
  stages(p.x, p.x_row, w, p.inputs, &ax, &bx);
  stages(p.h, p.h_row, w + (long long)p.inputs * p.w_row, p.hidden, &ah, &bh);
  const int slabs_x = (p.inputs + DEPTH - 1) / DEPTH, slabs = slabs_x + (p.hidden + DEPTH - 1) / DEPTH;

  waves::f32x16_t acc, more;
#pragma unroll
  for (int v = 0; v < 16; ++v) acc[v] = more[v] = 0.0f;
  waves::u32x4_t ra[LOADS], rb[LOADS];
  auto request = [&](int s) {
    if (s < slabs_x) {
      ax.load(ra, s * DEPTH);
      bx.load(rb, s * DEPTH);
    } else {
      ah.load(ra, (s - slabs_x) * DEPTH);
      bh.load(rb, (s - slabs_x) * DEPTH);
    }
  };
  int s = wave;
  if (s < slabs) request(s);
  for (; s < slabs; s += WAVES) {
    // (where a piece goes is the same in both ranges; what of it counts is not)
    StageA sa = ax;
    StageB sb = bx;
    if (s >= slabs_x) {
      sa.K = ah.K;
      sb.K = bh.K;
    }
    const int k0 = (s < slabs_x ? s : s - slabs_x) * DEPTH;
    sa.store(ra, k0, lds_a);
    sb.store(rb, k0, lds_b);
    if (s + WAVES < slabs) request(s + WAVES);
    // (the slab is this wave's alone: see gemm_waves_kernel)
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    waves::u32x4_t fa[4], fb[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      fa[q] = sa.read(lds_a, 0, q);
      fb[q] = sb.read(lds_b, 0, q);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int i = 0; i < waves::kMfmas<T>; ++i) {
        waves::f32x16_t& sum = sizeof(S) == 4 && (q & 1) ? more : acc;
        sum = waves::mfma<T>(fb[q], fa[q], i, sum);
      }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
  if (sizeof(S) == 4) acc += more;

  // the waves' partial tiles, as in gemm_waves_kernel; a lane of the first four waves adds up four columns of one gate, and their
  // rounded sums meet once more behind the partial tiles
  __syncthreads();
  {
    const int r = lane & 31, h = lane >> 5;
    const uint32_t at = lds + (uint32_t)(wave * TILE + r * 128 + ((h ^ ((r >> 1) & 7)) << 4));
#pragma unroll
    for (int g = 0; g < 4; ++g)
      *reinterpret_cast<SRT_LDS waves::f32x4_t*>(at ^ (uint32_t)(g * 32)) = waves::f32x4_t{acc[4 * g], acc[4 * g + 1], acc[4 * g + 2], acc[4 * g + 3]};
  }
  __syncthreads();
  const uint32_t sums = lds + WAVES * TILE;   // [32 rows][33 columns]: gate g of column j at 8 g + j
  if (tid < 256) {
    const int row = tid >> 3, c = tid & 7;
    const uint32_t at = lds + (uint32_t)(row * 128 + ((c ^ ((row >> 1) & 7)) << 4));
    waves::f32x4_t part[WAVES];
#pragma unroll
    for (int i = 0; i < WAVES; ++i) part[i] = *reinterpret_cast<const SRT_LDS waves::f32x4_t*>(at + (uint32_t)(i * TILE));
#pragma unroll
    for (int step = 1; step < WAVES; step *= 2)
#pragma unroll
      for (int i = 0; i < WAVES; i += 2 * step) part[i] += part[i + step];
    const int j = j0 + (c & 1) * 4;
    const S* bias = (const S*)p.bias + (long long)((c >> 1) * p.hidden) * p.bias_step;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      *reinterpret_cast<SRT_LDS float*>(sums + (uint32_t)((row * 33 + 4 * c + e) * 4)) =
          T::to_float(T::from_float(part[0][e] + T::to_float(bias[(long long)min(j + e, p.hidden - 1) * p.bias_step])));
  }
  __syncthreads();
  if (tid < 256) {
    const int row = tid >> 3, j = tid & 7, m = m0 + row, n = j0 + j;
    if (m >= p.rows || n >= p.hidden) return;
    float gate[4];
#pragma unroll
    for (int g = 0; g < 4; ++g) gate[g] = *reinterpret_cast<const SRT_LDS float*>(sums + (uint32_t)((row * 33 + 8 * g + j) * 4));
    const float cell = T::to_float(((const S*)p.cell)[(long long)m * p.cell_row + (long long)n * p.cell_col]);
    S nc, nh;
    lstm_gate<T>(gate[0], gate[1], gate[2], gate[3], cell, &nc, &nh);
    ((S*)p.new_cell)[(long long)m * p.new_cell_row + n] = nc;
    ((S*)p.new_hidden)[(long long)m * p.new_hidden_row + n] = nh;
  }
}

template <typename T>
hipError_t launch(const CellProblem& p, hipStream_t stream) {
  constexpr int lds_bytes = WAVES * 8192;
  static std::atomic<uint32_t> configured{0};
  const void* kernel = reinterpret_cast<const void*>(lstm_cell_kernel<T>);
  if (hipError_t e = ensure_lds_limit(kernel, lds_bytes, configured); e != hipSuccess) return e;
  hipLaunchKernelGGL(lstm_cell_kernel<T>, dim3(8 * ((groups_of(p.hidden) + 7) / 8), (p.rows + 31) / 32), dim3(64 * WAVES), lds_bytes, stream, p);
  return launch_status(stream);
}

// Whether one launch is ahead of the three.  On the device it is while k is short against the product's own kernels, which cut a long one over idle
// units and read the weight in larger tiles; a program's step is ahead up to 35 us of it, which its own three calls take on the host (37 us, of
// which one call takes 20).  By the depth D = I + H and the slabs a unit walks (D times its tiles); device times of 420 cells of 1-512 x 64-16384 x
// 8-2048, three / one, us, bf16: 32 x 1024 x 1024 18.8 / 9.5, 8 x 2048 x 1024 21.7 / 12.3, 64 x 512 x 2048 24.2 / 30.4 (taken: under 35), but 128 x
// 4096 x 1024 27.5 / 50.7, 8 x 8192 x 256 26.4 / 36.9; fp32 64 x 1024 x 1024 21.0 / 18.8, 128 x 1024 x 1024 36.3 / 33.4, but 64 x 1024 x 2048 41.5 / 48.5,
// 64 x 8192 x 2048 122 / 214.  Up to four groups of columns a product of few columns idles as well: 64 x 16384 x 8 55.9 / 21.9.  A program's
// step is 0.4 % (bf16) and 0.2 % (fp32) behind the better of the two in the mean, 10 % and 5 % by the bound of two tiles a unit alone.
bool launch_choice(const CellProblem& p, bool f32) {
  const long long tiles = (long long)((p.rows + 31) / 32) * groups_of(p.hidden), cus = compute_units();
  const long long depth = (long long)p.inputs + p.hidden;
  if (tiles > 2 * cus || (depth > (f32 ? 8192 : 5200) && p.hidden > 32)) return false;
  // (widths off the groups of eight, whose weight rows are mostly off 16 bytes, take up to twice as long, one / three, us: bf16 6 x 2975 x 2079 75 / 37,
  // f16 2 x 1245 x 2415 55 / 35, f32 78 x 2842 x 663 55 / 36.  84 programs' steps between these bounds and the other widths': three calls 1.11x as
  // fast in steps that follow each other, and in the first one on new operands 1.05x in 16 bits, 0.87x in fp32)
  if (p.hidden % 8 != 0) return depth * tiles <= (f32 ? 3400 : p.hidden % 2 == 0 ? 4500 : tiles > cus ? 3400 : 3800) * cus;
  return depth * tiles <= (f32 ? 4200 : 5200) * cus;
}

bool row_ok(long long stride) { return stride >= 0 && stride <= 0x7fffffffLL; }

}  // namespace
}  // namespace srt

extern "C" srtStatus srtLstmCell(const void* x, const srtTensorDescriptor* xDesc, const void* hidden, const srtTensorDescriptor* hiddenDesc,
                                 const void* weight, const srtTensorDescriptor* weightDesc, const void* bias, const srtTensorDescriptor* biasDesc,
                                 const void* cell, const srtTensorDescriptor* cellDesc, void* newCell, const srtTensorDescriptor* newCellDesc,
                                 void* newHidden, const srtTensorDescriptor* newHiddenDesc, srtStream stream) {
  const srtTensorDescriptor* all[7] = {xDesc, hiddenDesc, weightDesc, biasDesc, cellDesc, newCellDesc, newHiddenDesc};
  for (const srtTensorDescriptor* d : all) {
    if (!d || !d->shape || !d->strides) return srtErrorInvalidValue;
    if (d->type != srtReal32F && d->type != srtReal16F && d->type != srtReal16BF) return srtErrorNotSupported;
    if (d->type != xDesc->type) return srtErrorNotSupported;
    if (d->order != srtOrderRow) return srtErrorNotSupported;
    if (d->rank != (d == biasDesc ? 1u : 2u)) return srtErrorNotSupported;
  }
  const size_t rows = xDesc->shape[0], inputs = xDesc->shape[1], units = hiddenDesc->shape[1];
  // shapes that are not a cell's are the caller's to run operator by operator (gates may broadcast, a weight may have more columns)
  if (hiddenDesc->shape[0] != rows || weightDesc->shape[0] != inputs + units || weightDesc->shape[1] != 4 * units ||
      biasDesc->shape[0] != 4 * units)
    return srtErrorNotSupported;
  for (const srtTensorDescriptor* d : {cellDesc, newCellDesc, newHiddenDesc})
    if (d->shape[0] != rows || d->shape[1] != units) return srtErrorNotSupported;
  const size_t per = xDesc->type == srtReal32F ? 4 : 8, lim = 1u << 26;
  if (rows == 0 || rows > lim || inputs > lim || units > lim || inputs < per || units < 8 || (units % 8 != 0 && units < 16)) return srtErrorNotSupported;
  for (const srtTensorDescriptor* d : {xDesc, hiddenDesc, weightDesc, newCellDesc, newHiddenDesc})
    if (d->strides[1] != 1 || !srt::row_ok((long long)d->strides[0])) return srtErrorNotSupported;
  if (!x || !hidden || !weight || !bias || !cell || !newCell || !newHidden) return srtErrorInvalidValue;
  if ((long long)cellDesc->strides[0] < 0 || (long long)cellDesc->strides[1] < 0 || (long long)biasDesc->strides[0] < 0) return srtErrorNotSupported;

  srt::CellProblem p;
  p.rows = (int)rows; p.inputs = (int)inputs; p.hidden = (int)units;
  p.x = x; p.h = hidden; p.w = weight; p.bias = bias; p.cell = cell; p.new_cell = newCell; p.new_hidden = newHidden;
  p.x_row = (long long)xDesc->strides[0]; p.h_row = (long long)hiddenDesc->strides[0]; p.w_row = (long long)weightDesc->strides[0];
  p.bias_step = (long long)biasDesc->strides[0];
  p.cell_row = (long long)cellDesc->strides[0]; p.cell_col = (long long)cellDesc->strides[1];
  p.new_cell_row = (long long)newCellDesc->strides[0]; p.new_hidden_row = (long long)newHiddenDesc->strides[0];
  if (!srt::launch_choice(p, per == 4) || (rows + 31) / 32 > 65535) return srtErrorNotSupported;

  // workgroups read x, h and the weight while others store: the results share no memory with any operand, nor with one another
  const size_t es = per == 4 ? 4 : 2;
  auto view = [&](const void* base, const srtTensorDescriptor* d) {
    const bool one = d->rank == 1;
    return srt::make_view(base, es, (long long)d->shape[0], (long long)d->strides[0], one ? 1 : (long long)d->shape[1], one ? 0 : (long long)d->strides[1], 1, 0);
  };
  const srt::StridedView nc = view(newCell, newCellDesc), nh = view(newHidden, newHiddenDesc);
  if (srt::spans_overlap(nc, nh)) return srtErrorNotSupported;
  const void* bases[5] = {x, hidden, weight, bias, cell};
  for (int i = 0; i < 5; ++i) {
    const srt::StridedView v = view(bases[i], all[i]);
    if (srt::spans_overlap(nc, v) || srt::spans_overlap(nh, v)) return srtErrorNotSupported;
  }
  hipStream_t hs = reinterpret_cast<hipStream_t>(stream);
  switch (xDesc->type) {
    case srtReal32F: return srt::from_hip(srt::launch<srt::F32>(p, hs));
    case srtReal16F: return srt::from_hip(srt::launch<srt::F16>(p, hs));
    default: return srt::from_hip(srt::launch<srt::BF16>(p, hs));
  }
}
