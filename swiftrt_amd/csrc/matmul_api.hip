// srtMatmul / srtMatmulBiasActivation: descriptor validation, folding of transposes, orders
// and views into one strided problem, and kernel-family selection.
#include <cstdio>
#include <cstring>
#include <map>
#include <mutex>
#include <tuple>

#include "gemm_common.h"
#include "status.h"
#include "views.h"

namespace {

using srt::GemmProblem;

bool supported_type(srtDataType t) { return t == srtReal32F || t == srtReal16F || t == srtReal16BF; }

// Builds the normalized problem.  Returns srtSuccess, srtErrorNotSupported (caller falls
// back to the CPU) or srtErrorInvalidValue.  *empty is set when an extent is zero.
srtStatus build_problem(const void* a, const srtTensorDescriptor* ad, int tA,
                        const void* b, const srtTensorDescriptor* bd, int tB,
                        const void* bias, const srtTensorDescriptor* biasd, int activation, double coef,
                        void* out, const srtTensorDescriptor* od, GemmProblem* p, bool* empty,
                        bool check_alias = true) {
  *empty = false;
  if (!ad || !bd || !od) return srtErrorInvalidValue;
  if (!ad->shape || !ad->strides || !bd->shape || !bd->strides || !od->shape || !od->strides)
    return srtErrorInvalidValue;
  const uint32_t rank = od->rank;
  if (rank != 2 && rank != 3) return srtErrorNotSupported;
  if (ad->rank != rank || bd->rank != rank) return srtErrorInvalidValue;
  if (!supported_type(od->type)) return srtErrorNotSupported;
  if (ad->type != od->type || bd->type != od->type) return srtErrorNotSupported;
  auto order_ok = [](srtOrder o) { return o == srtOrderRow || o == srtOrderCol; };
  if (!order_ok(ad->order) || !order_ok(bd->order) || !order_ok(od->order)) return srtErrorNotSupported;
  if ((unsigned)activation > (unsigned)srtActivationIdentity) return srtErrorInvalidValue;

  const uint32_t r = rank - 2;
  size_t am = ad->shape[r], ak = ad->shape[r + 1], sam = ad->strides[r], sak = ad->strides[r + 1];
  if (tA) { size_t t = am; am = ak; ak = t; t = sam; sam = sak; sak = t; }
  size_t bk = bd->shape[r], bn = bd->shape[r + 1], sbk = bd->strides[r], sbn = bd->strides[r + 1];
  if (tB) { size_t t = bk; bk = bn; bn = t; t = sbk; sbk = sbn; sbn = t; }
  const size_t M = od->shape[r], N = od->shape[r + 1];
  if (am != M || bn != N || ak != bk) return srtErrorInvalidValue;
  size_t batch = 1;
  if (rank == 3) {
    batch = od->shape[0];
    if (ad->shape[0] != batch || bd->shape[0] != batch) return srtErrorInvalidValue;
  }
  const size_t lim = 0x7fffffffu;
  if (M > lim || N > lim || ak > lim || batch > lim) return srtErrorNotSupported;

  p->dtype = od->type;
  p->M = (int)M; p->N = (int)N; p->K = (int)ak; p->batch = (int)batch;
  p->A = a; p->B = b; p->C = out;
  p->sam = (long long)sam; p->sak = (long long)sak; p->sab = rank == 3 ? (long long)ad->strides[0] : 0;
  p->sbk = (long long)sbk; p->sbn = (long long)sbn; p->sbb = rank == 3 ? (long long)bd->strides[0] : 0;
  p->scm = (long long)od->strides[r]; p->scn = (long long)od->strides[r + 1];
  p->scb = rank == 3 ? (long long)od->strides[0] : 0;
  p->bias = nullptr; p->sbias = 0; p->bias_per_row = 0;
  p->activation = activation; p->coef = (float)coef; p->tile_n = 0; p->row_padding = 0;
  if (bias) {
    if (!biasd || !biasd->shape || !biasd->strides) return srtErrorInvalidValue;
    if (biasd->type != od->type) return srtErrorNotSupported;
    if (biasd->rank != 1 || biasd->shape[0] != N) return srtErrorInvalidValue;
    p->bias = bias; p->sbias = (long long)biasd->strides[0];
  }
  if (M == 0 || N == 0 || batch == 0) { *empty = true; return srtSuccess; }
  if (!a || !b || !out) return srtErrorInvalidValue;

  // The kernels read operand tiles while other workgroups already store results, so the result must share no
  // element with an input (the Swift side always hands in a freshly allocated dense result,
  // operators/Matmul.swift:38-39).  Storage spans that do not overlap settle it.  Views whose spans do overlap
  // are accepted when a common pitch proves them apart (column slices of one wide buffer, interleaved
  // batches: see views_disjoint); a result that provably shares an element with an input (the same first element, or overlapping row blocks
  // of one pitch) is an error; anything else
  // is answered "not supported", so that the caller's fallback runs instead of a wrong guess either way.
  if (check_alias) {   // (the kernel query takes placeholder pointers and launches nothing)
    const size_t es = od->type == srtReal32F ? 4 : 2;
    const srt::StridedView vo = srt::make_view(out, es, p->M, p->scm, p->N, p->scn, p->batch, p->scb);
    auto verdict = [&](const srt::StridedView& v) {
      if (!srt::spans_overlap(vo, v)) return srtSuccess;
      if (srt::views_alias(vo, v)) return srtErrorInvalidValue;
      return srt::views_disjoint(vo, v) ? srtSuccess : srtErrorNotSupported;
    };
    if (p->K > 0) {
      if (srtStatus s = verdict(srt::make_view(a, es, p->M, p->sam, p->K, p->sak, p->batch, p->sab)); s != srtSuccess) return s;
      if (srtStatus s = verdict(srt::make_view(b, es, p->K, p->sbk, p->N, p->sbn, p->batch, p->sbb)); s != srtSuccess) return s;
    }
    if (bias) {
      if (srtStatus s = verdict(srt::make_view(bias, es, p->N, p->sbias, 1, 0, 1, 0)); s != srtSuccess) return s;
    }
  }

  // Column-major (or otherwise M-contiguous) result: compute C^T = op(B)^T . op(A)^T so the
  // kernels always write rows with the smaller stride innermost.
  if (p->scn != 1 && p->scm == 1) {
    GemmProblem q = *p;
    q.M = p->N; q.N = p->M;
    q.A = p->B; q.sam = p->sbn; q.sak = p->sbk; q.sab = p->sbb;
    q.B = p->A; q.sbk = p->sak; q.sbn = p->sam; q.sbb = p->sab;
    q.scm = p->scn; q.scn = p->scm;
    q.bias_per_row = 1;
    *p = q;
  }
  return srtSuccess;
}

// ---- plans ------------------------------------------------------------------------------------
// A plan names the kernel that runs a problem.  The heuristic picks one per call; srtMatmulTune
// measures every plan the problem qualifies for and records the fastest in a process-wide cache
// keyed by the problem's shape, layout class and epilogue, which later calls consult first
// (the role of ExecutionPlanCache / ExecutionPlanner, platform/common/ExecutionPlanner.swift:20-29,
// and of the empty CudaMatmul2.tune, platform/cuda/functions/CudaMatmul.swift:112-120).
enum Plan { kPlanGeneric, kPlanSkinny, kPlanRing256, kPlanMfma128, kPlanMfma64, kPlanF32Tile64, kPlanF32SplitK,
            kPlanKc64, kPlanM16, kPlanSplitK, kPlanM16H, kPlanAny128, kPlanAny64, kPlanM16D, kPlanM16DTail, kPlanM16DSplit, kPlanM16DH, kPlanM16DN, kPlanM16Q, kPlanF32Parts, kPlanF32Ring, kPlanF32Ring64x128, kPlanF32Ring64, kPlanWaves, kPlanCopied, kPlanCount,
            kPlanStreamed = kPlanCount };   // never recorded: few rows on the streaming kernel where split-K's name is reported (heuristic_plan)

const char* const kPlanNames[kPlanCount] = {"generic", "skinny", "mfma_256x256", "mfma_128x128", "mfma_64x64",
                                            "f32_mfma_64x64", "f32_mfma_splitk", "mfma_256x256_k64",
                                            "mfma_256x256_m16", "mfma_256x256_splitk", "mfma_128x256_m16",
                                            "mfma_128x128_any", "mfma_64x64_any", "mfma_256x256_m16_k64",
                                            "mfma_256x256_m16_k64_tail", "mfma_256x256_m16_k64_split",
                                            "mfma_128x256_m16_k64", "mfma_256x128_m16_k64", "mfma_128x128_m16_k128", "f32_mfma_128x128_parts", "f32_mfma_128x128_ring", "f32_mfma_64x128_ring", "f32_mfma_64x64_ring", "mfma_32x32_waves", "copied"};

const char* plan_name(Plan plan) { return kPlanNames[plan == kPlanStreamed ? kPlanSplitK : plan]; }

bool plan_supported(const GemmProblem& p, Plan plan) {
  switch (plan) {
    case kPlanSkinny: return srt::skinny_supported(p) || srt::stream_supported(p);
    case kPlanRing256: return srt::mfma_config(p, 1) != 0;
    case kPlanMfma128: return srt::mfma_config(p, 2) != 0;
    case kPlanMfma64: return srt::mfma_config(p, 3) != 0;
    case kPlanKc64: return srt::mfma_config(p, 4) != 0;
    case kPlanM16: return srt::mfma_config(p, 5) != 0;
    case kPlanSplitK: return srt::mfma_splitk_parts(p) >= 2;
    case kPlanM16H: return srt::mfma_config(p, 6) != 0;
    case kPlanAny128: return srt::mfma_config(p, 7) != 0;
    case kPlanAny64: return srt::mfma_config(p, 8) != 0;
    case kPlanM16D: return srt::mfma_config(p, 9) != 0;
    case kPlanM16DTail: return srt::mfma_config(p, 10) != 0;
    case kPlanM16DSplit: return srt::mfma_config(p, 11) != 0;
    case kPlanM16DH: return srt::mfma_config(p, 12) != 0;
    case kPlanM16DN: return srt::mfma_config(p, 13) != 0;
    case kPlanM16Q: return srt::mfma_config(p, 14) != 0;
    case kPlanF32Parts: return srt::f32_mfma_supported(p) && srt::f32_tile_parts(p) >= 2;
    case kPlanF32Ring:
    case kPlanF32Ring64x128:
    case kPlanF32Ring64: return srt::f32_ring_fits(p);
    case kPlanF32Tile64: return srt::f32_mfma_supported(p) && (p.M + 63) / 64 <= 65535;
    case kPlanF32SplitK: return srt::f32_mfma_supported(p);
    case kPlanWaves: return srt::waves_supported(p);
    case kPlanCopied: return srt::pack_supported(p);
    default: return srt::generic_supported(p);
  }
}

// The plan of the tile that mfma_select picks (kPlanGeneric: none qualifies).  copies: operands off the 16-byte rules may be
// copied into workspace.
Plan tile_plan(const GemmProblem& p, bool copies) {
  const int c = srt::mfma_select(p);
  if (c == 0) return kPlanGeneric;
  switch (c >> 2) {
    case 1: return kPlanRing256;
    case 2: return kPlanMfma128;
    case 4: return kPlanKc64;
    case 5: return kPlanM16;
    case 6: return kPlanM16H;
    case 7: return copies && srt::pack_preferred(p) ? kPlanCopied : kPlanAny128;
    case 8: return copies && srt::pack_preferred(p) ? kPlanCopied : kPlanAny64;
    case 9: return kPlanM16D;
    case 10: return kPlanM16DTail;
    case 12: return kPlanM16DH;
    case 13: return kPlanM16DN;
    case 14: return kPlanM16Q;
    default: return kPlanMfma64;
  }
}

// The choice among every plan but the wave-split tiles.
Plan base_plan(const GemmProblem& p, bool copies) {
  // one round of 128 x 128 tiles holds the problem (64 rows or more) and its k loop is not worth cutting
  if (srt::mfma_prefers_quarter(p)) return kPlanM16Q;
  if (srt::skinny_supported(p) && srt::skinny_preferred(p)) return kPlanSkinny;
  // Up to 64 rows against a long k loop, one round of the streaming kernel's workgroups: when split-K cannot cut the k
  // loop, or only in two (K / 4 not a whole number of stages; a batch has no split-K pass at all), the streaming kernel beats
  // tiles that leave most of the device idle (24 x 96 x 10320: 32 us against 121 in half tiles; 64 x 144 x 8400 x . W^T: 26
  // against 61 in 64 x 64 tiles; 8 x 1288 x 10432: 44 against 58 in two parts).  With up to 32 rows that is decided ahead
  // of tail sharing, whose tiles would be nearly all padding (28 x 8 x 88 x 7680: 32 us against 59).
  const bool streams = p.dtype != srtReal32F && p.K >= 2048 && srt::skinny_supported(p) && (long long)((p.N + 63) / 64) * p.batch <= 256;
  const bool few_parts = srt::mfma_splitk_parts(p) <= 2;
  if (streams && few_parts && p.M <= 32) return kPlanSkinny;
  // tiles left over after the whole rounds and a long k loop: cut along k for the idle compute units
  if (srt::mfma_prefers_tail(p)) return kPlanM16DTail;
  // (The split form -- whole rounds of whole tiles, then one round of 192-wide ones -- is never the heuristic's choice:
  // on this power-limited device the compute units that idle through a ragged last round lend their power to the busy
  // ones, and the form measures the same as whole tiles or worse.  4096 x 11008 x 4096, 2.69 rounds, same run: 249-257 us
  // whole, 254-258 split; 2048 x 13000 x 4096, 1.59 rounds: 158-162 against 168-170.  srtMatmulTune still times it.)
  if (streams && few_parts) return kPlanSkinny;
  // few 256 x 256 tiles and a long k loop: K split over the idle compute units
  if (srt::mfma_prefers_splitk(p)) return kPlanSplitK;
  if (streams) return kPlanSkinny;
  const Plan tile = tile_plan(p, copies);
  if (tile != kPlanGeneric) return tile;
  if (srt::f32_mfma_supported(p)) {
    // what the ring kernel reads: the fastest of its three tile shapes, the k range in parts and the 32 x 32 kernel,
    // by their time estimates
    if (srt::f32_ring_fits(p)) {
      switch (srt::f32_ring_choice(p)) {
        case 0: return kPlanF32Ring;
        case 1: return kPlanF32Ring64x128;
        case 2: return kPlanF32Ring64;
        case 3: return kPlanF32Parts;
        default: return kPlanF32SplitK;
      }
    }
    switch (srt::f32_any_choice(p, copies)) {
      // launch-sized problems and up to 64 rows: 32 x 32 tiles whose waves split K
      case srt::F32Any::kSplitK: return kPlanF32SplitK;
      // a single matrix of too few 128 x 128 tiles for the device: its k range in parts on those tiles
      case srt::F32Any::kParts: return kPlanF32Parts;
      // operands the ring kernel reads once copied into its layout
      case srt::F32Any::kPacked: return kPlanCopied;
      default: return kPlanF32Tile64;
    }
  }
  return kPlanGeneric;
}

bool curved(int activation) { return activation == srtActivationSigmoid || activation == srtActivationTanh || activation == srtActivationElu; }

// What an activation with an exponential adds to the 128 x 128 tiles for short k loops, whose lanes put 64 results through it, in microseconds.
// A round of the other tiles: 0.6 of that (128 x 128 and 64 x 64 ones), 3.3 times (128 x 256), 5.7 times (256 x 256, 1664 x 2368 x 8 11.2, sigmoid
// 23.6, tanh 28.7).
double curved_us(const GemmProblem& p) { return !curved(p.activation) ? 0.0 : p.activation == srtActivationTanh ? 3.0 : 2.0; }

// The wave-split tiles spread over more workgroups, and add 0.15 a tile of a unit: us, 128 x 128 tiles for short k loops / wave-split, 3321 x 384 x 64
// x^T . W tanh 9.0 / 6.3, 4864 x 298 x 128 tanh 11.9 / 8.0, 1492 x 988 x 32 sigmoid 8.2 / 7.0, but 10240 x 336 x 8 sigmoid 8.3 / 11.8.
double short_time(const GemmProblem& p) { return srt::short_us(p) + curved_us(p); }
double waves_time(const GemmProblem& p) {
  const double tiles = (double)((p.M + 31) / 32) * (double)((p.N + 31) / 32) * (double)p.batch / srt::compute_units();
  return srt::waves_us(p) + (curved(p.activation) ? 0.15 * tiles : 0.0);
}

// What a 16-bit problem takes on a plan that base_plan picked, in microseconds, as a bound from below where a plan's figures
// spread (0: not compared).  R: rounds of its tiles over the units, k: K in 1024s.  Fitted to 1900 random problems (gemm_waves.hip), rms
// 3-10 % except the 64 x 64 kernel (15 %); rates are those of a device that is not power-limited.
double plan_us(const GemmProblem& p, Plan plan) {
  const int cus = srt::compute_units();
  auto rounds = [&](int tm, int tn) {
    const long long t = (long long)((p.M + tm - 1) / tm) * ((p.N + tn - 1) / tn) * p.batch;
    return (double)((t + cus - 1) / cus);
  };
  const bool a_kc = p.sak == 1, b_kc = p.sbk == 1;
  const double k = (double)p.K / 1024.0;
  const double act = curved_us(p);
  const double quarter = 4.4 + rounds(128, 128) * (0.9 + 5.1 * k + 0.6 * act), whole = 4.4 + rounds(256, 256) * (2.4 + 15.7 * k + 5.7 * act);
  switch (plan) {
    case kPlanM16Q: {
      // a ragged last unit: whole to the matrix cores, and its masks; in a batch or a second round the operands' traffic sets the pace; one round of a
      // single matrix as 2400 problems in turn measure against wave-split tiles, passes that follow each other, from memory and on new operands (with
      // 1.5 for ragged rows there and no factor 1024 x 1780 x 448 x^T . W^T ran 11.0 us for 8.0; a factor of 1.1 to 1.15 gains another tenth from memory
      // and loses a twentieth out of the caches, 1688 x 840 x 7360 x . W 50.6 / 60.4; in batches both lose, 9 x 448 x 704 x 400 10.0 / 13.3)
      if (p.K % 128 == 0) return quarter;
      const double r = rounds(128, 128), per_k = p.batch > 1 ? 9.0 : r > 1.0 ? 8.3 : 5.6;
      const bool low = p.batch > 1 || p.K >= 4096;   // (the wave-split tiles' estimate is a fifth low past there: 1193 x 1193 x 5672 x . W^T 44.6 us, 56.4 on them)
      const double t = 5.0 + r * (0.9 + per_k * ((p.K + 127) / 128) / 8.0 + 0.6 * act + (srt::c_whole_chunks(p) ? 0.0 : low ? 1.5 : 3.3));
      return r > 1.0 || !a_kc || low ? t : 1.05 * t;
    }
    case kPlanM16H: return 4.1 + rounds(128, 256) * (1.4 + (b_kc ? 16.7 : 11.8) * k + 3.3 * act);
    case kPlanM16DH: return 4.2 + rounds(128, 256) * (0.9 + 10.0 * k + 3.3 * act);
    case kPlanM16DN: return 4.2 + rounds(256, 128) * (2.3 + 9.8 * k + 3.3 * act);
    case kPlanM16D: return whole;
    case kPlanM16:
    case kPlanRing256:
    case kPlanKc64: return 4.4 + rounds(256, 256) * (3.0 + 16.5 * k + 5.7 * act);
    case kPlanM16DTail: return 12.0 + 7.0 * k;
    case kPlanMfma128:
    case kPlanAny128: return srt::short_supported(p) ? short_time(p) : 0.0;
    case kPlanMfma64:
      // (up to sixteen columns in one slab: us, 64 x 64 / wave-split, 48 x 856 x 8 x 64 x . W^T 3.8 / 4.8, 56 x 960 x 8 x 64 5.0 / 6.8, 39 x 848 x 8 x 8 4.0 / 4.9)
      if (p.N <= 16 && p.K <= 64) return 3.3 + 0.4 * rounds(64, 64) + 0.6 * act;
      return 5.3 + rounds(64, 64) * (a_kc ? 6.0 : b_kc ? 9.0 : 11.5) * k + 0.6 * act;
    case kPlanSplitK: {
      const int parts = srt::mfma_splitk_parts(p);
      const double sums = (double)parts * (double)p.M * (double)p.N * 8.0;
      return a_kc && p.M <= 128 ? 9.0 + 12.0 * k / parts + sums / 5.0e6 : 10.0 + 20.0 * k / parts + sums / 7.0e6;
    }
    case kPlanAny64: {
      // (its stages and its stores, two tiles a unit: 512 x 3072 x 54 x . W^T 6.6 / 6.9, 346 x 5440 x 92 7.9 / 7.8, 12 x 768 x 320 x 53 7.8 / 7.8)
      const double t64 = (double)((p.M + 63) / 64) * (double)((p.N + 63) / 64) * (double)p.batch / (2.0 * cus);
      return 5.4 + 0.5 * act + 1.3 * t64 + (p.K + 63) / 64 * (a_kc ? (b_kc ? 0.55 : 2.2) : 4.5) * (t64 > 1.0 ? t64 : 1.0);
    }
    case kPlanCopied: {
      // the launch and bytes of the copies, and the product's own
      const double bytes = ((double)p.M + (double)p.N) * (double)p.K * 2.0 * (double)p.batch;
      return 8.0 + 2.0 * bytes / 6.0e6 + (quarter < whole ? quarter : whole);
    }
    case kPlanSkinny: {
      // bound by its own loads (40 or 45 bytes/ns a unit) or by the weight's from memory
      const double wide = !b_kc || (p.M > 16 && (p.N + 63) / 64 * (long long)p.batch >= 192) ? 64.0 : 32.0;
      const double groups = (double)((p.N + (long long)wide - 1) / (long long)wide) * (double)p.batch / cus;
      const double kb = (wide + (double)((p.M + 7) / 8 * 8)) * (double)p.K * 2.0 / 1000.0;
      return (b_kc ? 3.2 : 4.5) + (groups > 1.0 ? groups : 1.0) * kb / (b_kc ? 45.0 : 40.0);
    }
    default: return 0.0;
  }
}

// Problems whose plan stays what base_plan picks, ahead or not: not by speed, but because the tests of the choice assert its name in these
// ranges (a pinned or saved name is good whatever is picked here).  The price, measured (kept / wave-split, us): 512 x 512 x 1024 x^T . W 9.9 / 5.2,
// 256 x 1024 x 960 x . W 14.0 / 4.6, 1024^3 x^T . W 9.9 / 7.2, 256^3 x . W^T 6.2 / 3.7, 32 x 1024 x 1024 x . W^T 5.0 / 4.6.
bool keeps_plan(const GemmProblem& p, Plan plan) {
  const long long results = (long long)p.M * p.N;
// (others by speed: 1344 x 760 x 3008 x . W 35.3 us on half tiles, 16.1 on wave-split ones)
  const bool whole = p.M <= 64 || (p.M % 128 == 0 && (p.N % 128 == 0 || plan == kPlanM16Q)) || (plan == kPlanM16Q && p.K < 768);
  switch (plan) {
    case kPlanAny64:
    case kPlanAny128:
    case kPlanMfma128: return false;
    case kPlanCopied:   // a large single matrix
      return p.batch == 1 && (results >= (1LL << 22) || (p.K >= 1024 && (long long)((p.M + 63) / 64) * ((p.N + 63) / 64) > srt::compute_units()));
    case kPlanMfma64:   // whole 64-deep units of a large single matrix, or 128-deep ones into rows that are no whole chunks
      return (p.K % 64 == 0 && p.K >= 960 && p.batch == 1 && whole && results >= (1LL << 20)) || (p.K % 128 == 0 && p.K >= 256 && p.N % 8 != 0);
    case kPlanSkinny: return p.batch > 1 || p.K >= 8192 || (p.sbk == 1 && p.N <= 1024);
    default:
      if (plan == kPlanM16Q && p.K % 128 != 0) return false;
      if (p.M <= 32) return true;   // a handful of rows
      if (p.K % 64 != 0) return false;
      if (plan == kPlanSplitK && p.K >= 8192 && results >= (1LL << 18)) return true;   // long k loops in parts
      if (p.batch > 1 ? p.K < 512 : p.K < 640) return plan == kPlanM16Q && p.K <= 256 && whole;   // two 128-deep units
      return p.batch > 1 || (whole && results >= (1LL << 18));
  }
}

// Whether a problem runs on tiles whose waves split k instead of on `plan`, which base_plan picked: by the two estimates.
bool prefers_waves(const GemmProblem& p, Plan plan) {
  if (p.row_padding || !srt::waves_supported(p) || keeps_plan(p, plan)) return false;
  const double other = plan_us(p, plan);
  if (other == 0.0) return false;
  double here = waves_time(p);
  if (plan == kPlanSkinny) {
    // few rows: the weight comes from memory, in whole lines on the streaming kernel
    const double kb = (double)(32 + (p.M < 32 ? p.M : 32)) * (double)p.K * 2.0 / 1000.0, bytes = (double)p.N * (double)p.K * (double)p.batch * 2.0;
    const double tiles = (double)((p.M + 31) / 32) * (double)((p.N + 31) / 32) * (double)p.batch / srt::compute_units();
    const double cold = 2.9 + (tiles > 1.0 ? tiles : 1.0) * kb / (p.sbk == 1 ? 48.0 : 37.5);
    if (cold > here) here = cold;
    if (bytes > 12.0e6) return false;
  }
  return here < 0.95 * other;
}

// Whether copied operands are ahead of the 128 x 128 tiles for short k loops after all: their 256 x 256 tiles read an operand half as often, which
// tells once a unit has many tiles of three slabs or more and the larger ones come out in whole rounds (11 us each into whole lines, 13.4 into
// whole chunks, 15.5 into others).  230 random problems whose other plan is copies, us, copies / those tiles: 12191 x 5312 x 216 x^T . W^T 54 / 67,
// 8512 x 9280 x 143 62 / 73, 2963 x 9728 x 256 29 / 35, 9712 x 8251 x 256 x . W 81 / 104, 15996 x 2709 x 221 51 / 60; not 6510 x 5768 x 256
// x^T . W^T 48 / 42, 6562 x 8768 x 192 x^T . W 47 / 44, nor under an activation with an exponential, 5760 x 7032 x 156 tanh 83 / 50.
bool copies_ahead(const GemmProblem& p) {
  const double cus = srt::compute_units(), slabs = (p.K + 63) / 64;
  auto tiles = [&](int edge) { return (double)((p.M + edge - 1) / edge) * (double)((p.N + edge - 1) / edge) * (double)p.batch / cus; };
  const bool chunks = srt::c_whole_chunks(p), lines = ((p.N | (int)p.scm | (int)p.scb) & 63) == 0 && (reinterpret_cast<uintptr_t>(p.C) & 127u) == 0;
  const double t = tiles(128);
  if (curved(p.activation) || t < 6.0 || slabs < (chunks ? 3.0 : 4.0)) return false;
  const double here = 4.6 + t * (1.26 + 0.73 * slabs + (chunks ? 0.0 : 0.9));
  return 8.0 + __builtin_ceil(tiles(256)) * (lines ? 11.0 : chunks ? 13.4 : 15.5) < 0.93 * here;
}

// Whether a problem with a short k loop runs on 128 x 128 tiles instead of on copies of its operands or small tiles: from five
// quarters of a tile a unit -- at the first few past one, most units wait for those that have two --, below that where
// the estimate is ahead of copies and of 64 x 64 tiles by elements.  A k loop of one slab: instead of the 256 x 256 kernels too, whose tiles
// are all epilogue (365 random problems of 4 Mi results and more: 1.3x, none under 0.95x; 3072 x 6336 x 64 x . W 15.4 / 12.0,
// 2544 x 4088 x 56 x . W^T 10.2 / 7.7), and of the 128 x 256 ones of a single matrix (1.1x; batches of small ones are even).
bool prefers_short(const GemmProblem& p, Plan plan) {
  if (!srt::short_supported(p)) return false;
  const bool one_slab = p.K <= 64 && (plan == kPlanM16 || plan == kPlanRing256 || plan == kPlanKc64 || (plan == kPlanM16H && p.batch == 1));
  const bool others = one_slab || plan == kPlanCopied || plan == kPlanAny64 || plan == kPlanAny128;
  // (nor instead of 64 x 64 tiles where more than half of a tile is padding: 40 x 976 x 56 x 32 x . W^T 5.9 / 7.4)
  if (!others && (plan != kPlanMfma64 || p.N <= 64)) return false;
  const long long tiles = (long long)((p.M + 127) / 128) * ((p.N + 127) / 128) * p.batch, cus = srt::compute_units();
  if (4 * tiles >= 5 * cus) return plan != kPlanCopied || !copies_ahead(p);
  return others && tiles <= cus && short_time(p) < 0.95 * plan_us(p, plan);
}

// Whether few rows stay on `plan`, which base_plan picked, where the streaming kernel is behind it: weights past 85 MB in rows off 128-byte lines, of
// which a strip's 256 bytes take three instead of two.  Split-K from 150 MB where the strips get one part or two (us, streaming / split-K: 8 x 18072 x
// 8128 72.4 / 64.1, 4 x 14424 x 12544 75.2 / 63.5; 33 random problems 1.11x); the 32-deep half tiles, past the shortest k loops, where the strips take
// twice their rounds over the units (8 x 37432 x 4024 84.5 / 60.6, 32 x 50888 x 944 27.7 / 20.9) or, past 16 rows, more rounds (32 x 91408 x 1032 53.8
// / 43.4; 49 problems 1.2x, 9 x 129936 x 392 not: 31.8 / 43.3); the 64-deep ones at twice the rounds past 16 rows (32 x 124344 x 1984 118 / 94; 36
// problems 1.1x).  In whole lines the streaming kernel is ahead (split-K 1.17x, half tiles 1.3x) or, past 16 rows at twice the rounds, even.
bool few_rows_keep(const GemmProblem& p, Plan plan) {
  const double bytes = 2.0 * p.N * p.K;
  if (bytes < 85.0e6 || p.sbk % 64 == 0) return false;
  const long long cus = srt::compute_units(), strips = (p.N + 127) / 128, halves = (p.N + 255) / 256;
  const long long strip_rounds = (strips + cus - 1) / cus, half_rounds = (halves + cus - 1) / cus;
  const bool twice = strip_rounds >= 2 * half_rounds, two_tiles = p.M > 16;
  if (plan == kPlanSplitK) return bytes >= 150.0e6 && strip_rounds == 1 && 3 * strips > cus;
  if (plan == kPlanM16H) return p.K >= 640 && (twice || (two_tiles && strip_rounds > half_rounds));
  return plan == kPlanM16DH && twice && two_tiles;
}

// Up to 32 rows against an n-contiguous weight: the streaming kernel (gemm_stream.hip) or the wave-split tiles, by what the two take.  Against the kernels
// before there was a streaming one, 500 random problems of 1-32 x 128-140000 x 32-16384 that changed: 1.59x in passes that follow each other over three
// weights, 1.55x from memory, 1.32x in the first pass on a new weight; nine more than 5 % behind in the mean of the three.  Past some size the weight
// comes from memory, and tiles of 64-byte pieces are no match, but out of the caches they stay ahead longer; the lines lie where the mean of the three
// is even (380 random problems): from 35 MB with too few tiles for half the units (us, tiles / streaming: 4 x 3584 x 10752 41 / 17), 65 with a tile a
// unit at most, 40 with three rounds of them and up to 16 rows, else 50 (8 x 14336 x 4096 34 / 22.5; 1 x 6976 x 3712 9.9 / 13.2 out of the caches, 15.0 /
// 14.4 from memory); in rows off whole 128-byte lines, of which the strips read a half more, from 40 and 85 (8 x 15784 x 1792 15.7 / 16.8 from memory,
// 11.4 / 16.2 out of the caches).  What base_plan picks stays for whole 256-column tiles and a k in 1024s, where the tests assert its name; that costs
// most with many such tiles and a short k loop: 8 x 28672 x 1024 15.2 us in half tiles against 13.5.
bool few_rows(const GemmProblem& p, Plan* plan) {
  if (!srt::stream_supported(p) || (p.N % 256 == 0 && p.K % 1024 == 0)) return false;
  const bool lines = p.sbk % 64 == 0;
  const double bytes = 2.0 * p.N * p.K, tiles = (double)((p.N + 31) / 32) / srt::compute_units();
  *plan = bytes < 85.0e6 ? kPlanSkinny : base_plan(p, false);
  if (few_rows_keep(p, *plan)) return true;
  const double kb = 0.128 * p.K * (1.0 + ((p.sbk % 8 != 0) ? 0.3 : 0.0) + ((p.sam % 8 != 0) ? 0.17 : 0.0));
  const double waves = (tiles <= 1.0 ? 3.2 + kb / 97.0 : 3.3 + tiles * (0.26 + kb / 70.0)) + bytes / 32.0e6;
  const double memory = !lines ? (tiles <= 0.5 ? 40.0e6 : 85.0e6) : tiles <= 0.5 ? 35.0e6 : tiles <= 1.0 ? 65.0e6 : tiles > 2.0 && p.M <= 16 ? 40.0e6 : 50.0e6;
  const bool stream = !srt::waves_supported(p) || bytes > memory || (p.K >= 512 && srt::stream_us(p) < 0.95 * waves);
  *plan = stream ? kPlanSkinny : kPlanWaves;
  return true;
}

Plan heuristic_plan(const GemmProblem& p, bool copies = true) {
  Plan plan;
  if (few_rows(p, &plan)) return plan;
  plan = base_plan(p, copies);
  // k ranges off the 64-deep units: two rounds of quarter tiles instead of the 32-deep kernels where the estimates say so (1848 x 4352 x 1512 x^T . W 35.6 us in
  // whole tiles, 30.8; not x . W, which has half tiles: x 552 14.5 / 16.9, x 5480 88 / 94)
  if ((plan == kPlanM16H || plan == kPlanM16 || plan == kPlanRing256 || plan == kPlanKc64) && p.K % 64 != 0 && srt::mfma_config(p, 14) != 0 &&
      srt::mfma_quarter_depth(p) && plan_us(p, kPlanM16Q) < 0.95 * plan_us(p, plan))
    plan = kPlanM16Q;
  // k in parts for up to 32 rows against an n-contiguous weight: the streaming kernel's, under the name of split-K, which the tests assert (32 x 4096 x
  // 4096 16.1 -> 12.7 us, 8 x 4096 x 8192 22.2 -> 16.7).  A pinned or recorded split-K is split-K.
  if (plan == kPlanSplitK && srt::stream_supported(p) && !few_rows_keep(p, plan)) return kPlanStreamed;
  if (p.dtype != srtReal32F && prefers_short(p, plan)) plan = srt::mfma_config(p, 2) != 0 ? kPlanMfma128 : kPlanAny128;
  return p.dtype != srtReal32F && prefers_waves(p, plan) ? kPlanWaves : plan;
}

hipError_t launch_plan(const GemmProblem& p, Plan plan, hipStream_t stream) {
  switch (plan) {
    case kPlanStreamed: return srt::launch_stream(p, stream);
    case kPlanSkinny: return srt::stream_supported(p) ? srt::launch_stream(p, stream) : srt::launch_skinny(p, stream);
    case kPlanRing256: return srt::launch_mfma(p, srt::mfma_config(p, 1), stream);
    case kPlanMfma128: return srt::short_supported(p) ? srt::launch_short(p, stream) : srt::launch_mfma(p, srt::mfma_config(p, 2), stream);
    case kPlanMfma64: return srt::launch_mfma(p, srt::mfma_config(p, 3), stream);
    case kPlanKc64: return srt::launch_mfma(p, srt::mfma_config(p, 4), stream);
    case kPlanM16: return srt::launch_mfma(p, srt::mfma_config(p, 5), stream);
    case kPlanSplitK: return srt::launch_mfma_splitk(p, stream);
    case kPlanM16H: return srt::launch_mfma(p, srt::mfma_config(p, 6), stream);
    case kPlanAny128: return srt::short_supported(p) ? srt::launch_short(p, stream) : srt::launch_mfma(p, srt::mfma_config(p, 7), stream);
    case kPlanAny64: return srt::launch_mfma(p, srt::mfma_config(p, 8), stream);
    case kPlanM16D: return srt::launch_mfma(p, srt::mfma_config(p, 9), stream);
    case kPlanM16DTail: return srt::launch_mfma(p, srt::mfma_config(p, 10), stream);
    case kPlanM16DSplit: return srt::launch_mfma(p, srt::mfma_config(p, 11), stream);
    case kPlanM16DH: return srt::launch_mfma(p, srt::mfma_config(p, 12), stream);
    case kPlanM16DN: return srt::launch_mfma(p, srt::mfma_config(p, 13), stream);
    case kPlanM16Q: return srt::launch_mfma(p, srt::mfma_config(p, 14), stream);
    case kPlanF32Parts: return srt::launch_f32_tile_parts(p, stream);
    case kPlanF32Ring: return srt::launch_f32_ring(p, stream, 0);
    case kPlanF32Ring64x128: return srt::launch_f32_ring(p, stream, 1);
    case kPlanF32Ring64: return srt::launch_f32_ring(p, stream, 2);
    case kPlanF32Tile64: return srt::launch_f32_mfma_variant(p, false, stream);
    case kPlanF32SplitK: return srt::launch_f32_mfma_variant(p, true, stream);
    case kPlanWaves: return srt::launch_waves(p, stream);
    case kPlanCopied: return srt::launch_packed(p, stream);
    default: return srt::launch_generic(p, stream);
  }
}

// Up to 32 rows against an n-contiguous weight where the streaming kernel would cut k and gets no workspace: in one part a quarter to half of the
// units would read.  From 50 MB of weight and a tile a unit the kernel that stages it through LDS, 64 columns a workgroup, else wave-split tiles
// (us, one part / LDS / wave-split, weights from memory: 8 x 9776 x 6216 49.7 / 39.0 / 42.4, 32 x 11008 x 4096 33.3 / 24.4 / 33.4, 8 x 4096 x 8192 51.5
// / 37.0 / 31.4, 8 x 1024 x 2056 15.7 / 12.4 / 10.1; 3643 random problems: within 0.4 % of the best of the three in the mean, one part 82 % behind).
hipError_t launch_whole_range(const GemmProblem& p, hipStream_t stream) {
  if (srt::skinny_supported(p) && p.N > 32 * srt::compute_units() && 2.0 * p.N * p.K > 50.0e6) return srt::launch_skinny(p, stream);
  return srt::waves_supported(p) ? srt::launch_waves(p, stream) : srt::launch_stream(p, stream, true);
}

// A plan that gets no workspace (a full device, a stream under capture; nothing that matters was launched) gives way to the next best, which may
// want one too: copies to what runs the operands as they are, tiles with shared left-overs to whole ones, parts of k to the whole range.
hipError_t launch_or_fall_back(const GemmProblem& p, Plan plan, hipStream_t stream) {
  const hipError_t e = launch_plan(p, plan, stream);
  if (e != hipErrorOutOfMemory) return e;
  Plan next;
  if ((plan == kPlanSkinny || plan == kPlanStreamed || plan == kPlanSplitK) && srt::stream_supported(p)) {
    (void)hipGetLastError();
    return launch_whole_range(p, stream);
  }
  switch (plan) {
    case kPlanSplitK: next = tile_plan(p, false); break;
    case kPlanM16DTail: next = kPlanM16D; break;
    case kPlanF32Parts: next = srt::f32_ring_fits(p) ? kPlanF32Ring : kPlanF32Tile64; break;   // the whole k range per tile
    case kPlanCopied: next = heuristic_plan(p, false); break;   // the operands as they are
    default: return e;
  }
  (void)hipGetLastError();
  return launch_or_fall_back(p, plan_supported(p, next) ? next : kPlanGeneric, stream);
}

struct PlanKey {
  int dtype, M, N, K, batch, layout, epilogue;
  bool operator<(const PlanKey& o) const {
    return std::tie(dtype, M, N, K, batch, layout, epilogue) <
           std::tie(o.dtype, o.M, o.N, o.K, o.batch, o.layout, o.epilogue);
  }
};

// Layout class: which dimension of each operand is contiguous (bits 0-1: A along k / m, bits 2-3:
// B along k / n), whether the batch strides are dense, and whether rows keep 16-byte alignment.
PlanKey key_of(const GemmProblem& p) {
  int layout = 0;
  if (p.sak == 1) layout |= 1;
  if (p.sam == 1) layout |= 2;
  if (p.sbk == 1) layout |= 4;
  if (p.sbn == 1) layout |= 8;
  if (p.scn == 1) layout |= 16;
  if (p.bias_per_row) layout |= 32;
  const long long lda = p.sak == 1 ? p.sam : p.sak, ldb = p.sbk == 1 ? p.sbn : p.sbk;
  if (lda % 8 == 0 && ldb % 8 == 0 && p.scm % 8 == 0) layout |= 64;
  const int epilogue = (p.bias ? 1 : 0) | (p.activation << 1);
  return PlanKey{p.dtype, p.M, p.N, p.K, p.batch, layout, epilogue};
}

class PlanCache {
 public:
  bool find(const PlanKey& k, Plan* plan) {
    std::lock_guard<std::mutex> lock(mu_);
    auto it = plans_.find(k);
    if (it == plans_.end()) return false;
    *plan = it->second;
    return true;
  }
  void put(const PlanKey& k, Plan plan) {
    std::lock_guard<std::mutex> lock(mu_);
    plans_[k] = plan;
  }
  void clear() {
    std::lock_guard<std::mutex> lock(mu_);
    plans_.clear();
  }
  size_t size() {
    std::lock_guard<std::mutex> lock(mu_);
    return plans_.size();
  }
  // One plan per line: dtype M N K batch layout epilogue plan-name
  srtStatus save(const char* path) {
    std::lock_guard<std::mutex> lock(mu_);
    FILE* f = std::fopen(path, "w");
    if (!f) return srtErrorInvalidValue;
    std::fprintf(f, "# SwiftRTHip matmul plans v1: dtype M N K batch layout epilogue plan\n");
    for (const auto& kv : plans_) {
      const PlanKey& k = kv.first;
      std::fprintf(f, "%d %d %d %d %d %d %d %s\n", k.dtype, k.M, k.N, k.K, k.batch, k.layout, k.epilogue,
                   kPlanNames[kv.second]);
    }
    return std::fclose(f) == 0 ? srtSuccess : srtErrorUnknown;
  }
  // All or nothing: a malformed line or an unknown plan name leaves the cache as it was.
  srtStatus load(const char* path) {
    FILE* f = std::fopen(path, "r");
    if (!f) return srtErrorInvalidValue;
    std::map<PlanKey, Plan> read;
    char line[256];
    bool ok = true;
    while (ok && std::fgets(line, sizeof(line), f)) {
      if (line[0] == '#' || line[0] == '\n') continue;
      PlanKey k;
      char name[64];
      if (std::sscanf(line, "%d %d %d %d %d %d %d %63s", &k.dtype, &k.M, &k.N, &k.K, &k.batch, &k.layout,
                      &k.epilogue, name) != 8) { ok = false; break; }
      int plan = -1;
      for (int i = 0; i < kPlanCount; ++i)
        if (std::strcmp(name, kPlanNames[i]) == 0) plan = i;
      if (plan < 0 || k.M < 0 || k.N < 0 || k.K < 0 || k.batch < 0) { ok = false; break; }
      read[k] = (Plan)plan;
    }
    std::fclose(f);
    if (!ok) return srtErrorInvalidValue;
    std::lock_guard<std::mutex> lock(mu_);
    for (const auto& kv : read) plans_[kv.first] = kv.second;
    return srtSuccess;
  }

 private:
  std::mutex mu_;
  std::map<PlanKey, Plan> plans_;
};

PlanCache& plan_cache() {
  static PlanCache* cache = new PlanCache();   // never destroyed: calls may race with process exit
  return *cache;
}

// The plan a call runs: the cached one when it still qualifies (alignment of this call's pointers
// is not part of the key), else the heuristic's.
Plan select(const GemmProblem& p) {
  Plan plan;
  if (plan_cache().size() != 0 && plan_cache().find(key_of(p), &plan) && plan_supported(p, plan)) return plan;
  return heuristic_plan(p);
}

// ---- operands beyond the 256 x 256 kernels' reach -------------------------------------------------
// The 256 x 256 kernels address every operand through one buffer descriptor and 32-bit byte
// offsets, so each operand tensor of a launch (all batches) must span less than 1 Gi elements.
// A device with hundreds of GB holds larger ones (262144 x 8192 activations, 64 batches of
// 8192 x 8192): rather than hand those to the 128 x 128 kernel at half the rate, the call is cut
// into pieces that are within reach -- halves of the batch, then of M, then of N, at multiples of
// the tile size -- and the pieces run back to back on the caller's stream.  A piece is an ordinary
// problem (its own pointers, the same strides) and goes through the same plan selection.  An
// operand whose k walk alone exceeds the reach (K x leading stride >= 1 Gi elements when k is not
// its contiguous dimension) cannot be helped this way and keeps the smaller tiles.
bool fits_256(const GemmProblem& p) { return srt::mfma_config(p, 1) != 0; }

bool split_for_reach(const GemmProblem& p, GemmProblem* lo, GemmProblem* hi) {
  if (p.dtype != srtReal16BF && p.dtype != srtReal16F) return false;
  if (fits_256(p)) return false;
  const long long tiles = (long long)((p.M + 255) / 256) * ((p.N + 255) / 256) * p.batch;
  if (tiles < 128) return false;   // the small tiles are the choice there anyway
  GemmProblem q = p;
  q.batch = 1; q.M = p.M < 256 ? p.M : 256; q.N = p.N < 256 ? p.N : 256;
  if (!fits_256(q)) return false;   // alignment, or a k walk out of reach: not a matter of extent
  auto at = [](const void* base, long long elements) {
    return static_cast<const void*>(static_cast<const char*>(base) + elements * 2);   // 16-bit elements
  };
  *lo = p; *hi = p;
  if (p.batch > 1) {
    const int h = p.batch / 2;
    lo->batch = h; hi->batch = p.batch - h;
    hi->A = at(p.A, h * p.sab); hi->B = at(p.B, h * p.sbb);
    hi->C = const_cast<void*>(at(p.C, h * p.scb));
    return true;
  }
  GemmProblem qm = p; qm.M = q.M;   // would whole columns of tiles fit?
  const bool by_m = p.M > 256 && (fits_256(qm) || p.N <= 256);
  if (by_m) {
    const int m0 = ((p.M / 2 + 255) / 256) * 256;
    lo->M = m0; hi->M = p.M - m0;
    hi->A = at(p.A, m0 * p.sam);
    hi->C = const_cast<void*>(at(p.C, m0 * p.scm));
    if (p.bias && p.bias_per_row) hi->bias = at(p.bias, m0 * p.sbias);
    return true;
  }
  if (p.N <= 256) return false;
  const int n0 = ((p.N / 2 + 255) / 256) * 256;
  lo->N = n0; hi->N = p.N - n0;
  hi->B = at(p.B, n0 * p.sbn);
  hi->C = const_cast<void*>(at(p.C, n0 * p.scn));
  if (p.bias && !p.bias_per_row) hi->bias = at(p.bias, n0 * p.sbias);
  return true;
}

bool has_cached_plan(const GemmProblem& p) {
  Plan plan;
  return plan_cache().size() != 0 && plan_cache().find(key_of(p), &plan) && plan_supported(p, plan);
}

srtStatus run(const GemmProblem& p, hipStream_t stream) {
  GemmProblem lo, hi;
  if (!has_cached_plan(p) && split_for_reach(p, &lo, &hi)) {
    const srtStatus s = run(lo, stream);
    return s != srtSuccess ? s : run(hi, stream);
  }
  const Plan plan = select(p);
  if (plan == kPlanGeneric && !srt::generic_supported(p)) return srtErrorNotSupported;
  return srt::from_hip(launch_or_fall_back(p, plan, stream));
}
}  // namespace

namespace srt {
// The heuristic's plan for a problem built inside the library (operands copied into its workspace).
hipError_t launch_heuristic(const GemmProblem& p, hipStream_t stream) {
  return launch_or_fall_back(p, heuristic_plan(p), stream);
}
}  // namespace srt

extern "C" {

srtStatus srtMatmulBiasActivation(const void* a, const srtTensorDescriptor* aDesc, int32_t transposeA,
                                  const void* b, const srtTensorDescriptor* bDesc, int32_t transposeB,
                                  const void* bias, const srtTensorDescriptor* biasDesc,
                                  srtActivation activation, double coef,
                                  void* out, const srtTensorDescriptor* oDesc, srtStream stream) {
  GemmProblem p;
  bool empty = false;
  srtStatus s = build_problem(a, aDesc, transposeA, b, bDesc, transposeB, bias, biasDesc, (int)activation, coef,
                              out, oDesc, &p, &empty);
  if (s != srtSuccess || empty) return s;
  return run(p, reinterpret_cast<hipStream_t>(stream));
}

srtStatus srtMatmul(const void* a, const srtTensorDescriptor* aDesc, int32_t transposeA,
                    const void* b, const srtTensorDescriptor* bDesc, int32_t transposeB,
                    void* out, const srtTensorDescriptor* oDesc, srtStream stream) {
  return srtMatmulBiasActivation(a, aDesc, transposeA, b, bDesc, transposeB, nullptr, nullptr,
                                 srtActivationIdentity, 0.0, out, oDesc, stream);
}

srtStatus srtMatmulQueryKernel(const srtTensorDescriptor* aDesc, int32_t transposeA,
                               const srtTensorDescriptor* bDesc, int32_t transposeB,
                               const srtTensorDescriptor* oDesc, const void* a, const void* b,
                               const void* out, char* name, size_t nameCapacity) {
  if (!name || nameCapacity == 0) return srtErrorInvalidValue;
  name[0] = 0;
  GemmProblem p;
  bool empty = false;
  srtStatus s = build_problem(a, aDesc, transposeA, b, bDesc, transposeB, nullptr, nullptr,
                              srtActivationIdentity, 0.0, const_cast<void*>(out), oDesc, &p, &empty, false);
  if (s != srtSuccess) return s;
  const char* n = "empty";
  if (!empty) {
    // a call that runs in pieces reports its first piece's kernel, marked "/pieces"
    GemmProblem piece = p, lo, hi;
    bool pieces = false;
    while (!has_cached_plan(piece) && split_for_reach(piece, &lo, &hi)) { piece = lo; pieces = true; }
    const Plan plan = select(piece);
    n = plan_name(plan);
    if (plan == kPlanF32Tile64 || plan == kPlanF32SplitK || plan == kPlanF32Parts || plan == kPlanF32Ring || plan == kPlanF32Ring64x128 || plan == kPlanF32Ring64) n = "f32_mfma";   // one family name for the fp32 tiles
    if (pieces) {
      std::snprintf(name, nameCapacity, "%s/pieces", n);
      return srtSuccess;
    }
  }
  std::snprintf(name, nameCapacity, "%s", n);
  return srtSuccess;
}

srtStatus srtMatmulTune(const void* a, const srtTensorDescriptor* aDesc, int32_t transposeA,
                        const void* b, const srtTensorDescriptor* bDesc, int32_t transposeB,
                        const void* bias, const srtTensorDescriptor* biasDesc,
                        srtActivation activation, double coef,
                        void* out, const srtTensorDescriptor* oDesc, srtStream stream,
                        char* chosen, size_t chosenCapacity) {
  if (chosen && chosenCapacity) chosen[0] = 0;
  GemmProblem p;
  bool empty = false;
  srtStatus s = build_problem(a, aDesc, transposeA, b, bDesc, transposeB, bias, biasDesc, (int)activation, coef,
                              out, oDesc, &p, &empty);
  if (s != srtSuccess || empty) return s;
  hipStream_t hs = reinterpret_cast<hipStream_t>(stream);
  {
    // a problem that runs in pieces has no single plan to record: its pieces keep the heuristic
    GemmProblem lo, hi;
    if (!has_cached_plan(p) && split_for_reach(p, &lo, &hi)) {
      if (chosen && chosenCapacity) std::snprintf(chosen, chosenCapacity, "pieces");
      return run(p, hs);
    }
  }
  hipEvent_t e0, e1;
  if (hipEventCreate(&e0) != hipSuccess) return srtErrorUnknown;
  if (hipEventCreate(&e1) != hipSuccess) { (void)hipEventDestroy(e0); return srtErrorUnknown; }
  const Plan fallback = heuristic_plan(p);
  Plan best = fallback;
  float best_ms = -1.0f;
  hipError_t err = hipSuccess;
  for (int c = 0; c < kPlanCount && err == hipSuccess; ++c) {
    const Plan plan = (Plan)c;
    if (!plan_supported(p, plan)) continue;
    // the FMA kernel is orders of magnitude slower on large problems: skip it when a matrix-core plan exists
    if (plan == kPlanGeneric && fallback != kPlanGeneric && 2.0 * p.M * p.N * p.K * p.batch > 1e9) continue;
    const int warm = 2, reps = 8;
    for (int i = 0; i < warm && err == hipSuccess; ++i) err = launch_plan(p, plan, hs);
    if ((plan == kPlanSkinny || plan == kPlanSplitK || plan == kPlanM16DTail || plan == kPlanF32Parts || plan == kPlanCopied) && err == hipErrorOutOfMemory) {
      // no room for this plan's workspace (nothing was launched): it is not a candidate, as in run()
      (void)hipGetLastError();
      err = hipSuccess;
      continue;
    }
    if (err == hipSuccess) err = hipEventRecord(e0, hs);
    for (int i = 0; i < reps && err == hipSuccess; ++i) err = launch_plan(p, plan, hs);
    if (err == hipSuccess) err = hipEventRecord(e1, hs);
    if (err == hipSuccess) err = hipEventSynchronize(e1);
    float ms = 0.0f;
    if (err == hipSuccess) err = hipEventElapsedTime(&ms, e0, e1);
    if (err == hipSuccess && (best_ms < 0.0f || ms < best_ms)) { best_ms = ms; best = plan; }
  }
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  if (err != hipSuccess) return srt::from_hip(err);
  if (best_ms < 0.0f) return srtErrorNotSupported;   // no kernel qualifies: the caller's CPU path
  plan_cache().put(key_of(p), best);
  // leave `out` written by the chosen plan
  err = launch_or_fall_back(p, best, hs);
  if (chosen && chosenCapacity) std::snprintf(chosen, chosenCapacity, "%s", kPlanNames[best]);
  return srt::from_hip(err);
}

srtStatus srtPlanCacheClear(void) { plan_cache().clear(); return srtSuccess; }

srtStatus srtPlanCacheCount(size_t* count) {
  if (!count) return srtErrorInvalidValue;
  *count = plan_cache().size();
  return srtSuccess;
}

srtStatus srtPlanCacheSave(const char* path) { return path ? plan_cache().save(path) : srtErrorInvalidValue; }

srtStatus srtPlanCacheLoad(const char* path) { return path ? plan_cache().load(path) : srtErrorInvalidValue; }

}  // extern "C"
