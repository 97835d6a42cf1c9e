// Intra-stage configuration search on MI355X (gfx950): row terms and stage summaries, the pruned
// reduction to one table of minima, finalize.  Everything is float64 VALU work with float32
// rounding points where the reference has them; there is no dense contraction here, so no MFMA.
//
// Bit-exactness rules for this file (results must equal the numpy formulation operation for
// operation): compile with -ffp-contract=off, keep the operand order of every sum exactly as
// written, use true divisions, and never reassociate.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <type_traits>

#include "mist_common.h"
#include "mist_search.h"
#include "mist_window_margin.h"
#define MIST_ARITH_FN __device__ __forceinline__
#include "exact_arith.h"

namespace {
thread_local char g_last_error[512] = "";
}  // namespace

namespace mist {
int fail(int code, const char *fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_last_error, sizeof(g_last_error), fmt, ap);
  va_end(ap);
  return code;
}
}  // namespace mist

namespace {

using mist::fail;

constexpr int kTermsBlock = 128;  // rows per workgroup of the row-term kernel
constexpr int kStageRows = 64;    // rows of a stage: one summary, one item of the reduction
constexpr int kSlots = 2 * MIST_P_TILE + 2;  // per-thread running minima: base, with_pre, post, no_pp
constexpr int kScoutSplit = 1;    // (mist_reduce_scout_split: workgroups of a decomposition no launch has any more)
// Relative room above MistProblem.stage_cost_incumbent / G.  The launches behind the seeds look for what lies
// below it: the less room, the fewer rows.  Calls, us, at 0.25 / 0.1 / 0.02 / 0.004: 70B on 32x8 7681 / 6497 / 5775
// / 5430, 13B on 8x8 2286 / 1976 / 1859 / 1770, 7B on 4x8 1477 / 1370 / 1200 / 1140.  A search that cannot tell from
// tables under the limit what the complete ones give evaluates again, at any room about as often: 25 / 23 / 17 / 22
// of 330 calls (less room, fewer (tp, G) with a partition below it; but fewer threshold candidates, too).  Results
// above the estimate, by up to 1.7 % where the scan tries none of its thresholds, want more than the last.
constexpr double kIncumbentSlack = 0.02;
// Stage summaries (written with or ahead of the row terms, read by filter, open and reduce): per stage of
// kStageRows workspace rows the term-wise minimum of the latency and memory columns and the
// maximum of MIST_T_OUT, kStageFloorPitch doubles per stage.
constexpr int kStageFloorPitch = 32;
constexpr int kStageMaxOut = MIST_T_GCB + 1;  // slot of max(MIST_T_OUT) behind the stage minima
// ... and behind it the minima of the post-layer terms that the last-stage / single-stage
// objectives add to every row: MIST_T_OPB, the smaller of MIST_T_NAG_CK / _NOCK, the smaller of
// MIST_T_NRS_CK / _NOCK.
constexpr int kStageMinOpb = kStageMaxOut + 1, kStageMinNag = kStageMaxOut + 2, kStageMinNrs = kStageMaxOut + 3;
static_assert(kStageMinNrs < kStageFloorPitch, "a stage summary is one 32-lane load");
static_assert(MIST_T_NAG_NOCK == MIST_T_NAG_CK + 1 && MIST_T_NRS_NOCK == MIST_T_NRS_CK + 1, "ck / nock pairs");
static_assert(kStageRows == 2 * kStageFloorPitch, "lane = (column, half of the rows)");

// Value of one lane (wave-uniform index) for the whole wavefront.
__device__ __forceinline__ double from_lane(double v, int lane) {
  const unsigned long long u = (unsigned long long)__double_as_longlong(v);
  const uint32_t lo = __builtin_amdgcn_readlane((int)(uint32_t)u, lane);
  const uint32_t hi = __builtin_amdgcn_readlane((int)(uint32_t)(u >> 32), lane);
  return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}
__device__ __forceinline__ int from_lane(int v, int lane) { return __builtin_amdgcn_readlane(v, lane); }
__device__ __forceinline__ float from_lane(float v, int lane) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}
__device__ __forceinline__ uint64_t from_lane(uint64_t v, int lane) {
  const uint32_t lo = __builtin_amdgcn_readlane((int)(uint32_t)v, lane);
  const uint32_t hi = __builtin_amdgcn_readlane((int)(uint32_t)(v >> 32), lane);
  return ((uint64_t)hi << 32) | lo;
}

// ------------------------------------------------------------------------------------------
// Communication models (mist/tools/optimize.py:257-303, 459-470).
// ------------------------------------------------------------------------------------------
__device__ __forceinline__ int size_index(double s) {
  return s == 1.0 ? 0 : (s == 2.0 ? 1 : (s == 4.0 ? 2 : 3));
}

__device__ __forceinline__ double gpu_gpu_latency(const double *gg, double mbytes, double inter,
                                                  double intra, double factor) {
  const double gbytes = mbytes / 1024.0;
  const double ngpu = intra * inter;
  double lat = 0.0;
  if (!(gbytes < 1e-5 || ngpu == 1.0)) {
    const double *cell = gg + (size_index(inter) * 4 + size_index(intra)) * 2;
    lat = gbytes / cell[0] * (ngpu - 1.0) / ngpu + cell[1];
  }
  return lat * factor;
}

__device__ __forceinline__ double host_link_latency(const double *kb, double mbytes) {
  const double gbytes = mbytes / 1024.0;
  const double lat = gbytes / kb[0] + kb[1];
  return gbytes == 0.0 ? 0.0 : lat;
}

// numpy's float64 floor_divide (npy_divmod), for a >= 0 and b > 0 as well as the general case.
__device__ __forceinline__ double np_floor_divide(double a, double b) {
  if (__builtin_expect(mist_arith::floor_divide_is_tame(a, b), 1))
    return mist_arith::floor_divide_tame(a, b);
  if (b == 0.0) return a / b;
  double mod = fmod(a, b);
  double div = (a - mod) / b;
  if (mod != 0.0) {
    if ((b < 0.0) != (mod < 0.0)) div -= 1.0;
  }
  double floordiv;
  if (div != 0.0) {
    floordiv = floor(div);
    if (div - floordiv > 0.5) floordiv += 1.0;
  } else {
    floordiv = copysign(0.0, a / b);
  }
  return floordiv;
}

// ------------------------------------------------------------------------------------------
// Four-resource interference model (mist/tools/optimize.py:1012-1122).  X = [C, G2G, C2G, G2C].
// Masks in evaluation order: 4-way, four 3-way, six 2-way; bit j set = resource j in the mask.
// ------------------------------------------------------------------------------------------
constexpr unsigned char kMaskBits[11] = {
    0xF,
    0x7, 0xB, 0xD, 0xE,
    0x3, 0x5, 0x9, 0x6, 0xA, 0xC,
};

// Index into kMaskBits of the mask equal to a pattern of two or more bits, as 16 nibbles of one
// constant (a table in memory would cost every peel a dependent load).
constexpr uint64_t pack_mask_of_pattern() {
  uint64_t packed = 0;
  for (int m = 0; m < 11; ++m) packed |= (uint64_t)m << (4 * kMaskBits[m]);
  return packed;
}
constexpr uint64_t kMaskOfPatternPacked = pack_mask_of_pattern();
__device__ __forceinline__ int mask_of_pattern(unsigned pattern) {
  return (int)((kMaskOfPatternPacked >> (4 * pattern)) & 0xF);
}
static_assert(((kMaskOfPatternPacked >> (4 * 0xF)) & 0xF) == 0 && ((kMaskOfPatternPacked >> (4 * 0x3)) & 0xF) == 5 &&
                  ((kMaskOfPatternPacked >> (4 * 0xC)) & 0xF) == 10 && ((kMaskOfPatternPacked >> (4 * 0xE)) & 0xF) == 4,
              "pattern -> mask index");

// The factor table lives in LDS and is read through a pointer of that address space: the model
// is out of line, and through a generic pointer every read would be a flat load.
typedef const __attribute__((address_space(3))) double LdsDouble;
constexpr int kFactorPitch = 8;  // per mask: the four factors, then their four reciprocals

// kInline: the model is expanded at every call site (for a kernel with few of them: its loads
// stay in flight across the evaluations, which a call would make it wait for) instead of called.
template <bool kInline>
struct InterferenceModel {
  LdsDouble *table;   // [11][kFactorPitch]: factor[m][0..3], 1 / factor[m][0..3] correctly rounded
  bool factors_tame;  // every factor lies in the divisor range of the reciprocal quotient

  // Operands (seconds) below this bound keep every scaled time and every quotient of a peel
  // inside the range where the reciprocal quotient is the IEEE quotient; a peel only divides
  // differences of scaled times of resources busier than 1e-8 s, which are zero or no smaller
  // than an ulp of 1e-8.
  static constexpr double kOperandBound = 0x1p500;

  // Arguments in the order of the reference's get_layer_critical_latency
  // (batched_module_analyzer.py:1413-1422): exec, gpu<->gpu, gpu->cpu, cpu->gpu.
  // kLive: bit i set when X[i] (exec, gpu<->gpu, cpu->gpu, gpu->cpu) can be non-zero at this call
  // site; the others are literal zeros there, never part of a mask, and their share of a round
  // (a multiplication and a division each) is left out at compile time.  The sums keep all four
  // operands, so the value is the one of the general form.
  // kByReciprocal: the quotients (s - overlap) / factor are taken with the stored reciprocals
  // (five multiply-adds, no branch, so that the four quotients of a peel interleave) instead of
  // the division sequence; eval() picks it when every operand of the wave is in range.
  template <unsigned kLive, bool kByReciprocal>
  __device__ __noinline__ double eval_called(double exec, double g2g, double g2c, double c2g) const {
    return eval_body<kLive, kByReciprocal>(exec, g2g, g2c, c2g);
  }
  template <unsigned kLive, bool kByReciprocal>
  __device__ __forceinline__ double eval_as(double exec, double g2g, double g2c, double c2g) const {
    if constexpr (kInline || __builtin_popcount(kLive) < 2)
      return eval_body<kLive, kByReciprocal>(exec, g2g, g2c, c2g);
    else
      return eval_called<kLive, kByReciprocal>(exec, g2g, g2c, c2g);
  }
  template <unsigned kLive, bool kByReciprocal>
  __device__ __forceinline__ double eval_body(double exec, double g2g, double g2c, double c2g) const {
    double x0 = (kLive & 1u) ? exec : 0.0, x1 = (kLive & 2u) ? g2g : 0.0;
    double x2 = (kLive & 4u) ? c2g : 0.0, x3 = (kLive & 8u) ? g2c : 0.0;
    double out = 0.0;
    // The reference tries the 11 masks in order and applies the one equal to the non-zero
    // pattern of X.  A pattern equals at most one mask, and after a peel the pattern has fewer
    // bits, i.e. it can only equal a mask further down the list (4-way, then 3-way, then
    // 2-way).  So the rounds are taken by the size of the pattern: a lane joins at the size of
    // its own pattern, and the wave runs each size once.
    // "not isclose(x, 0)" with numpy's default tolerances: |x| > 1e-8.
    auto pattern = [&]() {
      return (((kLive & 1u) && !(fabs(x0) <= 1e-8)) ? 1u : 0u) |
             (((kLive & 2u) && !(fabs(x1) <= 1e-8)) ? 2u : 0u) |
             (((kLive & 4u) && !(fabs(x2) <= 1e-8)) ? 4u : 0u) |
             (((kLive & 8u) && !(fabs(x3) <= 1e-8)) ? 8u : 0u);
    };
    // a / f for a = s - overlap >= +0 (never -0: a difference of equal numbers is +0).
    auto quotient = [&](double a, double f, double y) {
      if (!kByReciprocal) return a / f;
      return mist_arith::quotient_by_reciprocal<false>(a, f, y, a * y);
    };
    // One peel as the reference writes it: every busy resource gives up the smallest scaled
    // time.  (s - ov) / f * 1.0 there: the product with 1.0 changes nothing.
    auto peel = [&](unsigned mask) {
      LdsDouble *row = table + mask_of_pattern(mask) * kFactorPitch;
      const double f0 = row[0], f1 = row[1], f2 = row[2], f3 = row[3];
      const double y0 = row[4], y1 = row[5], y2 = row[6], y3 = row[7];
      const double s0 = x0 * f0, s1 = x1 * f1, s2 = x2 * f2, s3 = x3 * f3;
      double ov = INFINITY;
      if ((kLive & 1u) && (mask & 1u)) ov = fmin(ov, s0);
      if ((kLive & 2u) && (mask & 2u)) ov = fmin(ov, s1);
      if ((kLive & 4u) && (mask & 4u)) ov = fmin(ov, s2);
      if ((kLive & 8u) && (mask & 8u)) ov = fmin(ov, s3);
      if ((kLive & 1u) && (mask & 1u)) x0 = quotient(s0 - ov, f0, y0);
      if ((kLive & 2u) && (mask & 2u)) x1 = quotient(s1 - ov, f1, y1);
      if ((kLive & 4u) && (mask & 4u)) x2 = quotient(s2 - ov, f2, y2);
      if ((kLive & 8u) && (mask & 8u)) x3 = quotient(s3 - ov, f3, y3);
      out = out + ov;
    };
    // The same peel for two busy resources with one division: the one with the smaller scaled
    // time is left with (s - s) / f = +0 (factors are positive and finite), the other with
    // (larger - smaller) / its factor; with equal times both quotients are +0.
    auto peel_pair = [&](unsigned mask) {
      LdsDouble *row = table + mask_of_pattern(mask) * kFactorPitch;
      const double f0 = row[0], f1 = row[1], f2 = row[2], f3 = row[3];
      const double s0 = x0 * f0, s1 = x1 * f1, s2 = x2 * f2, s3 = x3 * f3;
      const bool b0 = (kLive & 1u) && (mask & 1u), b1 = (kLive & 2u) && (mask & 2u);
      const bool b2 = (kLive & 4u) && (mask & 4u), b3 = (kLive & 8u) && (mask & 8u);
      double lo = INFINITY, hi = -INFINITY;
      if (b0) { lo = fmin(lo, s0); hi = fmax(hi, s0); }
      if (b1) { lo = fmin(lo, s1); hi = fmax(hi, s1); }
      if (b2) { lo = fmin(lo, s2); hi = fmax(hi, s2); }
      if (b3) { lo = fmin(lo, s3); hi = fmax(hi, s3); }
      double den = 1.0, rden = 1.0;
      if (b0 && s0 == hi) { den = f0; rden = row[4]; }
      if (b1 && s1 == hi) { den = f1; rden = row[5]; }
      if (b2 && s2 == hi) { den = f2; rden = row[6]; }
      if (b3 && s3 == hi) { den = f3; rden = row[7]; }
      const double rest = quotient(hi - lo, den, rden);
      if (b0) x0 = s0 == hi ? rest : 0.0;
      if (b1) x1 = s1 == hi ? rest : 0.0;
      if (b2) x2 = s2 == hi ? rest : 0.0;
      if (b3) x3 = s3 == hi ? rest : 0.0;
      out = out + lo;
    };
    constexpr int kLiveCount = __builtin_popcount(kLive);
    if constexpr (kLiveCount == 4) {
      const unsigned nz = pattern();
      if (nz == 15u) peel(nz);
    }
    if constexpr (kLiveCount >= 3) {
      const unsigned nz = pattern();
      if (__popc(nz) == 3) peel(nz);
    }
    if constexpr (kLiveCount >= 2) {
      const unsigned nz = pattern();
      if (__popc(nz) == 2) peel_pair(nz);
    }
    return out + (((x0 + x1) + x2) + x3);
  }

  template <unsigned kLive>
  __device__ __forceinline__ double eval(double exec, double g2g, double g2c, double c2g) const {
    if constexpr (__builtin_popcount(kLive) < 2) {
      return eval_as<kLive, false>(exec, g2g, g2c, c2g);  // nothing to divide
    } else {
      // NaN and infinities fail the comparisons and take the division sequence, wave-wide.
      const bool tame = factors_tame &&
                        (!(kLive & 1u) || fabs(exec) < kOperandBound) &&
                        (!(kLive & 2u) || fabs(g2g) < kOperandBound) &&
                        (!(kLive & 4u) || fabs(c2g) < kOperandBound) &&
                        (!(kLive & 8u) || fabs(g2c) < kOperandBound);
      if (__builtin_expect(__all(tame), 1)) return eval_as<kLive, true>(exec, g2g, g2c, c2g);
      return eval_called<kLive, false>(exec, g2g, g2c, c2g);  // never expanded in place: cold
    }
  }

  __device__ __forceinline__ double operator()(double exec, double g2g, double g2c, double c2g) const {
    return eval<15u>(exec, g2g, g2c, c2g);
  }
  // Call sites whose literal zeros are known: operands named by what is live.
  __device__ __forceinline__ double exec_g2g_c2g(double exec, double g2g, double c2g) const {
    return eval<1u | 2u | 4u>(exec, g2g, 0.0, c2g);
  }
  __device__ __forceinline__ double exec_g2g_g2c(double exec, double g2g, double g2c) const {
    return eval<1u | 2u | 8u>(exec, g2g, g2c, 0.0);
  }
  __device__ __forceinline__ double g2g_c2g(double g2g, double c2g) const {
    return eval<2u | 4u>(0.0, g2g, 0.0, c2g);
  }
  __device__ __forceinline__ double g2g_g2c(double g2g, double g2c) const {
    return eval<2u | 8u>(0.0, g2g, g2c, 0.0);
  }
  __device__ __forceinline__ double exec_g2c(double exec, double g2c) const {
    return eval<1u | 8u>(exec, 0.0, g2c, 0.0);
  }
  __device__ __forceinline__ double g2c_only(double g2c) const {
    return eval<8u>(0.0, 0.0, g2c, 0.0);
  }
};

struct Family {
  double layer, first, last, extra_pre, extra_post;
};

__device__ __forceinline__ Family pick_family(bool second, const Family &a, const Family &b) {
  Family r;
  r.layer = second ? b.layer : a.layer;
  r.first = second ? b.first : a.first;
  r.last = second ? b.last : a.last;
  r.extra_pre = second ? b.extra_pre : a.extra_pre;
  r.extra_post = second ? b.extra_post : a.extra_post;
  return r;
}

// Slot of stage `stage` of group `group_index` in the stage-summary workspace.  Groups lie back
// to back in the row workspace and need not start at a multiple of kStageRows; adding the group
// index keeps the slots of consecutive groups apart (at most rows / kStageRows + groups + 1 slots).
__device__ __forceinline__ int64_t stage_floor_slot(const MistGroupDesc *g, int group_index,
                                                    int64_t stage) {
  return g->row_offset / kStageRows + group_index + stage;
}

__device__ __forceinline__ const MistGroupDesc *find_group(const MistGroupDesc *groups,
                                                           const int32_t *prefix, int n_groups,
                                                           int block, int *local) {
  int lo = 0, hi = n_groups;  // prefix[lo] <= block < prefix[hi]
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (prefix[mid] <= block) lo = mid; else hi = mid;
  }
  *local = block - prefix[lo];
  return groups + lo;
}

// Workspace order.  The reference numbers a group's rows parallelism-major with the activation
// offload ratio fastest (batched_module_analyzer.py:490-534); the workspace holds them per
// (parallelism row, activation ratio) in tiles of kOoTile optimizer ratios, and inside a tile
// pair by pair:
//   position = (par * n_ao + ao) * n_oo * n_pair + tile * kOoTile * n_pair + pair * width + oo % kOoTile
// with tile = oo / kOoTile and width = ratios in that tile (kOoTile, fewer in the last one).  A
// stage (64 consecutive positions) then covers 16 neighbouring (weight,
// gradient) pairs at 4 neighbouring optimizer ratios: rows of similar latency AND footprint, so
// the stage's term-wise minimum is close to a real row and its bounds prune.  (With all pairs of
// one optimizer ratio in a run, a stage spanned half of the pair list: its minimum was as fast as
// the rows without offloading and as small as those with all of it.)  Results carry row numbers.
constexpr int kOoTile = 4;

struct RowParts {
  int par, pair, oo, ao;
};

// Position inside the (par, ao) block of n_oo * n_pair rows.
__device__ __forceinline__ int tile_position(const MistGroupDesc *g, int oo, int pair) {
  const int tile = oo / kOoTile;
  const int width = min(kOoTile, g->n_oo - tile * kOoTile);
  return tile * kOoTile * g->n_pair + pair * width + (oo - tile * kOoTile);
}

// (positions fit 32 bits: the tables hold row numbers as int32)
__device__ __forceinline__ RowParts parts_of_position(const MistGroupDesc *g, uint32_t pos) {
  RowParts r;
  r.par = (int)(pos / (uint32_t)g->n_off);
  int rem = (int)(pos - (uint32_t)r.par * (uint32_t)g->n_off);
  const int per_ao = g->n_oo * g->n_pair;
  r.ao = rem / per_ao;
  rem -= r.ao * per_ao;
  const int tile = rem / (kOoTile * g->n_pair);
  rem -= tile * kOoTile * g->n_pair;
  const int width = min(kOoTile, g->n_oo - tile * kOoTile);
  r.pair = rem / width;
  r.oo = tile * kOoTile + (rem - r.pair * width);
  return r;
}

__device__ __forceinline__ int32_t row_of_position(const MistGroupDesc *g, int64_t pos) {
  const RowParts r = parts_of_position(g, (uint32_t)pos);
  return (int32_t)((int64_t)r.par * g->n_off + (r.pair * g->n_oo + r.oo) * g->n_ao + r.ao);
}

__device__ __forceinline__ int64_t position_of_row(const MistGroupDesc *g, int64_t row) {
  const int par = (int)(row / g->n_off);
  const int off = (int)(row % g->n_off);
  const int n_tail = g->n_oo * g->n_ao;
  const int pair = off / n_tail;
  const int oo = (off / g->n_ao) % g->n_oo;
  const int ao = off % g->n_ao;
  return (int64_t)par * g->n_off + (int64_t)ao * g->n_oo * g->n_pair + tile_position(g, oo, pair);
}

// ------------------------------------------------------------------------------------------
// Kernel 1: row-invariant terms.  One thread per candidate row (workspace position).
// ------------------------------------------------------------------------------------------
// Of a row's 36 evaluations of the interference model only the eight of the forward phase of the
// first micro-batch see the optimizer ratio (through the optimizer-state swaps); the other 28
// are the same for the n_oo rows of one "key" = (parallelism, activation ratio, offload pair).
// key_terms_kernel evaluates those once per key into MIST_KEY_TERMS doubles, row_terms_kernel
// reads them: the same operations on the same operands as when every row evaluates everything
// (which it does when the caller passes no key-term workspace, and for the gathered rows of the seed
// launch, which are computed ahead of all others).
constexpr int kKeyBwd = 0;        // [last?0:1 micro-batch][nock, ck] x (layer, first, last, extra_pre, extra_post)
constexpr int kKeyFwd = 20;       // forward, not the first micro-batch: [nock, ck] x (layer, last, extra_post)
constexpr int kKeyFwdFirst = 26;  //   its `first` and `extra_pre`, which do not depend on ckpt
constexpr int kKeyFwdExtraPre = 27;
constexpr int kKeyRow = 28;       // terms up to here are what row_terms reads of a key
// ... and for the stage summaries the columns that are the same for the n_oo rows of the key,
constexpr int kKeyCols = 28;      // S_LAYER_CK .. S_LAST_NOCK (of G > 1), then
constexpr int kKeyState0 = 34;    // FWD_STATES0, BWD_STATES0, PWG, S_CK, S_NOCK, D_CK, D_NOCK,
constexpr int kKeyPeaks = 41;     // FWD_PEAK, BWD_PEAK, OUT, GCB,
constexpr int kKeyPost = 45;      // OPB, the smaller NAG, the smaller NRS;
constexpr int kKeyColsEnd = 48;
// what the rows' first forward phase and memory factor take from the key
constexpr int kKeySoW = 48, kKeySiG = 49, kKeySoA = 50;  // so_W, si_G, so_A_ck, so_A_nock
constexpr int kKeyFactor = 52;    // memory factor without / with optimizer offloading
constexpr int kKeyGather = 54;    // AG_w * ore
static_assert(MIST_KEY_TERMS == 56 && MIST_KEY_TERMS % 2 == 0, "key terms are read as 16-byte pairs");
constexpr int kKeyPitch = MIST_KEY_TERMS + 1;  // of a key in LDS

// Model tables of a workgroup in LDS (tables indexed at run time: indexing the by-value kernel
// argument would make every lane keep a private copy of the whole struct in scratch memory).
// Returns whether every interference factor is in the divisor range of the reciprocal quotient.
__device__ __forceinline__ bool load_model_tables(const MistProblem &prob,
                                                  double (*lds_factor)[kFactorPitch],
                                                  double *lds_gpu_gpu) {
  bool factors_tame = true;
  if (threadIdx.x < 44) {
    const double f = prob.interf_factor[threadIdx.x / 4][threadIdx.x % 4];
    lds_factor[threadIdx.x / 4][threadIdx.x % 4] = f;
    lds_factor[threadIdx.x / 4][4 + threadIdx.x % 4] = 1.0 / f;
    factors_tame = f >= mist_arith::kDivisorMin && f <= mist_arith::kDivisorMax;
  }
  if (threadIdx.x >= 64 && threadIdx.x < 96) lds_gpu_gpu[threadIdx.x - 64] = prob.gpu_gpu[threadIdx.x - 64];
  return __syncthreads_and(factors_tame) != 0;
}

// batched_module_analyzer.py:1181-1199
__device__ __forceinline__ double memory_factor(const MistProblem &prob, const double *par, double wo, double go,
                                                double oo, double ao) {
  double mf = 1.0;
  mf += prob.frag_factor;
  mf += wo > 0.0 ? 0.025 : 0.0;
  mf += go > 0.0 ? 0.025 : 0.0;
  mf += oo > 0.0 ? 0.03 : 0.0;
  mf += ao > 0.0 ? 0.04 : 0.0;
  mf += par[MIST_PAR_WRE] != 0.0 ? 0.025 : 0.0;
  mf += par[MIST_PAR_GRE] != 0.0 ? 0.025 : 0.0;
  mf += par[MIST_PAR_TP] > 1.0 ? 0.04 : 0.0;
  mf += par[MIST_PAR_B] >= 4.0 ? 0.01 : 0.0;
  return mf;
}

// Memory pieces of a row that do not depend on the optimizer ratio (:1216-1272, 2091-2162).
struct KeyMemory {
  double pWG, S_ck, S_nock, D_ck, D_nock, two_buf, fwd_states0;
};
__device__ __forceinline__ KeyMemory key_memory(const MistGroupDesc *g, const double *par, double wo, double go,
                                                double ao) {
  const double dp = par[MIST_PAR_DP];
  const double W = par[MIST_PAR_W], Gr = par[MIST_PAR_G], O = par[MIST_PAR_O];
  const double raw_ck = par[MIST_PAR_RAW_CK], raw_nock = par[MIST_PAR_RAW_NOCK];
  const double wre_size = par[MIST_PAR_WRE] == 1.0 ? dp : 1.0;
  const double gre_size = par[MIST_PAR_GRE] == 1.0 ? dp : 1.0;
  const double ore_size = par[MIST_PAR_ORE] == 1.0 ? dp : 1.0;
  KeyMemory m;
  const double pW = W / wre_size * (1.0 - wo);
  const double pG = Gr / gre_size * (1.0 - go);
  m.pWG = pW + pG;
  m.S_ck = raw_ck * (1.0 - ao);
  m.D_ck = raw_ck * ao;
  m.S_nock = raw_nock * (1.0 - ao);
  m.D_nock = raw_nock * ao;
  const bool wbuf_on = wre_size > 1.0 || g->pp_wre == 1 || wo > 0.0;
  const bool gbuf_on = gre_size > 1.0 || g->pp_gre == 1 || go > 0.0;
  const double Wbuf = wbuf_on ? fmax(fmax(g->pre_full_w, g->post_full_w), W) : 0.0;
  const double Gbuf = gbuf_on ? fmax(fmax(g->pre_full_g, g->post_full_g), Gr) : 0.0;
  m.two_buf = 2.0 * (Wbuf + Gbuf);
  m.fwd_states0 = m.two_buf + np_floor_divide(O, ore_size);
  return m;
}

// Operands of the interference evaluations that do not depend on the optimizer ratio: swap and
// collective latencies (:1362-1408) of one (parallelism row, offload pair, activation ratio).
struct KeyInputs {
  double exec_fwd, exec_bwd_nock, exec_bwd_ck, extra_fwd, extra_bwd, extra_fb;
  double wre, gre, ore;
  double so_W, si_W, so_G, si_G, so_A_ck, si_A_ck, so_A_nock, si_A_nock;
  double AG_w, RS_g, AR_g;
  double E_f, ag_wre, g2c_B, c2g_B, first_g2c, g2g_B[2];
};

__device__ __forceinline__ KeyInputs key_inputs(const MistProblem &prob, const double *lds_gpu_gpu,
                                                const MistGroupDesc *g, const double *par,
                                                double wo, double go, double ao) {
  KeyInputs in;
  const double dp = par[MIST_PAR_DP];
  in.wre = par[MIST_PAR_WRE];
  in.gre = par[MIST_PAR_GRE];
  in.ore = par[MIST_PAR_ORE];
  const double W = par[MIST_PAR_W], Gr = par[MIST_PAR_G];
  const double raw_ck = par[MIST_PAR_RAW_CK], raw_nock = par[MIST_PAR_RAW_NOCK];
  in.exec_fwd = par[MIST_PAR_EXEC_FWD];
  in.exec_bwd_nock = par[MIST_PAR_EXEC_BWD];
  in.extra_fwd = par[MIST_PAR_EXTRA_FWD];
  in.extra_bwd = par[MIST_PAR_EXTRA_BWD];
  const double wre_size = in.wre == 1.0 ? dp : 1.0;
  const double gre_size = in.gre == 1.0 ? dp : 1.0;
  in.so_W = host_link_latency(prob.gpu_cpu, W / wre_size * wo);
  in.si_W = host_link_latency(prob.cpu_gpu, W / wre_size * wo);
  in.so_G = host_link_latency(prob.gpu_cpu, Gr / gre_size * go);
  in.si_G = host_link_latency(prob.cpu_gpu, Gr / gre_size * go);
  in.so_A_ck = host_link_latency(prob.gpu_cpu, raw_ck * ao);
  in.si_A_ck = host_link_latency(prob.cpu_gpu, raw_ck * ao);
  in.so_A_nock = host_link_latency(prob.gpu_cpu, raw_nock * ao);
  in.si_A_nock = host_link_latency(prob.cpu_gpu, raw_nock * ao);
  const double n_nodes = (double)g->num_nodes;
  const double dp_inter = dp > n_nodes ? n_nodes : dp;
  const double dp_intra = dp > n_nodes ? floor(dp / n_nodes) : 1.0;
  in.AG_w = gpu_gpu_latency(lds_gpu_gpu, W, dp_inter, dp_intra, 1.0);
  in.RS_g = gpu_gpu_latency(lds_gpu_gpu, Gr, dp_inter, dp_intra, 1.1);
  in.AR_g = gpu_gpu_latency(lds_gpu_gpu, Gr, dp_inter, dp_intra, 2.1);
  const bool adv = prob.adv_first_block != 0;
  in.E_f = in.exec_fwd - in.extra_fwd;
  in.ag_wre = in.AG_w * in.wre;
  in.g2c_B = in.so_G;
  in.c2g_B = in.si_W + in.si_G;
  in.first_g2c = adv ? in.g2c_B : 0.0;
  in.g2g_B[0] = in.ag_wre + in.RS_g * in.ore + in.AR_g * (1.0 - in.ore);
  in.g2g_B[1] = in.ag_wre + in.RS_g * in.gre;
  in.extra_fb = in.extra_fwd + in.extra_bwd;
  in.exec_bwd_ck = in.exec_fwd + in.exec_bwd_nock;
  return in;
}

// Post-layer collectives left over beside the last layer (:2251-2292).
struct PostTerms {
  double nag_ck, nag_nock, nrs_ck, nrs_nock;
};
__device__ __forceinline__ PostTerms post_terms(const MistGroupDesc *g, const KeyInputs &in) {
  PostTerms p;
  const double ovw_ck = fmax(in.exec_fwd - 0.0 - in.so_A_ck, 0.0);
  const double ovw_nock = fmax(in.exec_fwd - 0.0 - in.so_A_nock, 0.0);
  p.nag_ck = fmax(g->post_ag - ovw_ck, 0.0);
  p.nag_nock = fmax(g->post_ag - ovw_nock, 0.0);
  const double ovg_ck = fmax(in.exec_bwd_ck - in.ag_wre - in.c2g_B - in.si_A_ck, 0.0);
  const double ovg_nock = fmax(in.exec_bwd_nock - in.ag_wre - in.c2g_B - in.si_A_nock, 0.0);
  p.nrs_ck = fmax(g->post_rs - ovg_ck, 0.0);
  p.nrs_nock = fmax(g->post_rs - ovg_nock, 0.0);
  return p;
}

// Forward phases (:1432-1621): phase 0 = first micro-batch (the optimizer-state swaps so_O /
// si_O run beside it), phase 1 = the others.
struct FwdOperands {
  double g2c, c2g, g2g;
};
__device__ __forceinline__ FwdOperands fwd_operands(const KeyInputs &in, bool first_micro_batch,
                                                    double so_O, double si_O) {
  if (first_micro_batch) return FwdOperands{so_O + in.so_W, si_O + in.si_G, in.AG_w * in.ore};
  return FwdOperands{0.0, in.si_W, in.AG_w * in.wre};
}
// the members of a forward family that do not depend on ckpt ...
template <class Interference>
__device__ __forceinline__ void fwd_common(const Interference &I, const KeyInputs &in,
                                           const FwdOperands &op, bool first_micro_batch, bool adv,
                                           double &first, double &extra_pre) {
  const double pre_g2g = (first_micro_batch || adv) ? op.g2g : 0.0;
  const double pre_c2g = adv ? op.c2g : 0.0;
  first = I.exec_g2g_c2g(in.E_f, op.g2g, op.c2g) + in.extra_fwd;
  extra_pre = I.g2g_c2g(pre_g2g, pre_c2g);
}
// ... and those that do (with_ckpt: the saved activations of a checkpointed layer are swapped)
template <class Interference>
__device__ __forceinline__ void fwd_of_ckpt(const Interference &I, const KeyInputs &in,
                                            const FwdOperands &op, bool with_ckpt, double &layer,
                                            double &last, double &extra_post) {
  const double g2c = op.g2c + (with_ckpt ? in.so_A_ck : in.so_A_nock);
  layer = I(in.E_f, op.g2g, g2c, op.c2g) + in.extra_fwd;
  last = I.exec_g2c(in.E_f, g2c) + in.extra_fwd;
  extra_post = I.g2c_only(g2c);
}

// Backward phases (:1646-1902): not_last = false for the last micro-batch.
template <class Interference>
__device__ __forceinline__ Family bwd_family(const Interference &I, const KeyInputs &in,
                                             bool not_last, bool with_ckpt) {
  const bool k = with_ckpt;
  const double E = k ? in.exec_bwd_ck - in.extra_fb : in.exec_bwd_nock - in.extra_bwd;
  const double extra = k ? in.extra_fb : in.extra_bwd;
  const double c2g = in.c2g_B + (k ? in.si_A_ck : in.si_A_nock);
  const double red_last =
      k ? (in.ore == 1.0 ? in.RS_g : in.AR_g) : in.RS_g * in.ore + in.AR_g * (1.0 - in.ore);
  const double red = not_last ? in.RS_g * in.gre : red_last;
  // With checkpointing the reference adds the (always zero) all-gather of saved tensors.
  const double g2g_phase = not_last ? in.g2g_B[1] : in.g2g_B[0];
  const double g2g_layer = k ? g2g_phase + 0.0 : g2g_phase;
  Family f;
  f.layer = I(E, g2g_layer, in.g2c_B, c2g) + extra;
  f.last = I.exec_g2g_c2g(E, in.ag_wre, c2g) + extra;
  f.first = I.exec_g2g_g2c(E, red, in.first_g2c) + extra;
  f.extra_pre = I.g2g_c2g(in.ag_wre, c2g);
  f.extra_post = I.g2g_g2c(red, in.first_g2c);
  return f;
}

// Workgroup = (32 keys of one group) x (4 lanes per key); grid.y = group, grid.x covers the
// group with the most keys.  Lane j of a key evaluates backward family j (= 2 * not_last + ckpt)
// and the forward family of the later micro-batches with ckpt = j & 1.
__global__ __launch_bounds__(kTermsBlock) void key_terms_kernel(
    const MistProblem prob, const MistGroupDesc *__restrict__ groups, double *__restrict__ key_terms) {
  const MistGroupDesc *g = groups + blockIdx.y;
  const int n_keys = g->n_par * g->n_ao * g->n_pair;
  constexpr int kKeysPerBlock = kTermsBlock / 4;
  if ((int)blockIdx.x * kKeysPerBlock >= n_keys) return;
  __shared__ __align__(16) double lds_factor[11][kFactorPitch];
  __shared__ double lds_gpu_gpu[32];
  __shared__ double lds_out[kKeysPerBlock][kKeyPitch];
  InterferenceModel<false> I;
  I.factors_tame = load_model_tables(prob, lds_factor, lds_gpu_gpu);
  I.table = (LdsDouble *)&lds_factor[0][0];
  const int key_here = (int)blockIdx.x * kKeysPerBlock + (int)threadIdx.x / 4;
  const int key = min(key_here, n_keys - 1);  // lanes past the end redo the last key, unwritten
  const int j = threadIdx.x & 3;
  const int pair = key % g->n_pair;
  const int ao_i = (key / g->n_pair) % g->n_ao;
  const int par_i = key / (g->n_pair * g->n_ao);
  const double *par = g->par[par_i];
  const double wo = g->wo[g->pair_wo[pair]], go = g->go[g->pair_go[pair]], ao = g->ao[ao_i];
  const KeyInputs in = key_inputs(prob, lds_gpu_gpu, g, par, wo, go, ao);
  const Family back = bwd_family(I, in, (j & 2) != 0, (j & 1) != 0);
  const FwdOperands op = fwd_operands(in, false, 0.0, 0.0);
  double first, extra_pre, layer, last, extra_post;
  fwd_common(I, in, op, false, prob.adv_first_block != 0, first, extra_pre);
  fwd_of_ckpt(I, in, op, (j & 1) != 0, layer, last, extra_post);
  double *out = lds_out[threadIdx.x / 4];
  double *b = out + kKeyBwd + j * 5;
  b[0] = back.layer;
  b[1] = back.first;
  b[2] = back.last;
  b[3] = back.extra_pre;
  b[4] = back.extra_post;
  if (j < 2) {
    double *f = out + kKeyFwd + j * 3;
    f[0] = layer;
    f[1] = last;
    f[2] = extra_post;
  } else {
    // (with ckpt in front of without)
    double *c = out + kKeyCols + (1 - (j & 1));
    c[0] = layer + back.layer;
    c[2] = extra_pre + back.extra_post + first + back.first;
    c[4] = extra_post + back.extra_pre + last + back.last;
    if (j == 3) out[kKeyPost] = fmax(g->post_bwd - back.extra_pre, 0.0);
  }
  if (j == 0) {
    out[kKeyFwdFirst] = first;
    out[kKeyFwdExtraPre] = extra_pre;
    const PostTerms post = post_terms(g, in);
    out[kKeyPost + 1] = fmin(post.nag_ck, post.nag_nock);
    out[kKeyPost + 2] = fmin(post.nrs_ck, post.nrs_nock);
    out[kKeyFactor] = memory_factor(prob, par, wo, go, 0.0, ao);
    out[kKeyFactor + 1] = memory_factor(prob, par, wo, go, 1.0, ao);
  } else if (j == 1) {
    const KeyMemory m = key_memory(g, par, wo, go, ao);
    double *c = out + kKeyState0;
    c[0] = m.fwd_states0;
    c[1] = m.two_buf;
    c[2] = m.pWG;
    c[3] = m.S_ck;
    c[4] = m.S_nock;
    c[5] = m.D_ck;
    c[6] = m.D_nock;
  } else if (j == 2) {
    double *c = out + kKeyPeaks;
    c[0] = par[MIST_PAR_FWD_PEAK];
    c[1] = par[MIST_PAR_BWD_PEAK];
    c[2] = par[MIST_PAR_OUT];
    c[3] = par[MIST_PAR_GCB];
  } else {
    out[kKeySoW] = in.so_W;
    out[kKeySiG] = in.si_G;
    out[kKeySoA] = in.so_A_ck;
    out[kKeySoA + 1] = in.so_A_nock;
    out[kKeyGather] = in.AG_w * in.ore;
    out[kKeyGather + 1] = 0.0;
  }
  __syncthreads();
  double *__restrict__ dst =
      key_terms + (g->key_offset + (int64_t)blockIdx.x * kKeysPerBlock) * MIST_KEY_TERMS;
  const int n_out = min(kKeysPerBlock, n_keys - (int)blockIdx.x * kKeysPerBlock) * MIST_KEY_TERMS;
  for (int i = threadIdx.x; i < n_out; i += kTermsBlock)
    dst[i] = lds_out[i / MIST_KEY_TERMS][i % MIST_KEY_TERMS];
}

__device__ __forceinline__ int64_t gathered_position(const MistGroupDesc *g, uint32_t q);

// Terms of the row at workspace position `row` of a group.  kFromKeys: what is the same for the
// n_oo rows of its key is read from `key_terms` (written by key_terms_kernel) instead of evaluated.
template <bool kFromKeys>
__device__ __forceinline__ void row_terms_of(const MistProblem &prob, const MistGroupDesc *__restrict__ g, uint32_t row,
                                             const double *__restrict__ key_terms, const double *lds_gpu_gpu,
                                             const InterferenceModel<kFromKeys> &I, double (&t)[MIST_ROW_TERMS]) {
  // ---- index decomposition (batched_module_analyzer.py:490-534) ----
  const RowParts parts = parts_of_position(g, row);
  const int par_i = parts.par, pair = parts.pair, oo_i = parts.oo, ao_i = parts.ao;
  const double wo = g->wo[g->pair_wo[pair]];
  const double go = g->go[g->pair_go[pair]];
  const double oo = g->oo[oo_i];
  const double ao = g->ao[ao_i];

  // the key terms are fetched first and used last: the loads are in flight across everything
  // computed here
  double v[kFromKeys ? kKeyRow : 2];
  if (kFromKeys) {
    const int64_t key = (int64_t)(par_i * g->n_ao + ao_i) * g->n_pair + pair;
    const double2 *__restrict__ kt =
        reinterpret_cast<const double2 *>(key_terms + (g->key_offset + key) * MIST_KEY_TERMS);
#pragma unroll
    for (int i = 0; i < kKeyRow / 2; ++i) {
      const double2 two = kt[i];
      v[2 * i] = two.x;
      v[2 * i + 1] = two.y;
    }
  }

  const double *par = g->par[par_i];
  const double ore_size = par[MIST_PAR_ORE] == 1.0 ? par[MIST_PAR_DP] : 1.0;
  const double O = par[MIST_PAR_O], raw_nock = par[MIST_PAR_RAW_NOCK];
  const double mf = memory_factor(prob, par, wo, go, oo, ao);
  const double mf_pp = mf + 0.025;
  const KeyMemory mem = key_memory(g, par, wo, go, ao);
  const double pO = O / ore_size * (1.0 - oo);

  // ---- swap and collective latencies (:1362-1408) ----
  const KeyInputs in = key_inputs(prob, lds_gpu_gpu, g, par, wo, go, ao);
  const double so_O = host_link_latency(prob.gpu_cpu, O / ore_size * oo);
  const double si_O = host_link_latency(prob.cpu_gpu, O / ore_size * oo);
  const bool adv = prob.adv_first_block != 0;

  // ---- forward (:1432-1621) and backward (:1646-1902) families ----
  Family fwd[2][2];  // [0 = first micro-batch, 1 = not first][0 = nock, 1 = ck]
  Family bwd[2][2];  // [0 = last micro-batch, 1 = not last][0 = nock, 1 = ck]
  {
    const FwdOperands op = fwd_operands(in, true, so_O, si_O);
    double first, extra_pre;
    fwd_common(I, in, op, true, adv, first, extra_pre);
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      fwd[0][k].first = first;
      fwd[0][k].extra_pre = extra_pre;
      fwd_of_ckpt(I, in, op, k != 0, fwd[0][k].layer, fwd[0][k].last, fwd[0][k].extra_post);
    }
  }
  if (kFromKeys) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const double *f = v + kKeyBwd + j * 5;
      bwd[j >> 1][j & 1] = Family{f[0], f[1], f[2], f[3], f[4]};
    }
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const double *f = v + kKeyFwd + k * 3;
      fwd[1][k] = Family{f[0], v[kKeyFwdFirst], f[1], v[kKeyFwdExtraPre], f[2]};
    }
  } else {
    const FwdOperands op = fwd_operands(in, false, 0.0, 0.0);
    double first, extra_pre;
    fwd_common(I, in, op, false, adv, first, extra_pre);
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      fwd[1][k].first = first;
      fwd[1][k].extra_pre = extra_pre;
      fwd_of_ckpt(I, in, op, k != 0, fwd[1][k].layer, fwd[1][k].last, fwd[1][k].extra_post);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) bwd[j >> 1][j & 1] = bwd_family(I, in, (j & 2) != 0, (j & 1) != 0);
  }

  // ---- stable / delta families (:1910-2028) ----
  const int st = g->grad_accum == 1 ? 0 : 1;  // phase index that forms the stable part
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    // selected field by field: indexing the arrays with a run-time phase would put them in
    // scratch memory
    const Family f = pick_family(st == 1, fwd[0][k], fwd[1][k]);
    const Family w = pick_family(st == 1, bwd[0][k], bwd[1][k]);
    const double s_layer = f.layer + w.layer;
    const double s_first = f.extra_pre + w.extra_post + f.first + w.first;
    const double s_last = f.extra_post + w.extra_pre + f.last + w.last;
    double d_layer = 0.0, d_first = 0.0, d_last = 0.0;
    if (st == 1) {
      const Family &f1 = fwd[0][k], &w1 = bwd[0][k];
      d_layer = f1.layer + w1.layer - s_layer;
      d_first = f1.extra_pre + w1.extra_post + f1.first + w1.first - s_first;
      d_last = f1.extra_post + w1.extra_pre + f1.last + w1.last - s_last;
    }
    // k == 1 is "with ckpt": the *_CK slot precedes the *_NOCK slot.
    t[MIST_T_S_LAYER_CK + (1 - k)] = s_layer;
    t[MIST_T_S_FIRST_CK + (1 - k)] = s_first;
    t[MIST_T_S_LAST_CK + (1 - k)] = s_last;
    t[MIST_T_D_LAYER_CK + (1 - k)] = d_layer;
    t[MIST_T_D_FIRST_CK + (1 - k)] = d_first;
    t[MIST_T_D_LAST_CK + (1 - k)] = d_last;
  }

  t[MIST_T_FWD_STATES0] = mem.fwd_states0;
  t[MIST_T_BWD_STATES0] = mem.two_buf;
  t[MIST_T_PWG] = mem.pWG;
  t[MIST_T_PO] = pO;
  t[MIST_T_PWGO] = mem.pWG + pO;
  t[MIST_T_S_CK] = mem.S_ck;
  t[MIST_T_S_NOCK] = mem.S_nock;
  t[MIST_T_D_CK] = mem.D_ck;
  t[MIST_T_D_NOCK] = mem.D_nock;
  t[MIST_T_MF_BASE] = mf_pp + 0.01;
  t[MIST_T_MF_PP] = mf_pp;
  t[MIST_T_MF] = mf;
  t[MIST_T_FWD_PEAK] = par[MIST_PAR_FWD_PEAK];
  t[MIST_T_BWD_PEAK] = par[MIST_PAR_BWD_PEAK];
  t[MIST_T_OUT] = par[MIST_PAR_OUT];
  t[MIST_T_GCB] = par[MIST_PAR_GCB];

  const PostTerms post = post_terms(g, in);
  t[MIST_T_NAG_CK] = post.nag_ck;
  t[MIST_T_NAG_NOCK] = post.nag_nock;
  t[MIST_T_NRS_CK] = post.nrs_ck;
  t[MIST_T_NRS_NOCK] = post.nrs_nock;
  t[MIST_T_OPB] = fmax(g->post_bwd - bwd[1][1].extra_pre, 0.0);
  t[MIST_T_RD] = raw_nock - mem.S_nock;
}

// Rows leave a workgroup as contiguous, fully coalesced ranges (a lane writing its own 272-byte row
// would touch 34 partial cache lines): wavefront by wavefront through one LDS buffer of kStageRows
// rows (row pitch 35 doubles: conflict-free).  One buffer for the block, not one per wavefront: LDS
// is what bounds the number of resident wavefronts here.
__device__ __forceinline__ void store_rows(const double *lds_rows, int n, double *__restrict__ out) {
  double2 *__restrict__ dst = reinterpret_cast<double2 *>(out);
  for (int i = threadIdx.x; i < n * (MIST_ROW_TERMS / 2); i += kTermsBlock) {
    const int at = i / (MIST_ROW_TERMS / 2) * (MIST_ROW_TERMS + 1) + 2 * (i % (MIST_ROW_TERMS / 2));
    dst[i] = make_double2(lds_rows[at], lds_rows[at + 1]);
  }
}

// kMode 0: every row of every group, and without key terms (kFromKeys) their stage summaries.
// kMode 1: only the rows the seed launch gathers (workgroup = (128 gathered rows, group)), so that
// it can start before anything else is there.
template <int kMode, bool kFromKeys>
__global__ __launch_bounds__(kTermsBlock) void row_terms_kernel(
    const MistProblem prob, const MistGroupDesc *__restrict__ groups, int n_groups,
    const int32_t *__restrict__ block_prefix, double *__restrict__ row_terms,
    double *__restrict__ stage_floor, const double *__restrict__ key_terms) {
  constexpr bool kFloors = kMode == 0 && !kFromKeys;
  int local_block;
  const MistGroupDesc *g;
  int64_t n_here_total;  // rows this launch computes for the group
  if (kMode == 1) {
    g = groups + blockIdx.y;
    local_block = blockIdx.x;
    n_here_total = g->scout_stride > 0 ? (int64_t)g->n_par * g->n_oo * g->n_ao * g->scout_stride : 0;
    if ((int64_t)local_block * kTermsBlock >= n_here_total) return;
  } else {
    g = find_group(groups, block_prefix, n_groups, blockIdx.x, &local_block);
    n_here_total = g->n_rows;
  }
  __shared__ double lds_out[kMode == 1 ? 1 : kStageRows * (MIST_ROW_TERMS + 1)];
  __shared__ __align__(16) double lds_factor[11][kFactorPitch];
  __shared__ double lds_gpu_gpu[32];
  __shared__ double lds_part[kFloors ? kTermsBlock / kStageRows - 1 : 1][2][kFloors ? kStageFloorPitch : 1];
  InterferenceModel<kFromKeys> I;  // with key terms only the first forward phase is evaluated here
  I.factors_tame = load_model_tables(prob, lds_factor, lds_gpu_gpu);
  I.table = (LdsDouble *)&lds_factor[0][0];
  const int64_t block_first = (int64_t)local_block * kTermsBlock;
  const int rows_here = (int)min((int64_t)kTermsBlock, n_here_total - block_first);
  // Lanes past the end recompute the last row (no divergent barrier); their result is dropped.
  const int64_t nth = block_first + min((int)threadIdx.x, rows_here - 1);
  const int64_t row = kMode == 1 ? gathered_position(g, (uint32_t)nth) : nth;  // workspace position
  double t[MIST_ROW_TERMS];  // compile-time indices only: registers
  row_terms_of<kFromKeys>(prob, g, (uint32_t)row, key_terms, lds_gpu_gpu, I, t);

  if (kMode == 1) {  // scattered rows: every lane writes its own
    if ((int)threadIdx.x < rows_here) {
      double2 *__restrict__ mine =
          reinterpret_cast<double2 *>(row_terms + (g->row_offset + row) * MIST_ROW_TERMS);
#pragma unroll
      for (int i = 0; i < MIST_ROW_TERMS / 2; ++i) mine[i] = make_double2(t[2 * i], t[2 * i + 1]);
    }
    return;
  }
  static_assert(kTermsBlock % kStageRows == 0 && kStageRows == 64, "a wavefront's rows are one stage");
  const int wave = threadIdx.x / kStageRows, lane = threadIdx.x % kStageRows;
  for (int stage_here = 0; stage_here < kTermsBlock / kStageRows; ++stage_here) {
    if (wave == stage_here) {
#pragma unroll
      for (int i = 0; i < MIST_ROW_TERMS; ++i) lds_out[lane * (MIST_ROW_TERMS + 1) + i] = t[i];
    }
    __syncthreads();
    const int stage_first = stage_here * kStageRows;
    const int stage_rows = min(kStageRows, rows_here - stage_first);  // <= 0: nothing left
    store_rows(lds_out, stage_rows, row_terms + (g->row_offset + block_first + stage_first) * MIST_ROW_TERMS);
    if (!kFloors) {
      __syncthreads();
      continue;
    }
    // Summary of the stage: thread = (column, one of kTermsBlock / 32
    // runs of the stage's rows); columns 0 .. MIST_T_GCB hold the minimum, column kStageMaxOut
    // the maximum of MIST_T_OUT, the three behind it minima of post-layer terms.  The runs of a
    // wavefront meet by shuffle, the wavefronts in LDS.
    constexpr int kRuns = kTermsBlock / kStageFloorPitch, kRunRows = kStageRows / kRuns;
    const int col = threadIdx.x & (kStageFloorPitch - 1), run = threadIdx.x / kStageFloorPitch;
    const int src_col = col == kStageMaxOut ? MIST_T_OUT
                        : col == kStageMinOpb ? MIST_T_OPB
                        : col == kStageMinNag ? MIST_T_NAG_CK
                        : col == kStageMinNrs ? MIST_T_NRS_CK : col;
    const int second_col = (col == kStageMinNag || col == kStageMinNrs) ? src_col + 1 : src_col;
    double lo_v = INFINITY, hi_v = 0.0;
    {
#pragma unroll
      for (int i = 0; i < kRunRows; ++i) {
        const int r = run * kRunRows + i;
        const double *row_at = lds_out + min(r, kStageRows - 1) * (MIST_ROW_TERMS + 1);
        const double x = fmin(row_at[src_col], row_at[second_col]);
        lo_v = fmin(lo_v, r < stage_rows ? x : INFINITY);
        hi_v = fmax(hi_v, r < stage_rows ? x : 0.0);
      }
    }
    lo_v = fmin(lo_v, __shfl_xor(lo_v, kStageFloorPitch));
    hi_v = fmax(hi_v, __shfl_xor(hi_v, kStageFloorPitch));
    if (wave > 0 && lane < kStageFloorPitch) {
      lds_part[wave - 1][0][kFloors ? col : 0] = lo_v;
      lds_part[wave - 1][1][kFloors ? col : 0] = hi_v;
    }
    __syncthreads();  // every read of this stage is done; the other wavefronts' parts are in LDS
    if (wave == 0 && lane < kStageFloorPitch && stage_rows > 0) {
#pragma unroll
      for (int w = 0; w < kTermsBlock / kStageRows - 1; ++w) {
        lo_v = fmin(lo_v, lds_part[w][0][kFloors ? col : 0]);
        hi_v = fmax(hi_v, lds_part[w][1][kFloors ? col : 0]);
      }
      const int64_t slot = stage_floor_slot(g, (int)(g - groups), block_first / kStageRows + stage_here);
      stage_floor[slot * kStageFloorPitch + col] = col == kStageMaxOut ? hi_v : lo_v;
    }
  }
}

constexpr int kNumXcd = 8;
// Workgroups are dealt round-robin to the 8 XCDs, each with its own L2.  Logical workgroups
// that read the same rows are consecutive, so runs of kXcdRun logical workgroups are given to
// one XCD (and the runs round-robin, which keeps the XCDs evenly loaded).  The grid is padded to
// a multiple of kNumXcd * kXcdRun; logical indices past the end do nothing.
constexpr int kXcdRun = 16;
__device__ __forceinline__ int xcd_run_block(int physical) {
  const int xcd = physical % kNumXcd, slot = physical / kNumXcd;
  return ((slot / kXcdRun) * kNumXcd + xcd) * kXcdRun + slot % kXcdRun;
}
__host__ __device__ constexpr int xcd_padded_grid(int n_blocks) {
  return (n_blocks + kNumXcd * kXcdRun - 1) / (kNumXcd * kXcdRun) * (kNumXcd * kXcdRun);
}

// Stage summaries of every row, from the key terms and without the rows themselves: the search
// reads the rows of a few stages (22B on 16x8: 67e6 rows, 18 GB, of which 9 % is read), which
// are computed when it is known which (stage_rows_kernel).  Wavefront = stage, lane = row.  The columns a key decides are
// taken from the stage's keys (16 of them as a rule), the six latencies and three memory columns
// that see the optimizer ratio are evaluated per row and meet through LDS.  Bound by the float64
// VALU: 8 evaluations of the interference model per row.
constexpr int kFloorCols = 9;               // 6 latencies, PO, PWGO, MF
constexpr int kFloorPitch = kStageRows + 1;
constexpr int kFloorThreads = 256, kFloorWaves = kFloorThreads / 64;
constexpr int kFloorRun = 32;  // terms blocks (two stages each) of a workgroup of stage_floor_runs_kernel
// Terms blocks from which on the runs are taken.  Their shared parts save a third of the float64 work (1200 vector
// instructions a stage, 810), but a workgroup waits for more in turn and, with 154 registers and three wavefronts a
// SIMD (every row on its own: 120 and four), leaves less room beside the seeds.  Calls of 7B on 4x8, 2x8, LLaMA-13B,
// GPT-22B and LLaMA-70B with finer and finer ratios, time of every row on its own over that of the runs:
//   blocks      7100 - 49800  65300 - 108500  135000 - 170300  224000 - 267000  348000 - 627000
//   inter-stage   1.00 - 1.01   1.00 - 1.02     1.01 - 1.04      1.01 - 1.01      1.01 - 1.07
//   uniform-pp    0.96 - 0.98   0.98 - 0.98     0.99 - 1.00      1.01 - 1.01         1.02
//   whole tables  0.99 - 1.01   1.00 - 1.01                      1.01 - 1.01
// (GPT-22B on 16x8, 528000 blocks: the launch alone 3.0 -> 2.6 ms, from the gathered rows to the filter 5.20 -> 4.64.)
constexpr int kFloorRunBlocks = 1 << 17;
// Parts of the lane's row, `lane` behind the first row of the wavefront: from that one's (wave-uniform), block by
// block (four divisions of the lane's own otherwise, 90 instructions).
__device__ __forceinline__ RowParts row_behind(const MistGroupDesc *g, const RowParts &first, int lane) {
  const int n_tiles = (g->n_oo + kOoTile - 1) / kOoTile;
  RowParts r = first;
  int tile = first.oo / kOoTile, width = min(kOoTile, g->n_oo - tile * kOoTile);
  int rest = first.pair * width + (first.oo - tile * kOoTile) + lane;
  while (__any(rest >= width * g->n_pair)) {
    if (rest < width * g->n_pair) continue;
    rest -= width * g->n_pair;
    if (++tile == n_tiles) {
      tile = 0;
      if (++r.ao == g->n_ao) {
        r.ao = 0;
        ++r.par;
      }
    }
    width = min(kOoTile, g->n_oo - tile * kOoTile);
  }
  // (below 2^16: at most kOoTile pairs of MIST_MAX_PAIRS)
  r.pair = width == 4 ? rest >> 2 : width == 3 ? rest * 43691 >> 17 : width == 2 ? rest >> 1 : rest;
  r.oo = tile * kOoTile + (rest - r.pair * width);
  return r;
}

// The forward parts that a row shares with others of its (parallelism row, activation ratio, tile of optimizer
// ratios): of the first layer and before it per (gradient ratio, optimizer ratio), of the last layer per (weight
// ratio, optimizer ratio), the optimizer's swaps per optimizer ratio.  One stage touches at most 64 / n_pair + 2 such
// blocks of (n_go + n_wo + 1) kOoTile pairs, n_go + n_wo <= n_pair + 1 or 64: 1584 doubles.
constexpr int kFloorShared = 2048;
struct FloorBlocks {
  int n_go, n_wo, n_tiles, per_block;
  __device__ __forceinline__ explicit FloorBlocks(const MistGroupDesc *g) : n_tiles((g->n_oo + kOoTile - 1) / kOoTile) {
    // (the ratios that occur in the pair list, which holds them in order)
    n_go = n_wo = 0;
    for (int i = threadIdx.x & 63; i < g->n_pair; i += 64) {
      n_go = max(n_go, (int)g->pair_go[i] + 1);
      n_wo = max(n_wo, (int)g->pair_wo[i] + 1);
    }
    for (int step = 1; step < 64; step <<= 1) {
      n_go = max(n_go, __shfl_xor(n_go, step));
      n_wo = max(n_wo, __shfl_xor(n_wo, step));
    }
    n_go = __builtin_amdgcn_readfirstlane(n_go);
    n_wo = __builtin_amdgcn_readfirstlane(n_wo);
    per_block = (n_go + n_wo + 1) * kOoTile * 2;
  }
  __device__ __forceinline__ int block_of(const MistGroupDesc *g, const RowParts &at) const {
    return (at.par * g->n_ao + at.ao) * n_tiles + at.oo / kOoTile;
  }
  __device__ __forceinline__ int first_of_go(int go, int oo) const { return (go * kOoTile + oo % kOoTile) * 2; }
  __device__ __forceinline__ int last_of_wo(int wo, int oo) const { return ((n_go + wo) * kOoTile + oo % kOoTile) * 2; }
  __device__ __forceinline__ int swaps(int oo) const { return ((n_go + n_wo) * kOoTile + oo % kOoTile) * 2; }
};

// What the first forward phase reads of a row's KeyInputs, and of its key.
__device__ __forceinline__ KeyInputs floor_inputs(const double *__restrict__ par, double2 links, double2 swapped, double gather) {
  KeyInputs in = {};
  in.exec_fwd = par[MIST_PAR_EXEC_FWD];
  in.extra_fwd = par[MIST_PAR_EXTRA_FWD];
  in.E_f = in.exec_fwd - in.extra_fwd;
  in.ore = 1.0;
  in.AG_w = gather;
  in.so_W = links.x;
  in.si_G = links.y;
  in.so_A_ck = swapped.x;
  in.so_A_nock = swapped.y;
  return in;
}

// The shared parts of blocks [block0, block0 + n_blocks), by the whole workgroup.
__device__ __forceinline__ void floor_shared_parts(const MistProblem &prob, const MistGroupDesc *__restrict__ g,
                                                   const FloorBlocks &blocks, const InterferenceModel<true> &I,
                                                   const double *__restrict__ key_terms, int block0, int n_blocks,
                                                   double *shared) {
  const bool adv = prob.adv_first_block != 0;
  // (entry by entry of all blocks: neighbouring lanes evaluate the same)
  const int per_entry = n_blocks * kOoTile, n_entries = (blocks.n_go + 2 * blocks.n_wo + 1) * per_entry;
  for (int e = threadIdx.x; e < n_entries; e += kFloorThreads) {
    const int entry = e / per_entry, what = e - entry * per_entry, slot = what / kOoTile, block = block0 + slot;
    const int par_ao = block / blocks.n_tiles, tile = block - par_ao * blocks.n_tiles, oo_i = tile * kOoTile + what % kOoTile;
    if (oo_i >= g->n_oo) continue;
    const double *par = g->par[par_ao / g->n_ao];
    const double oo = g->oo[oo_i], dp = par[MIST_PAR_DP];
    const double O_shard = par[MIST_PAR_O] / (par[MIST_PAR_ORE] == 1.0 ? dp : 1.0);
    const double so_O = host_link_latency(prob.gpu_cpu, O_shard * oo);
    const double si_O = host_link_latency(prob.cpu_gpu, O_shard * oo);
    // (the gather and the swaps of saved activations are those of any key of the block)
    const double *__restrict__ key = key_terms + (g->key_offset + (int64_t)par_ao * g->n_pair) * MIST_KEY_TERMS;
    const double2 swapped = make_double2(key[kKeySoA], key[kKeySoA + 1]);
    double *out = shared + slot * blocks.per_block;
    if (entry < blocks.n_go) {
      const double gre_size = par[MIST_PAR_GRE] == 1.0 ? dp : 1.0;
      const double si_G = host_link_latency(prob.cpu_gpu, par[MIST_PAR_G] / gre_size * g->go[entry]);
      const KeyInputs in = floor_inputs(par, make_double2(0.0, si_G), swapped, key[kKeyGather]);
      double first, extra_pre;
      fwd_common(I, in, fwd_operands(in, true, so_O, si_O), true, adv, first, extra_pre);
      *reinterpret_cast<double2 *>(out + blocks.first_of_go(entry, oo_i)) = make_double2(first, extra_pre);
    } else if (entry < blocks.n_go + 2 * blocks.n_wo) {
      const int k = (entry - blocks.n_go) & 1, wo = (entry - blocks.n_go) >> 1;  // (with ckpt in front of without)
      const double wre_size = par[MIST_PAR_WRE] == 1.0 ? dp : 1.0;
      const double so_W = host_link_latency(prob.gpu_cpu, par[MIST_PAR_W] / wre_size * g->wo[wo]);
      const KeyInputs in = floor_inputs(par, make_double2(so_W, 0.0), swapped, key[kKeyGather]);
      const FwdOperands op = fwd_operands(in, true, so_O, si_O);
      out[blocks.last_of_wo(wo, oo_i) + k] = I.exec_g2c(in.E_f, op.g2c + (k == 0 ? in.so_A_ck : in.so_A_nock)) + in.extra_fwd;
    } else {
      *reinterpret_cast<double2 *>(out + blocks.swaps(oo_i)) = make_double2(so_O, si_O);
    }
  }
}

// (kShared false: the stage's blocks have no room, as with a pair list of a few pairs from long lists of ratios)
template <bool kShared>
__device__ __forceinline__ void stage_floor_of(const MistProblem &prob, const MistGroupDesc *__restrict__ g, int gi, int stage,
                                               const FloorBlocks *blocks, int block0, const double *shared,
                                               const InterferenceModel<true> &I, const double *__restrict__ key_terms,
                                               double *__restrict__ stage_floor, double *mine, int *keys) {
  const int lane = threadIdx.x & 63;
  // (lanes past the end repeat the last row: minima do not change)
  const int64_t row0 = (int64_t)stage * kStageRows;
  const RowParts at = row_behind(g, parts_of_position(g, (uint32_t)row0), (int)min((int64_t)lane, g->n_rows - 1 - row0));
  const int key = (at.par * g->n_ao + at.ao) * g->n_pair + at.pair;
  const double2 *__restrict__ kt =
      reinterpret_cast<const double2 *>(key_terms + (g->key_offset + key) * MIST_KEY_TERMS);
  double2 bwd[5], cols[3], links[3];
#pragma unroll
  for (int i = 0; i < 5; ++i) bwd[i] = kt[kKeyBwd / 2 + i];
#pragma unroll
  for (int i = 0; i < 3; ++i) links[i] = kt[kKeySoW / 2 + i];
#pragma unroll
  for (int i = 0; i < 3; ++i) cols[i] = kt[kKeyCols / 2 + i];
  const double pWG = reinterpret_cast<const double *>(kt)[kKeyState0 + 2];
  const double gather = reinterpret_cast<const double *>(kt)[kKeyGather];

  const double *par = g->par[at.par];
  const double oo = g->oo[at.oo];
  const KeyInputs in = floor_inputs(par, links[0], links[1], gather);
  const double O_shard = par[MIST_PAR_O] / (par[MIST_PAR_ORE] == 1.0 ? par[MIST_PAR_DP] : 1.0);
  double first, extra_pre;
  double2 of_last, swaps;
  if constexpr (kShared) {
    const double *its = shared + (blocks->block_of(g, at) - block0) * blocks->per_block;
    const double2 of_first = *reinterpret_cast<const double2 *>(its + blocks->first_of_go(g->pair_go[at.pair], at.oo));
    first = of_first.x;
    extra_pre = of_first.y;
    of_last = *reinterpret_cast<const double2 *>(its + blocks->last_of_wo(g->pair_wo[at.pair], at.oo));
    swaps = *reinterpret_cast<const double2 *>(its + blocks->swaps(at.oo));
  } else {
    swaps = make_double2(host_link_latency(prob.gpu_cpu, O_shard * oo), host_link_latency(prob.cpu_gpu, O_shard * oo));
    const FwdOperands op = fwd_operands(in, true, swaps.x, swaps.y);
    fwd_common(I, in, op, true, prob.adv_first_block != 0, first, extra_pre);
    of_last = make_double2(I.exec_g2c(in.E_f, op.g2c + in.so_A_ck) + in.extra_fwd,
                           I.exec_g2c(in.E_f, op.g2c + in.so_A_nock) + in.extra_fwd);
  }
  const FwdOperands op = fwd_operands(in, true, swaps.x, swaps.y);
  const bool accumulates = g->grad_accum != 1;
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const double g2c = op.g2c + (k ? in.so_A_ck : in.so_A_nock), last = k ? of_last.x : of_last.y;
    const double layer = I(in.E_f, op.g2g, g2c, op.c2g) + in.extra_fwd, extra_post = I.g2c_only(g2c);
    // backward family of the last micro-batch: layer, first, last, extra_pre, extra_post
    const double b_layer = k ? bwd[2].y : bwd[0].x, b_first = k ? bwd[3].x : bwd[0].y;
    const double b_last = k ? bwd[3].y : bwd[1].x, b_pre = k ? bwd[4].x : bwd[1].y;
    const double b_post = k ? bwd[4].y : bwd[2].x;
    double v_layer = layer + b_layer;
    double v_first = extra_pre + b_post + first + b_first;
    double v_last = extra_post + b_pre + last + b_last;
    if (accumulates) {  // the delta part
      v_layer = v_layer - (k ? cols[0].x : cols[0].y);
      v_first = v_first - (k ? cols[1].x : cols[1].y);
      v_last = v_last - (k ? cols[2].x : cols[2].y);
    }
    mine[(0 + (1 - k)) * kFloorPitch + lane] = v_layer;
    mine[(2 + (1 - k)) * kFloorPitch + lane] = v_first;
    mine[(4 + (1 - k)) * kFloorPitch + lane] = v_last;
  }
  const double pO = O_shard * (1.0 - oo);
  mine[6 * kFloorPitch + lane] = pO;
  mine[7 * kFloorPitch + lane] = pWG + pO;
  mine[8 * kFloorPitch + lane] = oo > 0.0 ? links[2].y : links[2].x;
  // the stage's keys, each once
  const bool new_key = lane == 0 || key != __shfl_up(key, 1);
  const uint64_t new_keys = __ballot(new_key);
  if (new_key) keys[__popcll(new_keys & ((1ull << lane) - 1ull))] = key;
  const int n_keys = __popcll(new_keys);
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();

  // ---- lane = (column of the keys, parity) ----
  double lo = INFINITY, hi = 0.0;
  {
    const int col = lane & 31, parity = lane >> 5;
    const double *__restrict__ src =
        key_terms + g->key_offset * MIST_KEY_TERMS + kKeyCols + min(col, kKeyColsEnd - kKeyCols - 1);
#pragma unroll 8
    for (int i = parity; i < n_keys; i += 2) {
      const double v = src[(int64_t)keys[i] * MIST_KEY_TERMS];
      lo = fmin(lo, v);
      hi = fmax(hi, v);
    }
    lo = fmin(lo, __shfl_xor(lo, 32));
    hi = fmax(hi, __shfl_xor(hi, 32));
  }
  // ---- lane = (column of the rows, a quarter of them) ----
  double row_lo = INFINITY;
  {
    const double *src = mine + min(lane & 15, kFloorCols - 1) * kFloorPitch + (lane >> 4) * 16;
#pragma unroll
    for (int i = 0; i < 16; ++i) row_lo = fmin(row_lo, src[i]);
    row_lo = fmin(row_lo, __shfl_xor(row_lo, 16));
    row_lo = fmin(row_lo, __shfl_xor(row_lo, 32));
  }
  double *__restrict__ out = stage_floor + stage_floor_slot(g, gi, stage) * kStageFloorPitch;
  // summary column `lane`: from which of the two, and from which column of it
  const double mf = from_lane(row_lo, 8);
  const bool latency_of_rows = accumulates ? (lane >= 6 && lane < 12) : lane < 6;
  const int key_col = lane < 6 ? lane
                      : lane <= MIST_T_BWD_STATES0 ? kKeyState0 - kKeyCols + (lane - MIST_T_FWD_STATES0)
                      : lane == MIST_T_PWG ? kKeyState0 - kKeyCols + 2
                      : lane <= MIST_T_D_NOCK ? kKeyState0 - kKeyCols + 3 + (lane - MIST_T_S_CK)
                      : lane <= MIST_T_GCB ? kKeyPeaks - kKeyCols + (lane - MIST_T_FWD_PEAK)
                      : lane == kStageMaxOut ? kKeyPeaks - kKeyCols + 2
                                             : kKeyPost - kKeyCols + (lane - kStageMinOpb);
  const double of_keys = __shfl(lo, max(key_col, 0));
  const double max_out = from_lane(hi, kKeyPeaks - kKeyCols + 2);
  const double of_rows = __shfl(row_lo, lane == MIST_T_PO ? 6 : lane == MIST_T_PWGO ? 7 : lane % 6);
  double v = of_keys;
  if (latency_of_rows || lane == MIST_T_PO || lane == MIST_T_PWGO) v = of_rows;
  else if (lane >= 6 && lane < 12) v = 0.0;  // one micro-batch: no delta part
  else if (lane == MIST_T_MF) v = mf;
  else if (lane == MIST_T_MF_PP) v = mf + 0.025;
  else if (lane == MIST_T_MF_BASE) v = mf + 0.025 + 0.01;
  else if (lane == kStageMaxOut) v = max_out;
  if (lane < kStageFloorPitch) out[lane] = v;
  // the wavefront's next stage writes `mine` and `keys` again
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// Workgroup = two stages, every row on its own.
__global__ __launch_bounds__(kTermsBlock) void stage_floor_kernel(
    const MistProblem prob, const MistGroupDesc *__restrict__ groups, int n_groups,
    const int32_t *__restrict__ block_prefix, double *__restrict__ stage_floor, const double *__restrict__ key_terms) {
  constexpr int kStages = kTermsBlock / kStageRows;
  __shared__ __align__(16) double lds_factor[11][kFactorPitch];
  __shared__ double lds_gpu_gpu[32];  // (of the tables, not read here)
  __shared__ double lds_cols[kStages][kFloorCols * kFloorPitch];
  __shared__ int lds_keys[kStages][kStageRows];
  int local_block;
  const MistGroupDesc *g = find_group(groups, block_prefix, n_groups, blockIdx.x, &local_block);
  const int gi = __builtin_amdgcn_readfirstlane((int)(g - groups));
  g = groups + gi;
  InterferenceModel<true> I;
  I.factors_tame = load_model_tables(prob, lds_factor, lds_gpu_gpu);
  I.table = (LdsDouble *)&lds_factor[0][0];
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x / kStageRows);
  const int stage = __builtin_amdgcn_readfirstlane(local_block) * kStages + wave;
  if ((int64_t)stage * kStageRows >= g->n_rows) return;
  stage_floor_of<false>(prob, g, gi, stage, nullptr, 0, nullptr, I, key_terms, stage_floor, lds_cols[wave], lds_keys[wave]);
}

// Workgroup = kFloorRun terms blocks, stage by stage in its wavefronts, with what their rows share evaluated before.
__global__ __launch_bounds__(kFloorThreads) void stage_floor_runs_kernel(
    const MistProblem prob, const MistGroupDesc *__restrict__ groups, int n_groups,
    const int32_t *__restrict__ block_prefix, int n_blocks, double *__restrict__ stage_floor,
    const double *__restrict__ key_terms) {
  __shared__ __align__(16) double lds_factor[11][kFactorPitch];
  __shared__ double lds_gpu_gpu[32];  // (of the tables, not read here)
  __shared__ double lds_cols[kFloorWaves][kFloorCols * kFloorPitch];
  __shared__ int lds_keys[kFloorWaves][kStageRows];
  __shared__ __align__(16) double shared[kFloorShared];
  InterferenceModel<true> I;
  I.factors_tame = load_model_tables(prob, lds_factor, lds_gpu_gpu);
  I.table = (LdsDouble *)&lds_factor[0][0];
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  constexpr int kStages = kTermsBlock / kStageRows;
  const int first_block = xcd_run_block(blockIdx.x) * kFloorRun;
  const int end = min(first_block + kFloorRun, n_blocks);
  for (int block = first_block; block < end;) {  // (a run may hold parts of several groups)
    int local_block;
    const MistGroupDesc *g = find_group(groups, block_prefix, n_groups, block, &local_block);
    const int gi = __builtin_amdgcn_readfirstlane((int)(g - groups));
    g = groups + gi;
    const int here = min(end, block_prefix[gi + 1]) - block;
    const int n_stages = (int)((g->n_rows + kStageRows - 1) / kStageRows);
    const int stage1 = min((local_block + here) * kStages, n_stages);
    const FloorBlocks blocks(g);
    for (int stage0 = local_block * kStages; stage0 < stage1;) {
      // as many stages as there is room for their blocks
      const int block0 = blocks.block_of(g, parts_of_position(g, (uint32_t)stage0 * kStageRows));
      int n = stage1 - stage0, n_touched;
      for (;; n = (n + 1) / 2) {
        const int64_t last = min((int64_t)(stage0 + n) * kStageRows, g->n_rows) - 1;
        n_touched = blocks.block_of(g, parts_of_position(g, (uint32_t)last)) - block0 + 1;
        if (n == 1 || n_touched * blocks.per_block <= kFloorShared) break;
      }
      if (n_touched * blocks.per_block > kFloorShared) {
        if (wave == 0)
          stage_floor_of<false>(prob, g, gi, stage0, &blocks, block0, shared, I, key_terms, stage_floor, lds_cols[0], lds_keys[0]);
        ++stage0;
        continue;
      }
      __syncthreads();  // the wavefronts are done with the blocks before
      floor_shared_parts(prob, g, blocks, I, key_terms, block0, n_touched, shared);
      __syncthreads();
      for (int stage = stage0 + wave; stage < stage0 + n; stage += kFloorWaves)
        stage_floor_of<true>(prob, g, gi, stage, &blocks, block0, shared, I, key_terms, stage_floor, lds_cols[wave], lds_keys[wave]);
      stage0 += n;
    }
    block += here;
  }
}

// ------------------------------------------------------------------------------------------
// Per-cell evaluation of the evaluate-every-cell, first-estimate, finalize and analysis kernels.
// ------------------------------------------------------------------------------------------
struct PairIndex {
  int l, c;  // layers in the stage (1..L), checkpointed layers (0..l)
};

// Valid (l, c <= l) pairs are numbered l-major: index(l, c) = l*(l+1)/2 - 1 + c.
__device__ __forceinline__ PairIndex decode_pair(int idx) {
  // (the float32 root is off by less than 1 up to 32765 layers; the loops settle it)
  int l = (int)((__builtin_amdgcn_sqrtf(__builtin_fmaf(8.0f, (float)idx, 9.0f)) - 1.0f) * 0.5f);
  while (l * (l + 1) / 2 - 1 > idx) --l;
  while ((l + 1) * (l + 2) / 2 - 1 <= idx) ++l;
  return PairIndex{l, idx - (l * (l + 1) / 2 - 1)};
}

struct CellLatency {
  float x, d;           // stable, delta rounded to float32 (batched_module_analyzer.py:2212-2213)
  double sp, dpre;      // with_pre stable / delta (float64)
  double spost, dpost;  // with_post
  double spp, dpp;      // pre_and_post (no_pp)
};

struct GroupConsts {
  double pre_fwd, pre_bwd, post_fwd;
  double w1, w2, w1d, w2d;  // pre-layer all-gather / reduce-scatter split into stable / delta
  bool pp_wre, pp_gre;
};

__device__ __forceinline__ GroupConsts group_consts(const MistGroupDesc *g) {
  GroupConsts k;
  k.pre_fwd = g->pre_fwd;
  k.pre_bwd = g->pre_bwd;
  k.post_fwd = g->post_fwd;
  k.pp_wre = g->pp_wre == 1;
  k.pp_gre = g->pp_gre == 1;
  k.w1 = k.pp_wre ? g->pre_ag : 0.0;
  k.w2 = k.pp_gre ? g->pre_rs : 0.0;
  k.w1d = k.pp_wre ? 0.0 : g->pre_ag;
  k.w2d = k.pp_gre ? 0.0 : g->pre_rs;
  return k;
}

// get_latencies (:2165-2216) and the pre / post additions (:2233-2351) for one row and (l, c).
template <bool kWithPost>
__device__ __forceinline__ CellLatency cell_latency(const double *__restrict__ t, int l, int c,
                                                    const GroupConsts &k) {
  const int lm2 = max(l - 2, 0);
  const int n_ck = min(max(c - 1, 0), lm2);
  const int n_nock = lm2 - n_ck;
  const bool all_ck = c == l, no_ck = c == 0;
  const double stable = (double)n_ck * t[MIST_T_S_LAYER_CK] + (double)n_nock * t[MIST_T_S_LAYER_NOCK] +
                        (all_ck ? t[MIST_T_S_FIRST_CK] : t[MIST_T_S_FIRST_NOCK]) +
                        (no_ck ? t[MIST_T_S_LAST_NOCK] : t[MIST_T_S_LAST_CK]);
  const double delta = (double)n_ck * t[MIST_T_D_LAYER_CK] + (double)n_nock * t[MIST_T_D_LAYER_NOCK] +
                       (all_ck ? t[MIST_T_D_FIRST_CK] : t[MIST_T_D_FIRST_NOCK]) +
                       (no_ck ? t[MIST_T_D_LAST_NOCK] : t[MIST_T_D_LAST_CK]);
  CellLatency r;
  r.x = (float)stable;
  r.d = (float)delta;
  const double x = (double)r.x, d = (double)r.d;
  r.sp = x + k.pre_fwd + k.pre_bwd + k.w1 + k.w2;
  r.dpre = d + k.w1d + k.w2d;
  if (kWithPost) {
    const double nag = c > 0 ? t[MIST_T_NAG_CK] : t[MIST_T_NAG_NOCK];
    const double nrs = c > 0 ? t[MIST_T_NRS_CK] : t[MIST_T_NRS_NOCK];
    const double ps1 = k.pp_wre ? nag : 0.0, ps2 = k.pp_gre ? nrs : 0.0;
    const double pd1 = k.pp_wre ? 0.0 : nag, pd2 = k.pp_gre ? 0.0 : nrs;
    const double opb = t[MIST_T_OPB];
    r.spost = x + k.post_fwd + opb + ps1 + ps2;
    r.dpost = d + pd1 + pd2;
    r.spp = x + k.pre_fwd + k.pre_bwd + k.post_fwd + opb + k.w1 + k.w2 + ps1 + ps2;
    r.dpp = d + k.w1d + k.w2d + pd1 + pd2;
  } else {
    r.spost = r.dpost = r.spp = r.dpp = 0.0;
  }
  return r;
}

// Lexicographic (cost, row) minimum.  The reference scans rows in ascending order with a strict
// "<" (mist/utils/pareto.py:134-142), i.e. it keeps the lowest row among those with the
// smallest cost; comparing (cost, row) pairs gives the same winner in any processing order.
__device__ __forceinline__ bool lex_less(double cost, int32_t row, double best, int32_t best_row) {
  return cost < best || (cost == best && row < best_row);
}

__device__ __forceinline__ void take_min(double &best, int32_t &best_row, bool feasible,
                                         double cost, int32_t row) {
  const bool better = feasible && lex_less(cost, row, best, best_row);
  best = better ? cost : best;
  best_row = better ? row : best_row;
}

// ------------------------------------------------------------------------------------------
// Kernels 2: evaluate + mask + argmin.
//
// Memory feasibility is monotone in p: the peaks are built from p * (non-negative) terms by
// additions only, every floating-point add / multiply is monotone in each operand, and the
// host rejects negative table values.  So per (row, l, c) the feasible p form a prefix
// [0, count) and a row matters to one number per variant: its cost against the minimum of slot
// count - 1 (the minima of a (l, c) pair do not decrease with p).
//
// The minima of every (group, (l, c) pair, variant, p, sample) live in one table in HBM
// (ReduceTables.best) that all wavefronts lower by float64 atomic minima (an objective can be
// negative: the first micro-batch may be cheaper than the later ones, which swap weights in, and
// with a small alpha and few accumulation steps its share of the difference outweighs the rest).
// Five launches:
//   seed     the rows of the group's scout pairs against empty minima, in LDS: upper bounds made
//            of real rows, final for most cells;
//   filter   stage summaries (term-wise minima of 64 rows, and of 8 such stages) against the
//            largest minimum of each pair; what some pair of a tile does not rule out becomes an
//            item (group, tile, stage) of a queue;
//   open     runs of items per wavefront: the summary with the minima of the slots the stage can reach;
//            which pairs stay open goes along;
//   reduce   what is left, shared out by pairs: linear bounds of 64 rows against a pair's minima, then
//            the reference's arithmetic for the candidates of several pairs.  A smaller cost than the
//            minimum at the row's own slot (count - 1) lowers it, and every row that was not above it
//            is noted with its cost in a log.  The slots below take part in finalize, which takes each
//            p's winner from the slots at and above it;
//   resolve  of the rows in the log whose cost is the final minimum the lowest number stays, which is the
//            reference's first-index-wins scan (pareto.py:134-142) in any processing order.  (A log that
//            ran full is left alone: the opened items go through the reduce launch's code once more.)
// What this replaces kept 34 (cost, row) minima per lane in registers (253 of them, two
// wavefronts per SIMD), one sample and 16 p values per pass over the rows, visited every stage
// summary with every tile and p tile, and committed rows one by one per lane: 7B on 4x8, one
// sample: 1.35 ms (0.42 of it seeds); now seeds 0.26 beside key terms and summaries, filter 0.04, open 0.04,
// reduce 0.19, resolve 0.01.  30 samples of the 7B plan's tables for one tensor-parallel size: 24 ms;
// now 3.2 (reduce 2.1, open 0.42, seeds 0.33, filter 0.17, resolve 0.08).
// ------------------------------------------------------------------------------------------
constexpr int kSuperStages = 8;    // stages per second-level summary
constexpr int kGatherFloor = 5;    // linear bounds of 64 gathered rows
constexpr int kQueueShards = 64;   // counters of the item queue: one would serve an append in ~8 ns
constexpr int kCounterPitch = 32;  // uint32 between counters: a cache line each
// Entries of the log that a reduce wavefront takes at a time, and the most entries of a log, 16 bytes each.  Used are
// 0.1 to 2 per entry of the minima as a rule (13e6 with 30 samples of one tensor-parallel size of the 7B plan), but
// 20e6 = 5 per entry of 70B with 48 layers on 25x8 and 39e6 = 2 of 75 layers on 8x8, both without checkpoint tuning,
// whose bound prunes little; a log that runs full costs three times the resolve launch it replaced (the two calls
// with room for 4 per entry and 25e6 at most: 11.1 and 30.5 ms, now 8.3 and 21.9, without a log 9.2 and 28.6).
constexpr int kLogChunk = 256;
constexpr int64_t kLogEntries = 96 << 20;
constexpr int kLogPerCell = 8;
constexpr int kLogTaken = 3 * kQueueShards + kNumXcd;  // counters: chunks taken, whether there were too few
constexpr int kLogFull = kLogTaken + 1;
constexpr int kGroupsDone = kLogFull + 1;  // workgroups of the estimate that have ended
constexpr int kCounters = kGroupsDone + 1;
constexpr int kOpenPairs = 1;  // words behind the counter of a shard's opened items: their open pairs
constexpr int kSeedThreads = 256;
constexpr int kReduceThreads = 256;
constexpr int kReduceBlocks = 2048;          // a multiple of kNumXcd
constexpr int kReduceWorkers = 768;           // three per CU, as many as are resident: 2048 end 6 us later
constexpr int kAgainBlocks = 768;            // three per CU: as a rule they return at once
constexpr int kStageRowsBlocks = 1024;       // four per CU, two stages at a time each
constexpr int kSuperBlocks = 64;             // workgroups per group of the second-level summaries
constexpr int kSeedLdsBytes = 40 * 1024;     // LDS aimed at per seed workgroup: four per CU
constexpr int kSeedWorkgroups = 2048;
constexpr int kSeedLdsMost = 160 * 1024;
// (row, pair) candidates a reduce wavefront collects: 64 that wait, and a pair's 64.
constexpr int kCandidates = 128;
constexpr int kCandidateDoubles = kCandidates * 2 / 8;
// Minima of one pair that every wavefront of a reduce workgroup can hold in LDS beside them: 2543
// values of p.
constexpr int kMostBufferedSlots = kSeedLdsMost / (8 * (kReduceThreads / 64)) - kCandidateDoubles;
static_assert(kQueueShards == 64, "a lane per shard");
// Room below r x and below the terms the composite objectives add (their roundings: a few 1e-16) ...
constexpr double kSlack = 1e-9;
// ... and below d / G, which the base objective rounds to float32 (one part in 2^24).  Relative to
// the operands, not to their sum: d can be negative, and where r x and d / G cancel the sum is far
// smaller than what was rounded.
constexpr double kShareSlack = 1e-7;

// A (group, tile, stage) of the queues in one word: 65535 groups, stages of fewer than 2^31 rows, and
// the rest for the tiles of the pair list (32765 layers).
constexpr int kItemStageBits = 25, kItemTileBits = 23;
static_assert((((int64_t)1 << 31) + kStageRows - 1) / kStageRows <= (int64_t)1 << kItemStageBits, "stages of a group");
struct Item {
  int group, tile, stage;
  __device__ __forceinline__ explicit Item(uint64_t word)
      : group((int)(word >> (kItemTileBits + kItemStageBits))),
        tile((int)(word >> kItemStageBits & ((1u << kItemTileBits) - 1u))),
        stage((int)(word & ((1u << kItemStageBits) - 1u))) {}
  __device__ __forceinline__ Item(int its_group, int its_tile, int its_stage)
      : group(its_group), tile(its_tile), stage(its_stage) {}
  __device__ __forceinline__ unsigned long long word() const {
    return (unsigned long long)group << (kItemTileBits + kItemStageBits) | (unsigned long long)tile << kItemStageBits |
           (unsigned long long)stage;
  }
};

// A row that was not above the minimum of its slot when it was looked at.
struct Hit {
  double cost;
  uint32_t cell;  // of `best`
  uint32_t row;
};
static_assert(sizeof(Hit) == 16, "two doubles of the workspace");

// MistProblem.incumbent_close: what reads the tables.
constexpr int kCloseSearch = 1, kCloseAssignment = 2;
// What a group's stage costs can be used for (form_reach).
struct GroupReach {
  double per_layer, rest;  // of every row at least rest + (layers - 2) x per_layer (two layers or fewer: rest)
  double cutoff;           // rows above it are not looked for
  double low;              // a minimum below it, of a stage of fewer than `first` layers, is final as it is
  int first, last;         // for an assignment: the layers a stage may have
};
static_assert(sizeof(GroupReach) == 5 * sizeof(double), "doubles of the workspace");
constexpr int kReachGroups = 2048;  // the most groups that get one: 48 KB of LDS

// (by value in the kernel arguments)
struct ReduceTables {
  double *best;  // [pair][slot][sample] (slots_of(num_p) slots): the smallest cost
  uint32_t *row;  // its lowest row, ~0 = none (from the resolve launch)
  Hit *log;             // [log_chunks][kLogChunk]
  uint32_t *log_count;  // [log_chunks]: entries of each
  double *super_floor;       // [supers][kStageFloorPitch]
  struct GroupReach *reach;  // [group], with MistProblem.incumbent_close
  double *reach_parts;       // [group][kSuperBlocks][2]: of each workgroup of the second-level summaries
  double *gather_floor;      // [stage][kGatherFloor]: what the seed launch asks of 64 gathered rows (one sample)
  // [kQueueShards][capacity]: Item, what the filter and then what the open launch left; open pairs of the
  // latter
  unsigned long long *item, *opened, *open_pairs;
  // [kQueueShards][capacity]: group << 32 | stage of the stages opened, each once; stage_flag (one
  // per stage summary) tells whether one is listed.  Null: the rows of all stages are there.
  unsigned long long *listed;
  uint32_t *stage_flag;
  // at kCounterPitch: [kQueueShards] items, [kQueueShards] opened (with their pairs), [kQueueShards] listed, [kNumXcd] drawn,
  // kLogTaken, kLogFull, kGroupsDone
  uint32_t *counter;
  uint32_t capacity, log_chunks;
  int n_samples;
};

struct LaneMemory {
  double fwd_states, bwd_states, cur_saved, mod_saved, ck_delta, fwd_pk, bwd_pk, out, gcb;
  double mf_base, mf_pp;

  // Peaks of the middle-stage variant for p pre-saved micro-batches (:2755-2786).
  __device__ __forceinline__ void peaks(int p, double &peak_f, double &peak_b) const {
    const double pf64 = (double)p;
    const double pipe_saved = pf64 * mod_saved + cur_saved;
    const double outp2 = out * pf64 * 2.0;
    const double out2 = out * 2.0;
    peak_f = fwd_states + pipe_saved + ck_delta + fwd_pk + outp2 + gcb;
    peak_b = bwd_states + pipe_saved + ck_delta + bwd_pk + outp2 + out2 + gcb;
  }
  // Left-hand sides of the reference's memory tests; a candidate is feasible iff <= capacity.
  __device__ __forceinline__ double scaled_base(int p) const {  // (:2805-2812)
    double pf, pb;
    peaks(p, pf, pb);
    return fmax(pf, pb) * mf_base;
  }
  __device__ __forceinline__ double scaled_pre(int p, double pre_saved,
                                               double pre_sas) const {  // (:2866-2875, 2893-2897)
    double pf, pb;
    peaks(p, pf, pb);
    const double pre_p = (double)p * pre_saved;
    return fmax(pre_p + pf + pre_sas, pre_p + pb + pre_sas) * mf_pp;
  }
  __device__ __forceinline__ bool feasible_base(int p, double cap) const {
    return scaled_base(p) <= cap;
  }
  __device__ __forceinline__ bool feasible_pre(int p, double cap, double pre_saved,
                                               double pre_sas) const {
    return scaled_pre(p, pre_saved, pre_sas) <= cap;
  }
};

__device__ __forceinline__ LaneMemory cell_memory(const double *__restrict__ t, int l, int c);

// The search's winners sit almost exclusively on rows whose (weight, gradient) offload pair is
// the first one, (0, 0): 99.8 % of all cells of the GPT-7B plan, 95 % for LLaMA-13B.  In the
// workspace order those rows are scattered (one per (parallelism row, activation ratio, optimizer
// ratio)); the seed launch gathers them, n_par * n_oo * n_ao rows per group.
// With scout_stride = m > 1 the rows of the pairs scout_pair[1 .. m-1] follow.
// (32-bit arithmetic: q and positions are below the number of rows)
__device__ __forceinline__ int64_t gathered_position(const MistGroupDesc *g, uint32_t q) {
  const uint32_t n_ao = (uint32_t)g->n_ao, n_oo = (uint32_t)g->n_oo, n_tail = n_oo * n_ao;
  const uint32_t per_pair = (uint32_t)g->n_par * n_tail;
  const uint32_t k = q / per_pair, rest = q - k * per_pair;
  const uint32_t par = rest / n_tail, tail = rest - par * n_tail;
  const uint32_t ao = tail / n_oo, oo = tail - ao * n_oo;
  const int pair = g->scout_pair[k];
  return (int64_t)(par * (uint32_t)g->n_off + ao * n_oo * (uint32_t)g->n_pair) + tile_position(g, (int)oo, pair);
}

// alpha / (1 - alpha) of the samples of one launch (by value in the kernel arguments)
struct RatioList {
  double r[MIST_MAX_SAMPLE_BATCH];
};
// sample position in the output tables of each sample of one finalize launch
struct SampleSlots {
  int32_t at[MIST_MAX_SAMPLE_BATCH];
};

// Smallest of the wavefront's values, in every lane (rows of 16 lanes, then across the rows).
__device__ __forceinline__ uint32_t wave_min(uint32_t v) {
#define MIST_MIN_DPP(CTRL) \
  v = min(v, (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, CTRL, 0xf, 0xf, false))
  MIST_MIN_DPP(0x111);  // row_shr:1
  MIST_MIN_DPP(0x112);
  MIST_MIN_DPP(0x114);
  MIST_MIN_DPP(0x118);
  MIST_MIN_DPP(0x142);  // row_bcast:15
  MIST_MIN_DPP(0x143);  // row_bcast:31
#undef MIST_MIN_DPP
  return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}
// A lane with `pending` whose cost is the smallest to float32.  (Keys of floats in their order: all
// bits flipped under a sign, else the sign bit.)
__device__ __forceinline__ int cheapest_lane(bool pending, double cost) {
  const int bits = __float_as_int((float)cost);
  const uint32_t key = pending ? (uint32_t)bits ^ ((uint32_t)(bits >> 31) | 0x80000000u) : ~0u;
  return __ffsll((unsigned long long)__ballot(key == wave_min(key))) - 1;
}
// One entry of the minima in device memory / in LDS (global_atomic_min_f64, ds_min_f64).
__device__ __forceinline__ void lower_minimum(double *entry, double cost) {
  __hip_atomic_fetch_min(entry, cost, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ double load_at_agent(const double *at) {
  return __hip_atomic_load(at, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void lower_minimum_in_lds(double *entry, double cost) {
  __hip_atomic_fetch_min(entry, cost, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// Slots of a pair in ReduceTables: base p = 0.., with_pre p = 0.., with_post, no_pp.
__host__ __device__ constexpr int slots_of(int num_p) { return 2 * num_p + 2; }

// What is the same for all rows of one (l, c) pair; l and c may be wave-uniform or per lane.
struct PairConsts {
  double n_ck, n_nock, lf, lm1, cf, l_minus_c, l_minus_c_1;
  bool all_ck, no_ck, ck_tail;
};
__device__ __forceinline__ PairConsts pair_consts(int l, int c) {
  PairConsts k;
  const int lm2 = max(l - 2, 0), n_ck = min(max(c - 1, 0), lm2);
  k.n_ck = (double)n_ck;
  k.n_nock = (double)(lm2 - n_ck);
  k.lf = (double)l;
  k.lm1 = (double)max(l - 1, 0);
  k.cf = (double)c;
  k.l_minus_c = (double)(l - c);
  k.l_minus_c_1 = (double)(l - c - 1);
  k.all_ck = c == l;
  k.no_ck = c == 0;
  k.ck_tail = c >= l - 1;
  return k;
}

// Stable / delta latency rounded to float32 (get_latencies, :2165-2216).
template <class Row>
__device__ __forceinline__ void pair_latency(const Row &t, const PairConsts &k, float &x, float &d) {
  const double stable = k.n_ck * t[MIST_T_S_LAYER_CK] + k.n_nock * t[MIST_T_S_LAYER_NOCK] +
                        (k.all_ck ? t[MIST_T_S_FIRST_CK] : t[MIST_T_S_FIRST_NOCK]) +
                        (k.no_ck ? t[MIST_T_S_LAST_NOCK] : t[MIST_T_S_LAST_CK]);
  const double delta = k.n_ck * t[MIST_T_D_LAYER_CK] + k.n_nock * t[MIST_T_D_LAYER_NOCK] +
                       (k.all_ck ? t[MIST_T_D_FIRST_CK] : t[MIST_T_D_FIRST_NOCK]) +
                       (k.no_ck ? t[MIST_T_D_LAST_NOCK] : t[MIST_T_D_LAST_CK]);
  x = (float)stable;
  d = (float)delta;
}

// Memory model (:2150-2162, 2358-2385, 2755-2786).  `t` may also be the term-wise minimum of a
// stage: every operation is monotone in every term, so the peaks of that pseudo row bound the
// peaks of each row of the stage from below.
template <class Row>
__device__ __forceinline__ LaneMemory pair_memory(const Row &t, const PairConsts &k) {
  LaneMemory mem;
  const double S_ck = t[MIST_T_S_CK], S_nock = t[MIST_T_S_NOCK];
  mem.fwd_states = t[MIST_T_FWD_STATES0] + k.lf * t[MIST_T_PWG] + k.lm1 * t[MIST_T_PO];
  mem.bwd_states = t[MIST_T_BWD_STATES0] + k.lf * t[MIST_T_PWGO];
  mem.cur_saved = k.all_ck ? (k.lf - 1.0) * S_ck : k.cf * S_ck + k.l_minus_c_1 * S_nock;
  mem.mod_saved = S_ck * k.cf + S_nock * k.l_minus_c;
  mem.ck_delta = k.ck_tail ? t[MIST_T_D_CK] : t[MIST_T_D_NOCK];
  mem.fwd_pk = t[MIST_T_FWD_PEAK];
  mem.bwd_pk = t[MIST_T_BWD_PEAK];
  mem.out = t[MIST_T_OUT];
  mem.gcb = t[MIST_T_GCB];
  mem.mf_base = t[MIST_T_MF_BASE];
  mem.mf_pp = t[MIST_T_MF_PP];
  return mem;
}

// Upper bound of the number of feasible p in [0, n): both peaks are a value at p = 0 plus p times the
// same step, so what p admits is a quotient.  Rounding moves a scaled peak by a few 1e-16 of itself,
// at most 1e-15 of the capacity while it fits, hence the quotient by less than 1e-5 where a step
// counts for more than 1e-9 of the capacity; the quotient is taken 1e-4 and 0.01 long.  (`m0`, the
// scaled peak at p = 0, is the reference's value.)
__device__ __forceinline__ int count_upper(double m0, double step, int n, double cap) {
  if (n <= 0 || !(m0 <= cap)) return 0;
  if (!(step > 1e-9 * cap)) return n;
  const float most = (float)(cap - m0) * __builtin_amdgcn_rcpf((float)step) * 1.0001f + 0.01f;
  return most < (float)(n - 1) ? (int)most + 1 : n;
}
// The number itself: from the bound down to the last p the exact test admits.
template <class Scaled>
__device__ __forceinline__ int count_exact(const Scaled &scaled, int count, double cap) {
  while (count > 0 && !(scaled(count - 1) <= cap)) --count;
  return count;
}

// Constants of a group, of one sample.
struct GroupModel {
  GroupConsts k;
  double cap, G64, inv_G64;
  float G32, inv_G32;
  double pre_saved, pre_sas, pre_states, post_states, post_fwd_peak, post_bwd_peak, post_output;
  bool pow2;  // x / G == x * (1 / G) bit for bit, and the division leaves the inner loop

  __device__ __forceinline__ double div_G(double v) const { return pow2 ? v * inv_G64 : v / G64; }
  __device__ __forceinline__ float div_G(float v) const { return pow2 ? v * inv_G32 : v / G32; }

  // At most d / G, and r * lower_x(x) + lower_share(d) at most the base objective of a row, by the
  // slacks.  Monotone in x and d, so that of a stage's pseudo row bounds its rows' from below.
  __device__ __forceinline__ double lower_share(float d) const {
    return (double)d * inv_G64 * (d < 0.0f ? 1.0 + kShareSlack : 1.0 - kShareSlack);
  }
  // (|x|: nothing checks that a provider's extra share of a latency is no larger than the whole)
  __device__ __forceinline__ double lower_x(float x) const {
    return (double)x - kSlack * fabs((double)x);
  }
  __device__ __forceinline__ double bound(double ratio, float x, float d) const {
    return ratio * lower_x(x) + lower_share(d);
  }
};
__device__ __forceinline__ GroupModel group_model(const MistProblem &prob, const MistGroupDesc *g) {
  GroupModel m;
  m.k = group_consts(g);
  m.cap = prob.mem_cap_mb;
  m.G64 = (double)g->grad_accum;
  m.G32 = (float)g->grad_accum;
  m.inv_G64 = 1.0 / m.G64;
  m.inv_G32 = 1.0f / m.G32;
  m.pre_saved = g->pre_saved;
  m.pre_sas = g->pre_states_and_saved;
  m.pre_states = g->pre_states;
  m.post_states = g->post_states;
  m.post_fwd_peak = g->post_fwd_peak;
  m.post_bwd_peak = g->post_bwd_peak;
  m.post_output = g->post_output;
  m.pow2 = (g->grad_accum & (g->grad_accum - 1)) == 0;
  return m;
}

// count_upper of the base and with_pre variants.
struct UpperCounts {
  int b, p;
};
__device__ __forceinline__ UpperCounts upper_counts(const LaneMemory &mem, const GroupModel &m, int n) {
  double peak_f, peak_b;
  mem.peaks(0, peak_f, peak_b);
  const double peak = fmax(peak_f, peak_b), step = mem.mod_saved + 2.0 * mem.out;
  return UpperCounts{count_upper(peak * mem.mf_base, step * mem.mf_base, n, m.cap),
                     count_upper((peak + m.pre_sas) * mem.mf_pp, (step + m.pre_saved) * mem.mf_pp, n, m.cap)};
}
struct RowCounts {
  int b, p;
};
__device__ __forceinline__ RowCounts exact_counts(const LaneMemory &mem, const GroupModel &m, int upper_b, int upper_p) {
  return RowCounts{
      count_exact([&](int p) { return mem.scaled_base(p); }, upper_b, m.cap),
      count_exact([&](int p) { return mem.scaled_pre(p, m.pre_saved, m.pre_sas); }, upper_p, m.cap)};
}

// Stage costs the caller's search can use at all (MistProblem.stage_cost_incumbent): rows above
// it are not looked for.  (The seed launch reads the first estimate, which a few rows gave
// before it; the later launches read the one the seeds gave.)
__device__ __forceinline__ double stage_cost_cutoff(const MistProblem &prob, double inv_G64) {
  return prob.stage_cost_incumbent == nullptr || prob.sample_size != 1 || prob.incumbent_close == kCloseAssignment
             ? (double)INFINITY
             : *prob.stage_cost_incumbent * inv_G64 * (1.0 + kIncumbentSlack);
}

// The same with what form_reach knows of the group: rows above `cutoff` are not looked for, nor any of a
// stage of fewer than `first` layers whose minimum is below `low`.
struct CostLimits {
  double cutoff, low;
  int first;
  __device__ __forceinline__ double closed_below(int layers) const { return layers < first ? low : -INFINITY; }
};
__device__ __forceinline__ CostLimits cost_limits(const MistProblem &prob, const ReduceTables &tabs, int group, double inv_G64) {
  if (prob.incumbent_close != kCloseSearch) return CostLimits{stage_cost_cutoff(prob, inv_G64), -INFINITY, 0};
  const GroupReach &r = tabs.reach[group];
  return CostLimits{r.cutoff, r.low, r.first};
}
// Whether a pair of that many layers is in an assignment that assignment_reach_kernel leaves.
__device__ __forceinline__ bool in_assignments(const MistProblem &prob, const ReduceTables &tabs, int group, int layers) {
  return prob.incumbent_close != kCloseAssignment || (layers >= tabs.reach[group].first && layers <= tabs.reach[group].last);
}
// A minimum as a threshold.
__device__ __forceinline__ double up_to(double minimum, double cutoff, double closed_below) {
  return minimum < closed_below ? -INFINITY : fmin(minimum, cutoff);
}

// Group-wide terms the composite objectives add to the base latency: with x, d the
// float32-rounded stable / delta latency,
//   with_pre  = r (x + pre_fwd + pre_bwd + w1 + w2) + (d + w1d + w2d) / G
//   with_post = r (x + post_fwd + [row terms >= 0]) + (d + [row terms >= 0]) / G
//   no_pp     = r (x + pre_fwd + pre_bwd + post_fwd + [..] + w1 + w2 + [..]) + (d + w1d + w2d + [..]) / G
// so each is at least r x + d / G plus the offset below, up to a few roundings of relative size
// 1e-16 of the operands (the added terms are not negative).  A row can reach a minimum `t` of such an
// objective only if GroupModel::bound <= t - offset: the bound is short by the slacks of r x and
// d / G, the offsets are taken 1e-9 short, so every operand has room for its roundings a million
// times over, and it is far less than anything that matters for pruning.  The row terms of the
// last two have their own minima over a stage (MIST_T_OPB, the NAG and NRS pairs).
struct Offsets {
  double pre, post, pp;
};
// what is the same for the whole group ...
__device__ __forceinline__ Offsets group_offsets(const GroupModel &m, double ratio) {
  const GroupConsts &k = m.k;
  const double shared = m.div_G(k.w1d + k.w2d);
  Offsets o;
  o.pre = (ratio * (k.pre_fwd + k.pre_bwd + k.w1 + k.w2) + shared) * (1.0 - kSlack);
  o.post = ratio * k.post_fwd * (1.0 - kSlack);
  o.pp = (ratio * (k.pre_fwd + k.pre_bwd + k.post_fwd + k.w1 + k.w2) + shared) * (1.0 - kSlack);
  return o;
}
// ... and what the minima of a stage summary's post-layer terms add to the last two
__device__ __forceinline__ double post_layer_offset(const GroupModel &m, double ratio, const double *__restrict__ floor) {
  const GroupConsts &k = m.k;
  const double opb = floor[kStageMinOpb], nag = floor[kStageMinNag], nrs = floor[kStageMinNrs];
  return (ratio * (opb + (k.pp_wre ? nag : 0.0) + (k.pp_gre ? nrs : 0.0)) +
          m.div_G((k.pp_wre ? 0.0 : nag) + (k.pp_gre ? 0.0 : nrs))) * (1.0 - kSlack);
}

// The last-stage / single-stage memory tests, p == 0 only (:2946-3106); `smallest_out`: what the
// backward peak may lose (the row's output; for a stage summary its largest).
template <class Row>
__device__ __forceinline__ void post_fits(const Row &t, const PairConsts &k, const LaneMemory &mem,
                                          const GroupModel &m, double out, double rd, bool &post, bool &pp) {
  double peak_f, peak_b;
  mem.peaks(0, peak_f, peak_b);
  const double f_in = mem.fwd_states + m.post_states + mem.mod_saved + m.post_fwd_peak + mem.gcb;
  const double b_in = mem.bwd_states + m.post_states + mem.mod_saved + m.post_bwd_peak + rd + mem.gcb;
  const double pf_post = fmax(f_in, peak_f + m.post_states);
  const double pb_post = fmax(b_in, peak_b - out + m.post_states) + m.post_output;
  post = fmax(pf_post, pb_post) * mem.mf_pp <= m.cap;
  const double pf_pp = pf_post + m.pre_states + m.pre_saved;
  const double pb_pp = pb_post + m.pre_states + m.pre_saved;
  pp = fmax(pf_pp, pb_pp) * t[MIST_T_MF] <= m.cap;
}

// The four objectives of one row (pareto.py:138; base with y = float32 delta / G in float32,
// :2815, the others in float64, :2898-2903, 3002-3007, 3084-3089).
struct Objectives {
  double base, pre, post, pp;
};
template <class Row>
__device__ __forceinline__ Objectives objectives(const Row &t, float x32, float d32, bool no_ck, double ratio,
                                                 const GroupModel &m, bool with_post) {
  const GroupConsts &k = m.k;
  const double x = (double)x32, d = (double)d32;
  Objectives o;
  o.base = ratio * x + (double)m.div_G(d32);
  o.pre = ratio * (x + k.pre_fwd + k.pre_bwd + k.w1 + k.w2) + m.div_G(d + k.w1d + k.w2d);
  o.post = o.pp = INFINITY;
  if (with_post) {
    const double nag = no_ck ? t[MIST_T_NAG_NOCK] : t[MIST_T_NAG_CK];
    const double nrs = no_ck ? t[MIST_T_NRS_NOCK] : t[MIST_T_NRS_CK];
    const double ps1 = k.pp_wre ? nag : 0.0, ps2 = k.pp_gre ? nrs : 0.0;
    const double pd1 = k.pp_wre ? 0.0 : nag, pd2 = k.pp_gre ? 0.0 : nrs;
    const double opb = t[MIST_T_OPB];
    o.post = ratio * (x + k.post_fwd + opb + ps1 + ps2) + m.div_G(d + pd1 + pd2);
    o.pp = ratio * (x + k.pre_fwd + k.pre_bwd + k.post_fwd + opb + k.w1 + k.w2 + ps1 + ps2) +
           m.div_G(d + k.w1d + k.w2d + pd1 + pd2);
  }
  return o;
}

// One candidate row in registers.
struct RowRegs {
  double v[MIST_ROW_TERMS];
  __device__ __forceinline__ double operator[](int i) const { return v[i]; }
};
template <int kFrom, int kTo>  // columns, even
__device__ __forceinline__ void load_terms(RowRegs &r, const double *__restrict__ row) {
  static_assert(kFrom % 2 == 0 && kTo % 2 == 0, "rows are read as 16-byte pairs");
  const double2 *__restrict__ src = reinterpret_cast<const double2 *>(row);
#pragma unroll
  for (int i = kFrom / 2; i < kTo / 2; ++i) {
    const double2 v = src[i];
    r.v[2 * i] = v.x;
    r.v[2 * i + 1] = v.y;
  }
}
static_assert(MIST_T_S_LAYER_CK == 0 && MIST_T_D_LAST_NOCK == 11 && MIST_T_GCB < 32,
              "latency terms, then memory terms, are the first columns");

// A row's part of GroupModel::bound as a linear form of a pair's layer counts, unrounded: 0.2 ppm of
// every operand short, so that float32 rounding of x (6e-8 of the operands, with what the sums and
// products lose) and of d / G (twice that) leave it below every objective of the row.
// (values in, not references to members: a choice between those would put the struct into memory)
__device__ __forceinline__ double choose(bool first, double a, double b) { return first ? a : b; }
struct LinearBound {
  double ck, nock;          // per checkpointed / other layer
  double all_ck, none, mid; // first and last layer of a stage with c == l, c == 0, other c
  __device__ __forceinline__ double at(double n_ck, double n_nock, bool is_all, bool is_none) const {
    return __builtin_fma(n_ck, ck, __builtin_fma(n_nock, nock, choose(is_all, all_ck, choose(is_none, none, mid))));
  }
};
constexpr double kLinearSlack = 2e-7;
template <class Term>
__device__ __forceinline__ LinearBound linear_form(const Term &term) {
  const double first_ck = term(MIST_T_S_FIRST_CK, MIST_T_D_FIRST_CK), last_ck = term(MIST_T_S_LAST_CK, MIST_T_D_LAST_CK);
  const double first_nock = term(MIST_T_S_FIRST_NOCK, MIST_T_D_FIRST_NOCK);
  LinearBound b;
  b.ck = term(MIST_T_S_LAYER_CK, MIST_T_D_LAYER_CK);
  b.nock = term(MIST_T_S_LAYER_NOCK, MIST_T_D_LAYER_NOCK);
  // (1e-40: float32 values below the normal range are rounded by up to 1e-45)
  b.all_ck = first_ck + last_ck - 1e-40;
  b.none = first_nock + term(MIST_T_S_LAST_NOCK, MIST_T_D_LAST_NOCK) - 1e-40;
  b.mid = first_nock + last_ck - 1e-40;
  return b;
}
__device__ __forceinline__ double less_slack(double v) { return __builtin_fma(-kLinearSlack, fabs(v), v); }
__device__ __forceinline__ LinearBound linear_bound(const RowRegs &t, double ratio, double inv_G) {
  return linear_form([&](int stable, int delta) { return less_slack(ratio * t[stable]) + less_slack(t[delta] * inv_G); });
}

// The scaled peaks at p = 0 and their steps in another order of operations than pair_memory (a few
// 1e-16 off), for bounds of the counts: 1e-12 of the capacity of room covers that for every step, the
// quotient is taken 1e-4 and 0.01 long as in count_upper.
struct LinearMemory {
  double fwd, bwd, pwg, po, pwgo, s_ck, s_nock, d_ck, d_nock, out2, mf_base, mf_pp;
};
__device__ __forceinline__ LinearMemory linear_memory(const RowRegs &t) {
  LinearMemory r;
  r.out2 = 2.0 * t[MIST_T_OUT];
  r.fwd = t[MIST_T_FWD_STATES0] + t[MIST_T_FWD_PEAK] + t[MIST_T_GCB];
  r.bwd = t[MIST_T_BWD_STATES0] + t[MIST_T_BWD_PEAK] + t[MIST_T_GCB] + r.out2;
  r.pwg = t[MIST_T_PWG];
  r.po = t[MIST_T_PO];
  r.pwgo = t[MIST_T_PWGO];
  r.s_ck = t[MIST_T_S_CK];
  r.s_nock = t[MIST_T_S_NOCK];
  r.d_ck = t[MIST_T_D_CK];
  r.d_nock = t[MIST_T_D_NOCK];
  r.mf_base = t[MIST_T_MF_BASE];
  r.mf_pp = t[MIST_T_MF_PP];
  return r;
}
__device__ __forceinline__ int count_bound(double m0, double step, int n, double cap_and_room) {
  const double room = cap_and_room - m0;
  const float most = __builtin_fmaf((float)room * __builtin_amdgcn_rcpf((float)step), 1.0001f, 0.01f);
  const int count = most < (float)(n - 1) ? (int)most + 1 : n;  // (a step of 0: infinite, or not a number)
  return room >= 0.0 ? count : 0;
}
// A pair's constants for them; wave-uniform.
struct LinearPair {
  int l, c;
  bool all_ck, none;
  double n_ck, n_nock;
  __device__ __forceinline__ LinearPair(int layers, int ckpt) : l(layers), c(ckpt), all_ck(ckpt == layers), none(ckpt == 0) {
    const int lm2 = max(l - 2, 0), ck = min(max(c - 1, 0), lm2);
    n_ck = (double)ck;
    n_nock = (double)(lm2 - ck);
  }
};
// What they give of a row and a pair: bounds of the counts of base and with_pre, and the larger sums of
// post_fits without the states of the post layer.
struct LinearReach {
  int count_b, count_p;
  double post;
};
__device__ __forceinline__ LinearReach linear_reach(const LinearMemory &mem, const LinearPair &p, const GroupModel &m,
                                                    int np, double cap_and_room) {
  const double lf = (double)p.l, lm1 = (double)(p.l - 1);
  double saved_now = lm1 * mem.s_ck, next = mem.s_ck, ck_delta = mem.d_ck;
  if (!p.all_ck) {
    saved_now = __builtin_fma((double)p.c, mem.s_ck, (double)(p.l - p.c - 1) * mem.s_nock);
    next = mem.s_nock;
  }
  if (p.c < p.l - 1) ck_delta = mem.d_nock;
  const double shared = saved_now + ck_delta, step = saved_now + next + mem.out2;
  const double fwd = __builtin_fma(lf, mem.pwg, __builtin_fma(lm1, mem.po, mem.fwd));
  const double bwd = __builtin_fma(lf, mem.pwgo, mem.bwd), peak = shared + fmax(fwd, bwd);
  LinearReach r;
  r.count_b = count_bound(peak * mem.mf_base, step * mem.mf_base, np, cap_and_room);
  r.count_p = count_bound((peak + m.pre_sas) * mem.mf_pp, (step + m.pre_saved) * mem.mf_pp, np, cap_and_room);
  r.post = shared + fmax(fwd, bwd - 0.5 * mem.out2 + m.post_output);
  return r;
}
// Whether with_post or, in a pair of all layers, no_pp may fit (the latter's factor is the smaller one, MIST_T_MF).
__device__ __forceinline__ bool post_may_fit(const LinearReach &r, const LinearMemory &mem, const LinearPair &p, int num_layers,
                                             const GroupModel &m, double cap_and_room) {
  const double factor = p.l == num_layers ? mem.mf_pp - (0.025 + 1e-9) : mem.mf_pp;
  return (r.post + m.post_states) * factor <= cap_and_room;
}

// The largest minimum of every variant of a lane's pair: a row above all of them changes nothing
// (the minima do not decrease with p; +inf while a slot is empty).
struct Loosest {
  double base, pre, post, pp;
};
// (`slots`: the pair's slots of one sample, `pitch` apart; a pair that is not `wanted` reads none)
__device__ __forceinline__ Loosest loosest_minima(bool wanted, const double *slots, int pitch, int P, int count_b,
                                                  int count_p, bool do_post, bool do_pp, double cutoff,
                                                  double closed_below = -INFINITY) {
  Loosest t{-INFINITY, -INFINITY, -INFINITY, -INFINITY};
  if (!wanted) return t;
  const double base = slots[max(count_b - 1, 0) * pitch], pre = slots[(P + max(count_p - 1, 0)) * pitch];
  const double post = slots[2 * P * pitch], pp = slots[(2 * P + 1) * pitch];
  if (count_b > 0) t.base = up_to(base, cutoff, closed_below);
  if (count_p > 0) t.pre = up_to(pre, cutoff, closed_below);
  if (do_post) t.post = up_to(post, cutoff, closed_below);
  if (do_pp) t.pp = up_to(pp, cutoff, closed_below);
  return t;
}
// One threshold for GroupModel::bound that every row which could reach one of them passes: in two
// parts, from the offsets of the group and with what a stage's post-layer terms add to the second.
struct Threshold {
  double front, post;  // base and with_pre; with_post and no_pp
  __device__ __forceinline__ Threshold(double its_front, double its_post) : front(its_front), post(its_post) {}
  __device__ __forceinline__ Threshold(const Loosest &t, const Offsets &group)
      : front(fmax(t.base, t.pre - group.pre)), post(fmax(t.post - group.post, t.pp - group.pp)) {}
  __device__ __forceinline__ double at(double post_layer) const { return fmax(front, post - post_layer); }
};

// ---- seeds ----
__device__ __forceinline__ void clear_queue(const ReduceTables &tabs) {
  if (blockIdx.x == 0 && blockIdx.y == 0)
    for (int i = threadIdx.x; i < kCounters; i += blockDim.x)
      tabs.counter[i * kCounterPitch] = tabs.counter[i * kCounterPitch + kOpenPairs] = 0;
}

// Smallest linear bounds of 64 gathered rows at a time, for the seed launch: workgroup `part` of
// `n_parts` of a group, a wavefront per 64 rows.
__device__ __forceinline__ void gather_floors(const MistProblem &prob, const MistGroupDesc *__restrict__ g, int gi,
                                              const double *__restrict__ row_terms, double ratio, double *gather_floor,
                                              int part, int n_parts) {
  if (g->scout_stride <= 0) return;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int waves = (int)blockDim.x / 64, n_gather = g->n_par * g->n_oo * g->n_ao * g->scout_stride;
  const double inv_G = 1.0 / (double)g->grad_accum;
  const double *__restrict__ src = row_terms + g->row_offset * MIST_ROW_TERMS;
  for (int stage = part * waves + wave; stage < (n_gather + 63) / 64; stage += n_parts * waves) {
    RowRegs t;
    load_terms<0, MIST_T_D_LAST_NOCK + 1>(
        t, src + gathered_position(g, (uint32_t)min(stage * 64 + lane, n_gather - 1)) * MIST_ROW_TERMS);
    const LinearBound b = linear_bound(t, ratio, inv_G);
    double low[kGatherFloor] = {b.ck, b.nock, b.all_ck, b.none, b.mid}, mine = 0.0;
#pragma unroll
    for (int i = 0; i < kGatherFloor; ++i) {
      for (int step = 1; step < 64; step <<= 1) low[i] = fmin(low[i], __shfl_xor(low[i], step));
      if (lane == i) mine = low[i];
    }
    if (lane < kGatherFloor) gather_floor[stage_floor_slot(g, gi, stage) * kGatherFloor + lane] = mine;
  }
}
constexpr int kGatherBlocks = 16;  // workgroups per group
__global__ __launch_bounds__(256) void gather_floor_kernel(const MistProblem prob, const MistGroupDesc *__restrict__ groups,
                                                           const double *__restrict__ row_terms, double ratio,
                                                           double *gather_floor) {
  gather_floors(prob, groups + blockIdx.y, blockIdx.y, row_terms, ratio, gather_floor, blockIdx.x, gridDim.x);
}

// Layers from which on a pair of the group may be in a pipeline below the limit, by about what form_reach will say,
// from the first estimate alone (the summaries are not there yet).  The pairs below are closed mostly, once their
// minimum is below about kLikelyLow of the cutoff: what is wrong about that only leaves them higher minima.  (Of the
// cutoff 0.7 / 0.8 / 0.88 / 0.95 / 1: 70B on 32x8 4147 / 4077 / 4059 / 4135 / 4229 us a search, 22B on 16x8 6351 / 6350
// / 6349 / 6531 / 6675, 13B on 8x8 1526 / 1518 / 1514 / 1502 / 1506, 7B on 4x8 1141 / 1135 / 1125 / 1113 / 1110.  The 5 %
// more layers that the other devices are taken to hold count for little: 0 / 5 / 10 / 20 % 70B 4068 / 4059 / 4062 / 4075,
// 22B 6341 / 6349 / 6354 / 6371, 13B 1512 / 1514 / 1510 / 1528, runs of one side differing by 20.)
constexpr double kLikelyLow = 0.88;
__device__ __forceinline__ int likely_first(const MistProblem &prob, const MistGroupDesc *g, double cutoff) {
  if (prob.incumbent_close != kCloseSearch || !(cutoff < INFINITY)) return 0;
  const float L = (float)prob.num_layers, D = (float)prob.incumbent_num_devices;
  return (int)(L - 1.05f * L * (D - (float)(g->num_nodes * g->num_gpus_per_node)) / D);
}
// First minima of such pairs, for which any row below what closes them does: a few rows of every kind, thread = (row,
// pair), leave their cost at their own count, then every slot takes the ones above.  The pairs that leaves open
// go on with all gathered rows.  (Nothing is gained where pairs are left at that: 22B on 16x8 6510 -> 6740 us, with 4
// instead of 10 ratios 7920; nor by closing alone, the time goes into the first rows of a pair.  With both: 22B
// 6483 -> 6158, 70B on 32x8 3890 -> 3719, 13B on 8x8 1599 -> 1541, 7B on 4x8 1051 -> 1030, drawn calls 1.1 %.)
constexpr int kLightTails = 10;  // (activation, optimizer) offload ratios of each parallelism row and offload pair
__device__ __forceinline__ void light_seeds(const MistProblem &prob, const MistGroupDesc *__restrict__ g,
                                            const double *__restrict__ src, double ratio, double cutoff, int first_pair,
                                            int n_here, int pair_split, double *lds_best) {
  const int L = prob.num_layers, P = g->num_p, n_slots = slots_of(P);
  const int pair = threadIdx.x % pair_split, n_tail = g->n_oo * g->n_ao;
  const int tails = min(kLightTails, n_tail), n_rows = g->n_par * tails * g->scout_stride;
  const GroupModel m = group_model(prob, g);
  const PairIndex pc = decode_pair(first_pair + min(pair, n_here - 1));
  const PairConsts k = pair_consts(pc.l, pc.c);
  const int np = pc.c == pc.l - 1 ? min(P, 1) : P;
  const bool do_post = pc.c != pc.l - 1, do_pp = do_post && pc.l == L;
  double *mine = lds_best + pair * n_slots;
  for (int r = threadIdx.x / pair_split; pair < n_here && r < n_rows; r += kSeedThreads / pair_split) {
    const int tail = tails > 1 ? r % tails * (n_tail - 1) / (tails - 1) : 0, par = r / tails % g->n_par, which = r / tails / g->n_par;
    const int q = (which * g->n_par + par) * n_tail + tail;
    RowRegs t;
    load_terms<0, MIST_ROW_TERMS>(t, src + gathered_position(g, (uint32_t)q) * MIST_ROW_TERMS);
    float x, d;
    pair_latency(t, k, x, d);
    const LaneMemory mem = pair_memory(t, k);
    const Objectives o = objectives(t, x, d, k.no_ck, ratio, m, do_post);
    const UpperCounts upper = upper_counts(mem, m, np);
    const RowCounts cnt = exact_counts(mem, m, upper.b, upper.p);
    bool ok_post = false, ok_pp = false;
    if (do_post) post_fits(t, k, mem, m, mem.out, k.no_ck ? t[MIST_T_RD] : 0.0, ok_post, ok_pp);
    auto offer = [&](bool ok, double cost, double *slot) {
      if (ok && cost <= cutoff) lower_minimum_in_lds(slot, cost);
    };
    offer(cnt.b > 0, o.base, mine + max(cnt.b - 1, 0));
    offer(cnt.p > 0, o.pre, mine + P + max(cnt.p - 1, 0));
    offer(ok_post, o.post, mine + 2 * P);
    offer(do_pp && ok_pp, o.pp, mine + 2 * P + 1);
  }
  __syncthreads();
  if ((int)threadIdx.x < 2 * pair_split) {
    double *slots = lds_best + threadIdx.x / 2 * n_slots + (threadIdx.x & 1) * P;
    double low = INFINITY;
    for (int p = P - 1; p >= 0; --p) {
      low = fmin(low, slots[p]);
      slots[p] = low;
    }
  }
}

// One sample.  Workgroup = (`pair_split` consecutive pairs of a tile, group) with their minima in
// LDS.  A wavefront takes 64 gathered rows: lane = pair, the smallest of their linear bounds against the
// pair's loosest minima and the cutoff (of 22B on 16x8's 582000 times 16 pairs 86000 have one left, 0.9e6
// pairs in all); then lane = row over those: the row's own bound, bounds of its counts against the minima
// there, the reference's arithmetic.  Of the rows below the minimum at their
// own count the cheapest lowers the slots up to its count (lane = slot) and drops the rows it
// dominates, until none is left - a few steps from empty minima, none later.
// (One LDS atomic per row at its own count, all rows of a stage at a few addresses: 0.96 ms for
// the 7B plan; the register minima this replaced, one row after the other per lane: 0.42 ms; the
// reference's latencies for every row and pair and its memory model below the cutoff, every row loaded
// for every 16 pairs: 22B on 16x8 7.5e8 wave instructions, 5.7 ms beside the summaries, 70B on 32x8 1.95 ms; now
// 2.4e8, 4.7 and 1.25.)
__global__ __launch_bounds__(kSeedThreads, 3) void seed_kernel(
    const MistProblem prob, const MistGroupDesc *__restrict__ groups, const double *__restrict__ row_terms,
    double ratio, ReduceTables tabs, int pair_split) {
  extern __shared__ double lds_best[];
  const MistGroupDesc *g = groups + blockIdx.y;
  const int parts = MIST_LC_TILE / pair_split;
  const int tile_rel = (int)blockIdx.x / parts, part = (int)blockIdx.x % parts;
  clear_queue(tabs);
  if (tile_rel >= g->n_lc_tiles) return;
  const int L = prob.num_layers, n_pairs = L * (L + 1) / 2 + L;
  const int P = g->num_p, n_slots = slots_of(P);
  const int first_pair = (g->lc_tile_begin + tile_rel) * MIST_LC_TILE + part * pair_split;
  const int n_here = min(pair_split, n_pairs - first_pair);
  const int n_entries = pair_split * n_slots;  // [pair][slot]
  for (int e = threadIdx.x; e < n_entries; e += kSeedThreads) lds_best[e] = INFINITY;
  __syncthreads();
  const double most = stage_cost_cutoff(prob, 1.0 / (double)g->grad_accum);
  const int likely = likely_first(prob, g, most);
  if (g->scout_stride > 0 && n_here > 0 && decode_pair(first_pair).l < likely) {
    light_seeds(prob, g, row_terms + g->row_offset * MIST_ROW_TERMS, ratio, most, first_pair, n_here, pair_split, lds_best);
    __syncthreads();
  }
  if (g->scout_stride > 0 && n_here > 0) {
    constexpr int kWaves = kSeedThreads / 64;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const GroupModel m = group_model(prob, g);
    const Offsets group = group_offsets(m, ratio);
    const double cutoff = most, cap_and_room = m.cap * (1.0 + 1e-12);
    const int n_gather = g->n_par * g->n_oo * g->n_ao * g->scout_stride;
    const int n_stages = (n_gather + 63) / 64;
    // units of work: (stage, share of the pairs), more than one share when there are few stages
    const int shares = max(1, min(n_here, kWaves / n_stages)), per_share = (n_here + shares - 1) / shares;
    const double *__restrict__ src = row_terms + g->row_offset * MIST_ROW_TERMS;
    // lane = pair of the workgroup
    const int my_pair = min(lane, n_here - 1);
    const PairIndex pc = decode_pair(first_pair + my_pair);
    const int lc = pc.l | pc.c << 15, my_np = pc.c == pc.l - 1 ? min(P, 1) : P;
    const LinearPair my_lp(pc.l, pc.c);
    const double closed_below = pc.l < likely ? kLikelyLow * cutoff : -INFINITY;
    const int64_t floor_slot = stage_floor_slot(g, blockIdx.y, 0);
    for (int unit = wave; unit < n_stages * shares; unit += kWaves) {
      const int q = unit / shares * 64 + lane;
      const int i0 = unit % shares * per_share, i1 = min(i0 + per_share, n_here);
      const bool live = q < n_gather;
      // what a row has to reach of the lane's pair (they fall while the loop runs), against the rows' bounds
      const bool its_post = pc.c != pc.l - 1;
      const double thr = Threshold(loosest_minima(true, lds_best + my_pair * n_slots, 1, P, my_np, my_np, its_post,
                                                  its_post && pc.l == L, cutoff, closed_below), group).at(0.0);
      const double *__restrict__ f = tabs.gather_floor + (floor_slot + unit / shares) * kGatherFloor;
      const LinearBound floor{f[0], f[1], f[2], f[3], f[4]};
      uint64_t open = __ballot(lane >= i0 && lane < i1 &&
                               floor.at(my_lp.n_ck, my_lp.n_nock, my_lp.all_ck, my_lp.none) <= thr);
      if (open == 0) continue;
      const double *__restrict__ my_row = src + gathered_position(g, (uint32_t)min(q, n_gather - 1)) * MIST_ROW_TERMS;
      RowRegs t;
      load_terms<0, MIST_T_D_LAST_NOCK + 1>(t, my_row);
      const LinearBound bound = linear_bound(t, ratio, m.inv_G64);
      LinearMemory memory = {};
      bool have_rest = false;
      for (; open != 0; open &= open - 1) {
        const int i = __ffsll((unsigned long long)open) - 1;
        const int its = from_lane(lc, i), l = its & 0x7fff, c = its >> 15;
        const LinearPair p(l, c);
        const double low = bound.at(p.n_ck, p.n_nock, p.all_ck, p.none);
        const bool wanted = live && low <= from_lane(thr, i);
        if (!__any(wanted)) continue;
        if (!have_rest) {
          load_terms<MIST_T_D_LAST_NOCK + 1, MIST_ROW_TERMS>(t, my_row);
          memory = linear_memory(t);
          have_rest = true;
        }
        // Cells with c == l - 1 are only kept for p == 0 of the base / with_pre variants
        // (batched_module_analyzer.py:3021-3023, 3103).
        const int np = c == l - 1 ? min(P, 1) : P;
        const bool do_post = c != l - 1, do_pp = do_post && l == L;
        double *mine = lds_best + i * n_slots;
        // the minima do not decrease with p: at the bound of its count a row meets the largest one
        // it could beat
        const LinearReach reach = linear_reach(memory, p, m, np, cap_and_room);
        bool may = (reach.count_b > 0 && low < mine[max(reach.count_b - 1, 0)]) ||
                   (reach.count_p > 0 && low + group.pre < mine[P + max(reach.count_p - 1, 0)]);
        if (do_post) {
          const double post = do_pp ? fmax(mine[2 * P] - group.post, mine[2 * P + 1] - group.pp) : mine[2 * P] - group.post;
          may = may || (low < post && post_may_fit(reach, memory, p, L, m, cap_and_room));
        }
        may = may && wanted;
        if (!__any(may)) continue;
        const PairConsts k = pair_consts(l, c);
        float x, d;
        pair_latency(t, k, x, d);
        const LaneMemory mem = pair_memory(t, k);
        const Objectives o = objectives(t, x, d, k.no_ck, ratio, m, do_post);
        const UpperCounts upper = upper_counts(mem, m, may ? np : 0);
        const RowCounts cnt = exact_counts(mem, m, upper.b, upper.p);
        bool ok_post = false, ok_pp = false;
        if (do_post) post_fits(t, k, mem, m, mem.out, k.no_ck ? t[MIST_T_RD] : 0.0, ok_post, ok_pp);
        auto offer = [&](int count, double cost, double *slots) {
          bool pending = count > 0 && cost < slots[max(count - 1, 0)];
          while (__any(pending)) {
            const int r = cheapest_lane(pending, cost);
            const double its_cost = from_lane(cost, r);
            const int its_count = from_lane(count, r);
            for (int j = lane; j < its_count; j += 64) lower_minimum_in_lds(slots + j, its_cost);
            pending = pending && lane != r && (count > its_count || cost < its_cost);
          }
        };
        offer(cnt.b, o.base, mine);
        offer(cnt.p, o.pre, mine + P);
        if (do_post) offer(may && ok_post ? 1 : 0, o.post, mine + 2 * P);
        if (do_pp) offer(may && ok_pp ? 1 : 0, o.pp, mine + 2 * P + 1);
      }
    }
  }
  __syncthreads();
  // (pairs past the last one of the list belong to the tile: they stay empty)
  const int64_t cell0 = g->cell_offset + ((int64_t)tile_rel * MIST_LC_TILE + part * pair_split) * n_slots;
  for (int e = threadIdx.x; e < n_entries; e += kSeedThreads) {
    tabs.best[cell0 + e] = lds_best[e];
    tabs.row[cell0 + e] = ~0u;
  }
}

// No seeds (none asked for, or the minima of one pair exceed the LDS): the tables of the launch, empty.
__global__ __launch_bounds__(256) void empty_minima_kernel(ReduceTables tabs, int64_t cells) {
  clear_queue(tabs);
  const int64_t first = (int64_t)blockIdx.x * blockDim.x + threadIdx.x, step = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = first; i < cells * tabs.n_samples; i += step) {
    tabs.best[i] = INFINITY;
    tabs.row[i] = ~0u;
  }
}

// Several samples.  What the objectives of a row are made of, r X + Y per variant, and its counts,
// for the lane = (row parity, sample) phases: a wavefront reads two rows at a time.
struct SampleRows {
  double2 xy[4][64];    // base, with_pre, with_post, no_pp: (X, Y)
  uint32_t counts[64];  // feasible p: base | with_pre << 15 | with_post << 30 | no_pp << 31
  uint32_t number[64];  // row number
};
// (counts of two words cost 30 samples of 7B on 1x8 5 %; calls with more values of p take their
// samples one by one)
constexpr int kMostCountedP = 0x7fff;
static_assert(MIST_MAX_SAMPLE_BATCH <= 32, "half a wavefront per row");
// Writes row `at` of the buffer.
__device__ __forceinline__ void put_sample_row(SampleRows *rows, int at, const RowRegs &t, float x32, float d32, bool no_ck,
                                               const GroupModel &m, int count_b, int count_p, bool post, bool pp,
                                               bool do_post) {
  const GroupConsts &k = m.k;
  const double x = (double)x32, d = (double)d32;
  rows->xy[0][at] = double2{x, (double)m.div_G(d32)};
  rows->xy[1][at] = double2{x + k.pre_fwd + k.pre_bwd + k.w1 + k.w2, m.div_G(d + k.w1d + k.w2d)};
  if (do_post) {
    const double nag = no_ck ? t[MIST_T_NAG_NOCK] : t[MIST_T_NAG_CK];
    const double nrs = no_ck ? t[MIST_T_NRS_NOCK] : t[MIST_T_NRS_CK];
    const double ps1 = k.pp_wre ? nag : 0.0, ps2 = k.pp_gre ? nrs : 0.0;
    const double pd1 = k.pp_wre ? 0.0 : nag, pd2 = k.pp_gre ? 0.0 : nrs;
    const double opb = t[MIST_T_OPB];
    rows->xy[2][at] = double2{x + k.post_fwd + opb + ps1 + ps2, m.div_G(d + pd1 + pd2)};
    rows->xy[3][at] = double2{x + k.pre_fwd + k.pre_bwd + k.post_fwd + opb + k.w1 + k.w2 + ps1 + ps2,
                              m.div_G(d + k.w1d + k.w2d + pd1 + pd2)};
  }
  rows->counts[at] = (uint32_t)count_b | (uint32_t)count_p << 15 | (post ? 1u << 30 : 0u) | (pp ? 1u << 31 : 0u);
}

// Workgroup = one pair of a group with the minima of all its samples in LDS, a column per sample; its
// wavefronts take 64 gathered rows each: lane = row for their latencies and counts, then lane = (row
// parity, sample): one LDS minimum per (row, variant, sample) at the row's own count, conflict-free
// but for the rows in flight.  The minima per p are the suffix minima of those buckets, a range of p
// per wavefront.
// (30 samples one after the other through seed_kernel: 3.1 ms for the tables of one tensor-parallel
// size of the 7B plan.  One wavefront a pair: its minima leave room for four on a CU, 0.47 ms; now 0.33. 7B on
// 4x8 0.43 -> 0.38, on 1x8 0.096 -> 0.075; eight wavefronts 0.39, 0.43, 0.11.)
constexpr int kSeedSampleWaves = 4;
__global__ __launch_bounds__(64 * kSeedSampleWaves) void seed_samples_kernel(
    const MistProblem prob, const MistGroupDesc *__restrict__ groups, const double *__restrict__ row_terms,
    const RatioList ratios, ReduceTables tabs, int sample_split) {
  extern __shared__ double lds_best[];
  const MistGroupDesc *g = groups + blockIdx.y;
  clear_queue(tabs);
  const int tile_rel = (int)blockIdx.x / MIST_LC_TILE, lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), n_waves = blockDim.x >> 6;
  if (tile_rel >= g->n_lc_tiles) return;
  const int L = prob.num_layers, n_pairs = L * (L + 1) / 2 + L;
  const int P = g->num_p, n_slots = slots_of(P);
  const int first_sample = (int)blockIdx.z * sample_split, S = min(sample_split, tabs.n_samples - first_sample);
  const int pair = g->lc_tile_begin * MIST_LC_TILE + (int)blockIdx.x;
  SampleRows *rows = reinterpret_cast<SampleRows *>(lds_best) + wave;
  double *mine = lds_best + sizeof(SampleRows) / 8 * n_waves;  // [slot][sample]
  for (int e = threadIdx.x; e < n_slots * S; e += blockDim.x) mine[e] = INFINITY;
  __syncthreads();
  const int sample = lane & 31;
  if (g->scout_stride > 0 && pair < n_pairs && in_assignments(prob, tabs, blockIdx.y, decode_pair(pair).l)) {
    const GroupModel m = group_model(prob, g);
    const PairIndex pc = decode_pair(pair);
    const int l = __builtin_amdgcn_readfirstlane(pc.l), c = __builtin_amdgcn_readfirstlane(pc.c);
    const PairConsts k = pair_consts(l, c);
    const int np = c == l - 1 ? min(P, 1) : P;
    const bool do_post = c != l - 1, do_pp = do_post && l == L;
    const double ratio = ratios.r[first_sample + min(sample, S - 1)];
    const int n_gather = g->n_par * g->n_oo * g->n_ao * g->scout_stride;
    const double *__restrict__ src = row_terms + g->row_offset * MIST_ROW_TERMS;
    for (int q0 = wave * 64; q0 < n_gather; q0 += 64 * n_waves) {
      const int n_rows = min(64, n_gather - q0);
      RowRegs t;
      load_terms<0, MIST_ROW_TERMS>(t, src + gathered_position(g, (uint32_t)min(q0 + lane, n_gather - 1)) * MIST_ROW_TERMS);
      float x, d;
      pair_latency(t, k, x, d);
      const LaneMemory mem = pair_memory(t, k);
      const UpperCounts upper = upper_counts(mem, m, lane < n_rows ? np : 0);
      const RowCounts cnt = exact_counts(mem, m, upper.b, upper.p);
      bool ok_post = false, ok_pp = false;
      if (do_post) post_fits(t, k, mem, m, mem.out, k.no_ck ? t[MIST_T_RD] : 0.0, ok_post, ok_pp);
      ok_post = ok_post && lane < n_rows;
      ok_pp = ok_pp && do_pp && lane < n_rows;
      // (rows that fit nowhere are left out)
      const uint64_t useful = __ballot(cnt.b > 0 || cnt.p > 0 || ok_post || ok_pp);
      __builtin_amdgcn_wave_barrier();
      if (useful >> lane & 1ull)
        put_sample_row(rows, __popcll(useful & ((1ull << lane) - 1ull)), t, x, d, k.no_ck, m, cnt.b, cnt.p, ok_post,
                       ok_pp, do_post);
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
      const int n_useful = __popcll(useful);
      for (int r = lane >> 5; r < n_useful; r += 2) {
        const uint32_t counts = rows->counts[r];
        const int nb = (int)(counts & 0x7fff), npre = (int)(counts >> 15 & 0x7fff);
        auto offer = [&](bool ok, int variant, int slot) {
          const double2 xy = rows->xy[variant][r];
          const double cost = ratio * xy.x + xy.y;
          if (ok && sample < S && cost < INFINITY) lower_minimum_in_lds(mine + slot * S + sample, cost);
        };
        offer(nb > 0, 0, nb - 1);
        offer(npre > 0, 1, P + npre - 1);
        if (do_post) {
          offer((counts >> 30 & 1u) != 0, 2, 2 * P);
          if (do_pp) offer((counts >> 31) != 0, 3, 2 * P + 1);
        }
      }
    }
  }
  __syncthreads();
  const int64_t cell0 = g->cell_offset + (int64_t)blockIdx.x * n_slots;
  const int v = lane >> 5;  // base, with_pre
  const int first_p = P * wave / n_waves, end_p = P * (wave + 1) / n_waves;
  double low = INFINITY;
  if (sample < S)
    for (int j = end_p; j < P; ++j) low = fmin(low, mine[(v * P + j) * S + sample]);
  if (sample < S) {
    const int64_t at = cell0 * tabs.n_samples + first_sample + sample;
    auto put = [&](int slot, double value) {
      tabs.best[at + (int64_t)slot * tabs.n_samples] = value;
      tabs.row[at + (int64_t)slot * tabs.n_samples] = ~0u;
    };
    for (int j = end_p - 1; j >= first_p; --j) {
      low = fmin(low, mine[(v * P + j) * S + sample]);
      put(v * P + j, low);
    }
    if (wave == 0) put(2 * P + v, mine[(2 * P + v) * S + sample]);
  }
}

// ---- summaries of kSuperStages stages ----
__device__ __forceinline__ int64_t super_floor_slot(const MistGroupDesc *g, int group_index, int64_t super) {
  return stage_floor_slot(g, group_index, 0) / kSuperStages + group_index + super;
}
// With `close` a workgroup also leaves the smallest linear bounds of its summaries (GroupReach): of stage costs,
// for an assignment of stable latencies.
__global__ __launch_bounds__(256) void super_floor_kernel(const MistGroupDesc *__restrict__ groups, int n_groups,
                                                          const double *__restrict__ stage_floor, double ratio, int close,
                                                          const ReduceTables tabs) {
  const int gi = blockIdx.y;
  const MistGroupDesc *g = groups + gi;
  const int64_t n_stages = (g->n_rows + kStageRows - 1) / kStageRows;
  const int col = threadIdx.x % kStageFloorPitch;
  const int per_block = blockDim.x / kStageFloorPitch;
  const double inv_G = close == kCloseAssignment ? 0.0 : 1.0 / (double)g->grad_accum;
  double per_layer = INFINITY, rest = INFINITY;
  for (int64_t super = (int64_t)blockIdx.x * per_block + threadIdx.x / kStageFloorPitch;
       super * kSuperStages < n_stages; super += (int64_t)gridDim.x * per_block) {
    const double *__restrict__ src = stage_floor + (stage_floor_slot(g, gi, super * kSuperStages)) * kStageFloorPitch;
    const int n = (int)min((int64_t)kSuperStages, n_stages - super * kSuperStages);
    double v = src[col];
    for (int i = 1; i < n; ++i) {
      const double o = src[i * kStageFloorPitch + col];
      v = col == kStageMaxOut ? fmax(v, o) : fmin(v, o);
    }
    tabs.super_floor[super_floor_slot(g, gi, super) * kStageFloorPitch + col] = v;
    if (tabs.listed != nullptr && col < n) tabs.stage_flag[stage_floor_slot(g, gi, super * kSuperStages) + col] = 0;
    if (close == 0) continue;
    // (the columns of a summary lie in 32 neighbouring lanes; every lane forms the same bounds)
    const LinearBound b = linear_form([&](int stable, int delta) {
      return less_slack(ratio * __shfl(v, stable, kStageFloorPitch)) + less_slack(__shfl(v, delta, kStageFloorPitch) * inv_G);
    });
    per_layer = fmin(per_layer, fmin(b.ck, b.nock));
    rest = fmin(rest, fmin(b.all_ck, fmin(b.none, b.mid)));
  }
  if (close == 0) return;
  __shared__ double parts[256 / kStageFloorPitch][2];
  if (col == 0) {
    parts[threadIdx.x / kStageFloorPitch][0] = per_layer;
    parts[threadIdx.x / kStageFloorPitch][1] = rest;
  }
  __syncthreads();
  if (threadIdx.x >= 2) return;
  double least = INFINITY;
  for (int i = 0; i < per_block; ++i) least = fmin(least, parts[i][threadIdx.x]);
  tabs.reach_parts[((int64_t)gi * kSuperBlocks + blockIdx.x) * 2 + threadIdx.x] = least;
}

// Lane = pair against a stage summary: the counts its pseudo row allows, hence which minima a row
// of the stage can reach, and the bound that its objective gives.
struct StageReach {
  int count_b, count_p;  // base, with_pre
  bool post, pp;
  float x, d;            // of the pseudo row
};
__device__ __forceinline__ StageReach stage_reach(const double *__restrict__ f, const PairConsts &k, int np,
                                                  bool do_post, bool do_pp, const GroupModel &m) {
  StageReach r;
  pair_latency(f, k, r.x, r.d);
  const LaneMemory mem = pair_memory(f, k);
  const UpperCounts upper = upper_counts(mem, m, np);
  r.count_b = upper.b;
  r.count_p = upper.p;
  bool post, pp;
  post_fits(f, k, mem, m, f[kStageMaxOut], 0.0, post, pp);
  r.post = do_post && post;
  r.pp = do_pp && pp;
  return r;
}

// ---- filter ----
// Workgroup = one wavefront = (row chunk, tile, p tile as a share of the chunk's summaries), lane
// = pair.  A summary is the same for all lanes; a visit is ~40 float64 instructions against the pair's
// loosest minima.
// Several samples: kFilterShares wavefronts of a workgroup take as many shares of a tile and its thresholds
// at every sample from LDS, where they get them with lane = (pair parity, sample): the minima of a slot lie
// side by side.  A summary is tried at the sample that the last one passed first.  (A wavefront a share and
// its samples one after the other, a line per lane, slot and sample, kept the address units busy 84 % of the
// time: 30 samples of 7B on 4x8 0.55 ms; 0.33 with the thresholds from LDS, 0.16 with a summary's latency
// computed once for all samples.)
constexpr int kFilterShares = 4;
constexpr int kFilterPitch = MIST_LC_TILE + 1;  // doubles; front and post of a sample
template <bool kSamples>
__global__ __launch_bounds__(kSamples ? kFilterShares * 64 : 64) void filter_kernel(
    const MistProblem prob, const MistGroupDesc *__restrict__ groups, int n_groups,
    const int32_t *__restrict__ block_prefix, int n_blocks, const double *__restrict__ stage_floor,
    const double *__restrict__ super_floor, const RatioList ratios, ReduceTables tabs) {
  const int block = xcd_run_block(blockIdx.x);
  if (block >= n_blocks) return;
  int local_block;
  const MistGroupDesc *g = find_group(groups, block_prefix, n_groups, block, &local_block);
  const int gi = __builtin_amdgcn_readfirstlane((int)(g - groups));
  g = groups + gi;
  local_block = __builtin_amdgcn_readfirstlane(local_block);
  const int n_p = g->n_p_tiles, n_tiles = g->n_lc_tiles * n_p;
  const int chunk = local_block / n_tiles, tile = local_block % n_tiles;
  const int share = tile % n_p, tile_rel = tile / n_p;
  const int n_stages = (int)((g->n_rows + kStageRows - 1) / kStageRows);
  int stage0 = (int)((int64_t)chunk * g->rows_per_chunk / kStageRows);
  int stage1 = min(stage0 + g->rows_per_chunk / kStageRows, n_stages);
  int super_first = stage0 / kSuperStages + share, super_last = (stage1 - 1) / kSuperStages, stride = n_p;
  if (kSamples) {
    const int64_t mine = (int64_t)chunk * n_p + share;  // the workgroups of the other shares have nothing to do
    if (mine % kFilterShares != 0) return;
    const int64_t all = ((int64_t)g->n_chunks * n_p + kFilterShares - 1) / kFilterShares * kFilterShares;
    const int64_t at = mine + __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int64_t n_supers = (n_stages + kSuperStages - 1) / kSuperStages;
    super_first = (int)(n_supers * at / all);
    super_last = (int)(n_supers * (at + 1) / all) - 1;
    stride = 1;
    stage0 = 0;
    stage1 = n_stages;
  }

  const int L = prob.num_layers, n_pairs = L * (L + 1) / 2 + L, lane = threadIdx.x & 63;
  const int pair_idx = (g->lc_tile_begin + tile_rel) * MIST_LC_TILE + lane;
  const bool listed = pair_idx < n_pairs;
  const PairIndex pc = decode_pair(listed ? pair_idx : 0);
  const bool active = listed && (!kSamples || in_assignments(prob, tabs, gi, pc.l));
  if (kSamples && !__any(active)) return;  // (all wavefronts of the workgroup: one tile)
  const PairConsts k = pair_consts(pc.l, pc.c);
  const int P = g->num_p, S = tabs.n_samples;
  const int np = !active ? 0 : (pc.c == pc.l - 1 ? min(P, 1) : P);
  const bool do_post = active && pc.c != pc.l - 1, do_pp = do_post && pc.l == L;
  const GroupModel m = group_model(prob, g);
  const CostLimits limits = cost_limits(prob, tabs, gi, m.inv_G64);
  const double *best = tabs.best + (g->cell_offset + (int64_t)tile_rel * MIST_LC_TILE * slots_of(P)) * S;
  extern __shared__ double lds_thresholds[];  // [sample][front, post][pair]
  if (kSamples) {
    const int sample = min(lane & 31, S - 1), parts = np | (int)do_post << 30 | (int)((unsigned)do_pp << 31);
    const Offsets offsets = group_offsets(m, ratios.r[sample]);
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    constexpr int kPairs = MIST_LC_TILE / kFilterShares;
#pragma unroll
    for (int i = 0; i < kPairs; i += 2) {
      const int pair = wave * kPairs + i + (lane >> 5);
      const uint32_t its = (uint32_t)__shfl(parts, pair);
      const int n = (int)(its & 0x7fff);
      const Threshold t(loosest_minima(true, best + (int64_t)pair * slots_of(P) * S + sample, S, P, n, n,
                                       (its >> 30 & 1u) != 0, its >> 31 != 0, limits.cutoff), offsets);
      lds_thresholds[2 * sample * kFilterPitch + pair] = t.front;
      lds_thresholds[(2 * sample + 1) * kFilterPitch + pair] = t.post;
    }
    __syncthreads();
  }

  // whether any lane's row can matter: the pseudo row against the loosest minima, of the sample before first
  const double loosest_ratio = ratios.r[kSamples ? min(lane & 31, S - 1) : 0];
  const Threshold loosest =
      kSamples ? Threshold(0.0, 0.0)
               : Threshold(loosest_minima(true, best + (int64_t)lane * slots_of(P), 1, P, np, np, do_post, do_pp, limits.cutoff,
                                          limits.closed_below(pc.l)),
                           group_offsets(m, loosest_ratio));
  if (!kSamples && !__any(loosest.at(0.0) > -INFINITY)) return;  // (nothing of the tile is looked for)
  int s = 0;
  auto passes = [&](const double *f) {
    float x, d;
    pair_latency(f, k, x, d);
    if (!kSamples) return (bool)__any(m.bound(loosest_ratio, x, d) <= loosest.at(post_layer_offset(m, loosest_ratio, f)));
    const double low_x = m.lower_x(x), low_share = m.lower_share(d);
    for (int n = 0; n < S; ++n) {
      const double ratio = from_lane(loosest_ratio, s);
      const Threshold t(lds_thresholds[2 * s * kFilterPitch + lane], lds_thresholds[(2 * s + 1) * kFilterPitch + lane]);
      if (__any(ratio * low_x + low_share <= t.at(post_layer_offset(m, ratio, f)))) return true;
      s = s + 1 == S ? 0 : s + 1;
    }
    return false;
  };
  const double *__restrict__ supers = super_floor + super_floor_slot(g, gi, 0) * kStageFloorPitch;
  const double *__restrict__ stages = stage_floor + stage_floor_slot(g, gi, 0) * kStageFloorPitch;
  // One sample: summaries go through LDS; the next one of eight stages is on its way while one is tried, the
  // stages of one that passes come together.  (Each read where it was needed: 22B on 16x8 0.90 ms, now 0.68.
  // Several samples take longer over a summary and would lose a workgroup a CU: 7B on 4x8 0.16 -> 0.17.)
  __shared__ double floors[kSamples ? 1 : 1 + kSuperStages][kStageFloorPitch];
  auto super_term = [&](int super) {
    return supers[(int64_t)min(super, super_last) * kStageFloorPitch + lane % kStageFloorPitch];
  };
  double term = !kSamples && super_first <= super_last ? super_term(super_first) : 0.0;
  // batches of 64 summaries; lane i keeps the open stages of the batch's i-th
  for (int first = super_first; first <= super_last; first += 64 * stride) {
    uint32_t open = 0;
    for (int i = 0; i < 64; ++i) {
      const int super = first + i * stride;
      if (super > super_last) break;
      const int st0 = max(super * kSuperStages, stage0), st1 = min((super + 1) * kSuperStages, stage1);
      uint32_t seen = 0;
      if constexpr (kSamples) {
        if (!passes(supers + (int64_t)super * kStageFloorPitch)) continue;
        for (int st = st0; st < st1; ++st)
          if (passes(stages + (int64_t)st * kStageFloorPitch)) seen |= 1u << (st - st0);
      } else {
        __builtin_amdgcn_wave_barrier();
        if (lane < kStageFloorPitch) floors[0][lane] = term;
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        term = super_term(super + stride);
        if (!passes(floors[0])) continue;
        constexpr int kAtOnce = 64 / kStageFloorPitch;
        double its_terms[kSuperStages / kAtOnce];
#pragma unroll
        for (int u = 0; u < kSuperStages / kAtOnce; ++u)
          its_terms[u] = stages[(int64_t)min(st0 + u * kAtOnce + lane / kStageFloorPitch, st1 - 1) * kStageFloorPitch +
                                lane % kStageFloorPitch];
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int u = 0; u < kSuperStages / kAtOnce; ++u)
          floors[1 + u * kAtOnce + lane / kStageFloorPitch][lane % kStageFloorPitch] = its_terms[u];
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        for (int st = st0; st < st1; ++st)
          if (passes(floors[1 + st - st0])) seen |= 1u << (st - st0);
      }
      open = lane == i ? seen : open;
    }
    // append the open stages to a shard of the queue, which one XCD works off, to the next ones if it is
    // full (all shards together hold every (tile, stage) of the launch).  One sample: the shard of the
    // chunk, so that the tiles which open a stage read its 17 KB of rows while they are in the L2 (the
    // shard of the tile, for the minima: six times the rows from memory, 10.6 GB of 22B on 16x8 and 3.8
    // instead of 3.2 ms of the reduce launch).  Several: the shard of the tile, whose minima are the
    // larger part (1 MB with 30 samples).
    const int mine = __popc(open);
    int end = mine;
    for (int step = 1; step < 64; step <<= 1) {
      const int o = __shfl_up(end, step);
      if (lane >= step) end += o;
    }
    const int total = from_lane(end, 63);
    int shard = (gi * 13 + (S > 1 ? tile_rel : chunk)) % kQueueShards;
    for (int done = 0; done < total; shard = (shard + 1) % kQueueShards) {
      uint32_t base = 0;
      if (lane == 0) base = atomicAdd(tabs.counter + shard * kCounterPitch, (uint32_t)(total - done));
      base = (uint32_t)from_lane((int)base, 0);
      const int room = base >= tabs.capacity ? 0 : (int)min((uint32_t)(total - done), tabs.capacity - base);
      int at = end - mine;  // index of this lane's next item among the batch's
      const int st0 = max((first + lane * stride) * kSuperStages, stage0);
      for (uint32_t rest = open; rest != 0; rest &= rest - 1, ++at) {
        if (at < done || at >= done + room) continue;
        const int st = st0 + __ffs(rest) - 1;
        tabs.item[(int64_t)shard * tabs.capacity + base + (at - done)] = Item(gi, tile_rel, st).word();
      }
      done += room;
    }
  }
}

// ---- open ----
// Flat list over the shards of a queue, in shard order (lane = shard).
struct FlatQueue {
  uint32_t end;  // of this lane's shard
  uint32_t total;
  __device__ __forceinline__ int64_t at(uint32_t i, uint32_t capacity) const {
    const int shard = __popcll((unsigned long long)__ballot(end <= i));
    const uint32_t first = shard > 0 ? (uint32_t)from_lane((int)end, shard - 1) : 0u;
    return (int64_t)shard * capacity + (i - first);
  }
};
__device__ __forceinline__ FlatQueue flat_queue(const ReduceTables &tabs, int queue) {
  const int lane = threadIdx.x & 63;
  FlatQueue q;
  q.end = min(tabs.counter[(queue * kQueueShards + lane) * kCounterPitch], tabs.capacity);
  for (int step = 1; step < 64; step <<= 1) {
    const uint32_t o = (uint32_t)__shfl_up((int)q.end, step);
    if (lane >= step) q.end += o;
  }
  q.total = (uint32_t)from_lane((int)q.end, 63);
  return q;
}

// A lane's pair of a tile.
struct TileLane {
  PairIndex pc;
  bool active, do_post, do_pp;
  int np;
};
__device__ __forceinline__ TileLane tile_lane(const MistProblem &prob, const MistGroupDesc *__restrict__ g, int tile_rel) {
  const int L = prob.num_layers, n_pairs = L * (L + 1) / 2 + L;
  const int pair_idx = (g->lc_tile_begin + tile_rel) * MIST_LC_TILE + (int)(threadIdx.x & 63);
  TileLane t;
  t.active = pair_idx < n_pairs;
  t.pc = decode_pair(t.active ? pair_idx : 0);
  t.np = !t.active ? 0 : (t.pc.c == t.pc.l - 1 ? min(g->num_p, 1) : g->num_p);
  t.do_post = t.active && t.pc.c != t.pc.l - 1;
  t.do_pp = t.do_post && t.pc.l == L;
  return t;
}

// A wavefront takes runs of neighbouring items: only what the memory bounds of their stages leave open
// stays, with a word of its open pairs (7B on 4x8: 454000 stages x tiles, 36300 pass the filter and
// 13700 of those are opened; 22B on 16x8: 21.1e6, 2.1e6, 0.45e6).  Items of a run are mostly the
// stages of one tile, whose pairs, constants and offsets stay in registers.
//   One sample: lane = pair; the latency of an item bounds it (an item of its own per wavefront, everything
//   computed again for each, 540 VALU instructions: 22B 2.9 ms; constants of the tile kept 2.2; the next
//   item's summary through LDS 1.9; one append a run instead of three dependent atomics an opened item 1.5;
//   70B on 32x8 0.92 -> 0.38.  Gathering minima only for pairs below the filter's thresholds: no change).
//   Several: lane = pair for what the stage can reach, then lane = (pair parity, sample): the minima of a
//   slot lie side by side, two lines per load (lane = pair through all samples, a line per lane and load,
//   kept the address units busy 82 % of the time: 30 samples of 7B for one tensor-parallel size 1.41 ms;
//   now 0.45, and it knows every open pair: the reduce launch tries 1.4e6 instead of 2.9e6).
constexpr int kOpenRun = 16;  // (items kept by lanes)
template <bool kSamples>
__global__ __launch_bounds__(kReduceThreads) void open_kernel(const MistProblem prob,
                                                              const MistGroupDesc *__restrict__ groups,
                                                              const double *__restrict__ stage_floor,
                                                              const RatioList ratios, const ReduceTables tabs) {
  constexpr int kWaves = kReduceThreads / 64;
  const int lane = threadIdx.x & 63, S = kSamples ? tabs.n_samples : 1;
  const int sample = kSamples ? min(lane & 31, S - 1) : 0;
  const FlatQueue queue = flat_queue(tabs, 0);
  const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(blockIdx.x * kWaves + (threadIdx.x >> 6)));
  const uint32_t n_waves = gridDim.x * kWaves, run = max(1u, min((uint32_t)kOpenRun, queue.total / (2 * n_waves)));
  const double ratio = ratios.r[sample];
  // of the tile the last item was of
  uint64_t tile_word = ~0ull;
  const MistGroupDesc *g = groups;
  TileLane p = {};
  PairConsts k = {};
  GroupModel m = {};
  Offsets group = {};
  CostLimits limits = {};
  int P = 1;
  const double *best = tabs.best;
  // (the next item's summary is on its way to LDS while one is worked on, and the word of the one after it)
  __shared__ double lds_floor[kWaves][2][kStageFloorPitch];
  double(*const floor_of)[kStageFloorPitch] = lds_floor[threadIdx.x >> 6];
  auto floor_term = [&](uint64_t word) {
    const Item item(word);
    return stage_floor[stage_floor_slot(groups + item.group, item.group, item.stage) * kStageFloorPitch +
                       lane % kStageFloorPitch];
  };
  // what a run opens is appended together, lane = item
  uint64_t kept_word = 0, kept_open = 0;
  uint32_t kept_shard = 0;
  int n_kept = 0;
  uint32_t kept_pairs = 0;
  auto append = [&]() {
    if (n_kept == 0) return;
    const bool mine = lane < n_kept;
    const int64_t shard0 = (int64_t)kept_shard * tabs.capacity;
    // (no more than the shard's items are opened: it cannot overflow)
    uint32_t base = 0;
    static_assert(kOpenPairs == 1, "both counters in one word");
    if (lane == 0)
      base = (uint32_t)atomicAdd(reinterpret_cast<unsigned long long *>(tabs.counter + (kQueueShards + kept_shard) * kCounterPitch),
                                 (unsigned long long)kept_pairs << 32 | (uint32_t)n_kept);
    base = (uint32_t)from_lane((int)base, 0);
    if (mine) {
      tabs.opened[shard0 + base + lane] = kept_word;
      tabs.open_pairs[shard0 + base + lane] = kept_open;
    }
    n_kept = 0;
    kept_pairs = 0;
    if (tabs.listed == nullptr) return;
    const Item item(kept_word);
    bool fresh = false;
    if (mine)
      fresh = atomicExch(tabs.stage_flag + stage_floor_slot(groups + item.group, item.group, item.stage), 1u) == 0;
    const uint64_t listed = __ballot(fresh);
    if (listed == 0) return;
    if (lane == 0)
      base = atomicAdd(tabs.counter + (2 * kQueueShards + kept_shard) * kCounterPitch, (uint32_t)__popcll(listed));
    base = (uint32_t)from_lane((int)base, 0);
    if (fresh)
      tabs.listed[shard0 + base + __popcll(listed & ((1ull << lane) - 1ull))] =
          (unsigned long long)item.group << 32 | (uint32_t)item.stage;
  };
  for (uint32_t first = wave * run; first < queue.total; first += n_waves * run) {
    const uint32_t end = min(first + run, queue.total);
    int64_t from = queue.at(first, tabs.capacity), from_next = queue.at(min(first + 1, end - 1), tabs.capacity);
    uint64_t word = from_lane((uint64_t)tabs.item[from], 0), ahead = tabs.item[from_next];
    double term = floor_term(word);
    for (uint32_t i = first; i < end; ++i) {
      double *const f = floor_of[i & 1];
      __builtin_amdgcn_wave_barrier();
      if (lane < kStageFloorPitch) f[lane] = term;
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
      const uint32_t shard = (uint32_t)(from / tabs.capacity);
      const Item item(word);
      const uint64_t its_word = word;
      from = from_next;
      word = from_lane(ahead, 0);
      term = floor_term(word);
      from_next = queue.at(min(i + 2, end - 1), tabs.capacity);
      ahead = tabs.item[from_next];
      const int gi = item.group, stage = item.stage;
      if (its_word >> kItemStageBits != tile_word) {
        tile_word = its_word >> kItemStageBits;
        g = groups + gi;
        p = tile_lane(prob, g, item.tile);
        if (kSamples && !in_assignments(prob, tabs, gi, p.pc.l)) {
          p.active = p.do_post = p.do_pp = false;
          p.np = 0;
        }
        k = pair_consts(p.pc.l, p.pc.c);
        m = group_model(prob, g);
        group = group_offsets(m, ratio);
        limits = cost_limits(prob, tabs, gi, m.inv_G64);
        P = g->num_p;
        best = tabs.best + (g->cell_offset + (int64_t)item.tile * MIST_LC_TILE * slots_of(P)) * S;
      }
      const StageReach reach = stage_reach(f, k, p.np, p.do_post, p.do_pp, m);
      const double post_layer = post_layer_offset(m, ratio, f);
      uint64_t open = 0;
      if (!kSamples) {
        // (what lies above the cutoff needs no minima)
        const double bound = m.bound(ratio, reach.x, reach.d);
        const Loosest low = loosest_minima(p.active && bound <= limits.cutoff, best + lane * slots_of(P), 1, P, reach.count_b,
                                           reach.count_p, reach.post, reach.pp, limits.cutoff, limits.closed_below(p.pc.l));
        open = __ballot(bound <= Threshold(low, group).at(post_layer));
      } else {
        const int parts = reach.count_b | reach.count_p << 15 | (int)reach.post << 30 | (int)((unsigned)reach.pp << 31);
        // two pairs at a time
        for (uint64_t rest = __ballot(p.active && parts != 0); rest != 0;) {
          const int even = __ffsll((unsigned long long)rest) - 1;
          rest &= rest - 1;
          const int odd = rest != 0 ? __ffsll((unsigned long long)rest) - 1 : even;
          rest &= rest - 1;
          const int mine = lane < 32 ? even : odd;
          const uint32_t its = (uint32_t)__shfl(parts, mine);
          const Loosest low = loosest_minima(true, best + (int64_t)mine * slots_of(P) * S + sample, S, P, (int)(its & 0x7fff),
                                             (int)(its >> 15 & 0x7fff), (its >> 30 & 1u) != 0, its >> 31 != 0, INFINITY);
          const uint64_t pass =
              __ballot(m.bound(ratio, __shfl(reach.x, mine), __shfl(reach.d, mine)) <= Threshold(low, group).at(post_layer));
          open |= ((uint32_t)pass != 0 ? 1ull << even : 0ull) | (pass >> 32 != 0 ? 1ull << odd : 0ull);
        }
      }
      if (open == 0) continue;
      if (n_kept > 0 && shard != kept_shard) append();
      kept_shard = shard;
      if (lane == n_kept) {
        kept_word = its_word;
        kept_open = open;
      }
      ++n_kept;
      kept_pairs += __popcll(open);
    }
    append();
  }
}

// ---- rows of the opened stages ----
// Workgroup = two stages of the list at a time.
__global__ __launch_bounds__(kTermsBlock) void stage_rows_kernel(
    const MistProblem prob, const MistGroupDesc *__restrict__ groups, double *__restrict__ row_terms,
    const double *__restrict__ key_terms, const ReduceTables tabs) {
  constexpr int kStages = kTermsBlock / kStageRows;
  __shared__ double lds_out[kStageRows * (MIST_ROW_TERMS + 1)];
  __shared__ __align__(16) double lds_factor[11][kFactorPitch];
  __shared__ double lds_gpu_gpu[32];
  const FlatQueue queue = flat_queue(tabs, 2);
  if (blockIdx.x * kStages >= queue.total) return;
  InterferenceModel<true> I;
  I.factors_tame = load_model_tables(prob, lds_factor, lds_gpu_gpu);
  I.table = (LdsDouble *)&lds_factor[0][0];
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x / kStageRows), lane = threadIdx.x % kStageRows;
  for (uint32_t first = blockIdx.x * kStages; first < queue.total; first += gridDim.x * kStages) {
    auto stage_of = [&](int k) {
      return from_lane((uint64_t)tabs.listed[queue.at(min(first + k, queue.total - 1), tabs.capacity)], 0);
    };
    double t[MIST_ROW_TERMS];
    {
      const uint64_t its = stage_of(wave);
      const MistGroupDesc *g = groups + (int)(its >> 32);
      const int64_t row0 = (int64_t)(uint32_t)its * kStageRows;
      row_terms_of<true>(prob, g, (uint32_t)min(row0 + lane, g->n_rows - 1), key_terms, lds_gpu_gpu, I, t);
    }
    for (int k = 0; k < kStages; ++k) {
      __syncthreads();
      if (wave == k) {
#pragma unroll
        for (int i = 0; i < MIST_ROW_TERMS; ++i) lds_out[lane * (MIST_ROW_TERMS + 1) + i] = t[i];
      }
      __syncthreads();
      if (first + k >= queue.total) continue;
      const uint64_t its = stage_of(k);
      const MistGroupDesc *g = groups + (int)(its >> 32);
      const int64_t row0 = (int64_t)(uint32_t)its * kStageRows;
      store_rows(lds_out, (int)min((int64_t)kStageRows, g->n_rows - row0),
                 row_terms + (g->row_offset + row0) * MIST_ROW_TERMS);
    }
  }
}

// ---- reduce / resolve ----
// A wavefront's place in the log: it takes a chunk at a time.
struct HitLog {
  uint32_t chunk = ~0u, used = kLogChunk;  // (wave-uniform; ~0: none)
  bool full = false;
  __device__ __forceinline__ void close(const ReduceTables &tabs) const {
    if (chunk != ~0u && (threadIdx.x & 63) == 0) tabs.log_count[chunk] = used;
  }
  // All lanes of the wavefront: what each notes of the four variants (`hit`: a bit per variant).
  __device__ __forceinline__ void put(const ReduceTables &tabs, uint32_t hit, const double (&cost)[4], const uint32_t (&cell)[4],
                                      uint32_t row) {
    uint64_t mask[4];
    uint32_t n = 0;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      mask[v] = __ballot((hit >> v & 1u) != 0);
      n += __popcll(mask[v]);
    }
    if (n == 0 || full) return;
    const int lane = threadIdx.x & 63;
    static_assert(kLogChunk >= 4 * 64, "what a wavefront notes at once");
    if (used + n > (uint32_t)kLogChunk) {
      close(tabs);
      uint32_t its = 0;
      if (lane == 0) its = atomicAdd(tabs.counter + kLogTaken * kCounterPitch, 1u);
      chunk = (uint32_t)from_lane((int)its, 0);
      used = 0;
      if (chunk >= tabs.log_chunks) {
        if (lane == 0) tabs.counter[kLogFull * kCounterPitch] = 1;
        chunk = ~0u;
        full = true;
        return;
      }
    }
    Hit *log = tabs.log + (int64_t)chunk * kLogChunk + used;
    used += n;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      if (hit >> v & 1u) log[__popcll(mask[v] & ((1ull << lane) - 1ull))] = Hit{cost[v], cell[v], row};
      log += __popcll(mask[v]);
    }
  }
};

// One item with the pairs in `pairs`, one sample.  kResolve: after a log that ran full, with final minima.
//   lane = pair   the slots the stage's pseudo row can reach, and with their minima a threshold;
//   lane = row    the rows below it, by their linear bounds: two FMAs and a compare per pair;
//   lane = row    of the pairs that have any: a bound of each row's count and the minimum there (one
//                 pair's minima at a time in `lds_row`, the next ones on their way in registers);
//   lane = (row, pair) of what is left, collected in `queue`: the reference's arithmetic.
// VALU issue bounds it: of 22B on 16x8's 12.6e6 pairs with an open stage 4.9e6 hold rows below the
// threshold, 23 of 64 rows each, and 0.9e6 a row that may reach a minimum.  (Every pair's rows through
// the reference's latencies, then memory, counts and objectives for all of them as soon as one was
// below the threshold: 1.9e9 wave instructions and 5.1 ms; now 1.05e9 and 3.2.  70B on 32x8 4.2 -> 2.6,
// 7B on 4x8 0.28 -> 0.19.  Four wavefronts per SIMD, with 128 registers, are no faster than three.)
// kInLds false: there are too many minima for the buffer (see kMostBufferedSlots), rows look them up in memory.
template <bool kResolve, bool kInLds>
__device__ __forceinline__ void reduce_item(const MistProblem &prob, const MistGroupDesc *__restrict__ g, int gi,
                                            int tile_rel, int stage, const double *__restrict__ row_terms,
                                            const double *__restrict__ stage_floor, double ratio,
                                            const ReduceTables &tabs, uint64_t pairs, double *lds, HitLog &log) {
  const int L = prob.num_layers, lane = threadIdx.x & 63;
  const int P = g->num_p, n_slots = slots_of(P);
  const GroupModel m = group_model(prob, g);
  const CostLimits limits = cost_limits(prob, tabs, gi, m.inv_G64);
  const double cutoff = limits.cutoff;
  const int64_t tile_cell = g->cell_offset + (int64_t)tile_rel * MIST_LC_TILE * n_slots;
  const double *best = tabs.best + tile_cell;  // [pair][slot]

  uint16_t *queue = reinterpret_cast<uint16_t *>(lds);  // pair << 6 | row
  double *lds_row = lds + kCandidateDoubles;
  // ---- lane = pair ----
  const double *__restrict__ f = stage_floor + stage_floor_slot(g, gi, stage) * kStageFloorPitch;
  double thr, thr_post;  // of this lane's pair: of any variant, of with_post and no_pp
  double off_pre;
  int lc;  // l | c << 15
  uint64_t todo;
  {
    const TileLane tl = tile_lane(prob, g, tile_rel);
    lc = tl.pc.l | tl.pc.c << 15;
    const StageReach reach = stage_reach(f, pair_consts(tl.pc.l, tl.pc.c), tl.np, tl.do_post, tl.do_pp, m);
    const double bound = m.bound(ratio, reach.x, reach.d);
    const Loosest low = loosest_minima((pairs >> lane & 1ull) != 0 && bound <= cutoff, best + lane * n_slots, 1, P,
                                       reach.count_b, reach.count_p, reach.post, reach.pp, cutoff,
                                       limits.closed_below(tl.pc.l));
    const Offsets off = group_offsets(m, ratio);
    const Threshold its(low, off);
    const double post_layer = post_layer_offset(m, ratio, f);
    thr = its.at(post_layer);
    thr_post = its.post - post_layer;
    off_pre = off.pre;
    todo = pairs & __ballot(bound <= thr);
  }
  if (todo == 0) return;

  // ---- lane = row ----
  const int64_t row0 = (int64_t)stage * kStageRows;
  const int n_stage = (int)min((int64_t)kStageRows, g->n_rows - row0);
  const double *__restrict__ rows = row_terms + (g->row_offset + row0) * MIST_ROW_TERMS;
  const uint64_t live = ~0ull >> (64 - n_stage);
  LinearBound bound;
  {
    RowRegs t;
    load_terms<0, MIST_T_D_LAST_NOCK + 1>(t, rows + min(lane, n_stage - 1) * MIST_ROW_TERMS);
    bound = linear_bound(t, ratio, m.inv_G64);
  }
  auto pair_at = [&](int pl) {
    const int its = from_lane(lc, pl);
    return LinearPair(its & 0x7fff, its >> 15);
  };
  uint64_t left = 0;  // pairs with rows below their threshold
  for (uint64_t rest = todo; rest != 0; rest &= rest - 1) {
    const int pl = __ffsll((unsigned long long)rest) - 1;
    const LinearPair p = pair_at(pl);
    const uint64_t pass = live & __ballot(bound.at(p.n_ck, p.n_nock, p.all_ck, p.none) <= from_lane(thr, pl));
    left |= pass != 0 ? 1ull << pl : 0ull;
  }
  if (left == 0) return;
  LinearMemory mem;
  {
    RowRegs t;
    load_terms<MIST_T_D_LAST_NOCK + 1, MIST_T_GCB + 1>(t, rows + min(lane, n_stage - 1) * MIST_ROW_TERMS);
    mem = linear_memory(t);
  }
  // minima of one pair, a slot per lane and register
  double ahead0 = 0.0, ahead1 = 0.0;
  auto fetch = [&](int pair) {
    if (!kInLds) return;
    const double *slots = best + pair * n_slots;
    ahead0 = slots[min(lane, n_slots - 1)];
    if (n_slots > 64) ahead1 = slots[min(lane + 64, n_slots - 1)];
  };
  auto settle = [&](int pair) {
    if (!kInLds) return;
    __builtin_amdgcn_wave_barrier();
    if (lane < n_slots) lds_row[lane] = ahead0;
    if (lane + 64 < n_slots) lds_row[lane + 64] = ahead1;
    for (int j = lane + 128; j < n_slots; j += 64) lds_row[j] = best[pair * n_slots + j];
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  };

  // ---- lane = (row, pair): the first `n` of the queue ----
  auto settle_candidates = [&](int n) {
    const uint32_t entry = queue[min(lane, n - 1)];
    const int pl = (int)(entry >> 6), its_row = (int)(entry & 63u);
    const int its = __shfl(lc, pl), l = its & 0x7fff, c = its >> 15;
    const bool in = lane < n;
    RowRegs t;
    load_terms<0, MIST_T_D_LAST_NOCK + 1>(t, rows + its_row * MIST_ROW_TERMS);
    const PairConsts k = pair_consts(l, c);
    float x, d;
    pair_latency(t, k, x, d);
    asm volatile("" : "+v"(x), "+v"(d)::"memory");
    load_terms<MIST_T_NAG_CK, MIST_ROW_TERMS>(t, rows + its_row * MIST_ROW_TERMS);
    const int np = c == l - 1 ? min(P, 1) : P;
    const bool do_post = in && c != l - 1, do_pp = do_post && l == L;
    Objectives o = objectives(t, x, d, k.no_ck, ratio, m, true);
    asm volatile("" : "+v"(o.base), "+v"(o.pre), "+v"(o.post), "+v"(o.pp)::"memory");
    load_terms<MIST_T_D_LAST_NOCK + 1, MIST_T_NAG_CK>(t, rows + its_row * MIST_ROW_TERMS);
    const LaneMemory lm = pair_memory(t, k);
    const UpperCounts upper = upper_counts(lm, m, in ? np : 0);
    const RowCounts cnt = exact_counts(lm, m, upper.b, upper.p);
    bool ok_post, ok_pp;
    post_fits(t, k, lm, m, lm.out, k.no_ck ? t[MIST_T_RD] : 0.0, ok_post, ok_pp);
    const int64_t cell = tile_cell + pl * n_slots;
    const int own_b = max(cnt.b - 1, 0), own_p = P + max(cnt.p - 1, 0);
    const double *slots = tabs.best + cell;
    const double now_b = slots[own_b], now_p = slots[own_p], now_post = slots[2 * P], now_pp = slots[2 * P + 1];
    const uint64_t reached = __ballot(o.base <= now_b || o.pre <= now_p || o.post <= now_post || o.pp <= now_pp);
    if (reached == 0) return;
    const uint32_t number = (uint32_t)row_of_position(g, row0 + its_row);
    // A lowered slot may lie below the slots under it; a row above it is above the winner of its own
    // slot too, which finalize takes from the slots at and above.
    const double cost[4] = {o.base, o.pre, o.post, o.pp};
    const uint32_t cells[4] = {(uint32_t)cell + own_b, (uint32_t)cell + own_p, (uint32_t)cell + 2 * P, (uint32_t)cell + 2 * P + 1};
    uint32_t hit = 0;
    auto offer = [&](bool ok, int variant, int own, double now) {
      const double its = cost[variant];
      if (!(ok && its <= now && its <= cutoff && its < INFINITY)) return;
      hit |= 1u << variant;
      if (kResolve) atomicMin(tabs.row + cell + own, number);
      else if (its < now) lower_minimum(tabs.best + cell + own, its);
    };
    offer(cnt.b > 0, 0, own_b, now_b);
    offer(cnt.p > 0, 1, own_p, now_p);
    offer(do_post && ok_post, 2, 2 * P, now_post);
    offer(do_pp && ok_pp, 3, 2 * P + 1, now_pp);
    if (!kResolve) log.put(tabs, hit, cost, cells, number);
  };

  const double cap_and_room = m.cap * (1.0 + 1e-12);
  int waiting = 0;
  fetch(__ffsll((unsigned long long)left) - 1);
  uint64_t rest = left;
  while (rest != 0 || waiting > 0) {
    if (rest != 0) {
      const int pl = __ffsll((unsigned long long)rest) - 1;
      settle(pl);
      rest &= rest - 1;
      if (rest != 0) fetch(__ffsll((unsigned long long)rest) - 1);
      const LinearPair p = pair_at(pl);
      const double low = bound.at(p.n_ck, p.n_nock, p.all_ck, p.none);
      const LinearReach reach = linear_reach(mem, p, m, p.c == p.l - 1 ? min(P, 1) : P, cap_and_room);
      auto minimum = [&](int slot) { return kInLds ? lds_row[slot] : best[(int64_t)pl * n_slots + slot]; };
      const double now_b = minimum(max(reach.count_b - 1, 0)), now_p = minimum(P + max(reach.count_p - 1, 0));
      const double closed_below = limits.closed_below(p.l);
      bool may = (reach.count_b > 0 && low <= up_to(now_b, cutoff, closed_below)) ||
                 (reach.count_p > 0 && low <= up_to(now_p, cutoff, closed_below) - off_pre);
      const bool may_post = low <= from_lane(thr_post, pl);
      if (__any(may_post)) may = may || (may_post && post_may_fit(reach, mem, p, L, m, cap_and_room));  // a pair in seven
      const uint64_t found = live & __ballot(may && low <= from_lane(thr, pl));
      if (found >> lane & 1ull)
        queue[waiting + __popcll(found & ((1ull << lane) - 1ull))] = (uint16_t)(pl << 6 | lane);
      waiting += __popcll(found);
      if (waiting == 0 || (waiting < 64 && rest != 0)) continue;
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    settle_candidates(min(waiting, 64));
    waiting = max(waiting - 64, 0);
    const uint16_t moved = queue[64 + lane];
    __builtin_amdgcn_wave_barrier();
    queue[lane] = moved;
  }
}

// The same for several samples.  The linear bounds of a row are those of its stable and of its delta part,
// so that a sample's is one FMA.  Per pair
//   lane = (one of two pairs, sample)  thresholds, and the samples that the stage's pseudo row passes (they
//                   lie side by side, 4 to 12 of 30 on the 7B plans);
//   lane = row      the rows below the threshold of some of them, and bounds of their counts;
//   lane = (row, sample)  as many rows side by side as the samples leave room for: bounds against the minima at
//                   the rows' counts, kRowLooks look-ups per slot in flight;
//   lane = (row, pair), then (row, sample)  of what is left, collected in `queue`: the reference's arithmetic,
//                   and a minimum per row, variant and sample.
// (A wavefront that took the samples one after the other, its minima through LDS: 14 ms for the tables of one
// tensor-parallel size of the 7B plan; lane = row for the reference's latencies and counts, then two rows by 32
// samples: 3.95 ms, 1160 vector instructions a pair; now 2.1 ms and 370, which wait for the look-ups most of
// the time.  Four wavefronts per SIMD spill, 4.0 ms; the next pairs' thresholds fetched ahead: 2.3, they are
// older by then.  30 samples of 7B on 4x8 1.65 -> 0.81 ms.)
constexpr int kRowLooks = 4;
constexpr int kLinearMemoryTerms = sizeof(LinearMemory) / 8;
struct SampleQueue {
  union {
    struct {
      double2 low[64], post[64];  // of a pair's rows: stable and delta part of the bounds
      uint32_t counts[64];        // bounds of the counts: base | with_pre << 15 | with_post or no_pp << 30
      uint8_t row[64];
    };
    SampleRows exact;  // of the candidates
  };
  double mem[kLinearMemoryTerms][64];  // of the stage's rows (24 registers through the whole item otherwise)
  double2 post_terms[64];
  uint32_t entry[kCandidates];         // pair | row << 6 | first sample << 12 | samples << 17
  uint32_t useful[64];                 // the same of the candidates that have a count
};
// `n` items of `width` lanes each, side by side.
struct LaneGroups {
  int width, n, item, offset;
  __device__ __forceinline__ LaneGroups(int lane, int w) : width(w) {
    const int inverse = (65536 + w - 1) / w;  // (exact for 64 lanes)
    n = 64 * inverse >> 16;
    item = lane * inverse >> 16;
    offset = lane - item * w;
  }
  // lane `item` = the lanes of `of` that are its
  __device__ __forceinline__ uint32_t bits(uint64_t of, int its) const {
    return (uint32_t)(of >> (its * width & 63)) & (uint32_t)((1ull << width) - 1ull);
  }
};
template <bool kResolve>
__device__ __forceinline__ void reduce_item_samples(const MistProblem &prob, const MistGroupDesc *__restrict__ g,
                                                    int gi, int tile_rel, int stage,
                                                    const double *__restrict__ row_terms,
                                                    const double *__restrict__ stage_floor, const RatioList &ratios,
                                                    const ReduceTables &tabs, uint64_t pairs, SampleQueue *queue,
                                                    HitLog &log) {
  SampleRows *const exact = &queue->exact;
  const int L = prob.num_layers, lane = threadIdx.x & 63, S = tabs.n_samples;
  const int my_sample = min(lane & 31, S - 1);
  const int P = g->num_p, n_slots = slots_of(P);
  const GroupModel m = group_model(prob, g);
  const int64_t tile_cell = g->cell_offset + (int64_t)tile_rel * MIST_LC_TILE * n_slots;
  const double *best = tabs.best + tile_cell * S;  // [pair][slot][sample]
  const double *__restrict__ f = stage_floor + stage_floor_slot(g, gi, stage) * kStageFloorPitch;
  const double ratio = ratios.r[my_sample];
  const Offsets off = group_offsets(m, ratio);
  const double post_layer = post_layer_offset(m, ratio, f);
  // ---- lane = pair: what the pseudo row of the stage can reach ----
  int lc, parts;  // l | c << 15; counts as in SampleRows
  float floor_x, floor_d;
  {
    const TileLane tl = tile_lane(prob, g, tile_rel);
    lc = tl.pc.l | tl.pc.c << 15;
    const StageReach reach = stage_reach(f, pair_consts(tl.pc.l, tl.pc.c), tl.np, tl.do_post, tl.do_pp, m);
    parts = reach.count_b | reach.count_p << 15 | (int)reach.post << 30 | (int)((unsigned)reach.pp << 31);
    floor_x = reach.x;
    floor_d = reach.d;
    pairs &= __ballot(tl.active && parts != 0);
  }
  if (pairs == 0) return;

  // ---- lane = row ----
  const int64_t row0 = (int64_t)stage * kStageRows;
  const int n_stage = (int)min((int64_t)kStageRows, g->n_rows - row0);
  const double *__restrict__ rows = row_terms + (g->row_offset + row0) * MIST_ROW_TERMS;
  const uint64_t live = ~0ull >> (64 - n_stage);
  LinearBound stable, delta;
  __builtin_amdgcn_wave_barrier();
  {
    RowRegs t;
    load_terms<0, MIST_ROW_TERMS>(t, rows + min(lane, n_stage - 1) * MIST_ROW_TERMS);
    stable = linear_form([&](int its, int) { return less_slack(t[its]); });
    delta = linear_form([&](int, int its) { return less_slack(t[its] * m.inv_G64); });
    const LinearMemory mem = linear_memory(t);
#pragma unroll
    for (int i = 0; i < kLinearMemoryTerms; ++i) queue->mem[i][lane] = reinterpret_cast<const double *>(&mem)[i];
    const double opb = t[MIST_T_OPB], nag = fmin(t[MIST_T_NAG_NOCK], t[MIST_T_NAG_CK]),
                 nrs = fmin(t[MIST_T_NRS_NOCK], t[MIST_T_NRS_CK]);
    double2 post_terms;
    post_terms.x = less_slack(opb) + less_slack(m.k.pp_wre ? nag : 0.0) + less_slack(m.k.pp_gre ? nrs : 0.0);
    post_terms.y = less_slack(m.div_G(m.k.pp_wre ? 0.0 : nag)) + less_slack(m.div_G(m.k.pp_gre ? 0.0 : nrs));
    queue->post_terms[lane] = post_terms;
  }
  const double cap_and_room = m.cap * (1.0 + 1e-12);

  // ---- lane = (row, pair): the first `n` of the queue; then lane = (row, sample) ----
  auto settle_candidates = [&](int n) {
    const uint32_t entry = queue->entry[min(lane, n - 1)];
    const int pl = (int)(entry & 63u), its_row = (int)(entry >> 6 & 63u);
    int width = (int)(entry >> 17);
    {
      const int its = __shfl(lc, pl), l = its & 0x7fff, c = its >> 15;
      const bool in = lane < n;
      RowRegs t;
      load_terms<0, MIST_ROW_TERMS>(t, rows + its_row * MIST_ROW_TERMS);
      const PairConsts k = pair_consts(l, c);
      float x, d;
      pair_latency(t, k, x, d);
      const LaneMemory lm = pair_memory(t, k);
      const bool do_post = in && c != l - 1;
      const UpperCounts upper = upper_counts(lm, m, in ? (c == l - 1 ? min(P, 1) : P) : 0);
      const RowCounts cnt = exact_counts(lm, m, upper.b, upper.p);
      bool ok_post, ok_pp;
      post_fits(t, k, lm, m, lm.out, k.no_ck ? t[MIST_T_RD] : 0.0, ok_post, ok_pp);
      ok_post = ok_post && do_post;
      ok_pp = ok_pp && do_post && l == L;
      const bool useful = cnt.b > 0 || cnt.p > 0 || ok_post || ok_pp;
      const uint64_t some = __ballot(useful);
      const int at = __popcll(some & ((1ull << lane) - 1ull));
      if (useful) {
        put_sample_row(exact, at, t, x, d, k.no_ck, m, cnt.b, cnt.p, ok_post, ok_pp, true);
        exact->number[at] = (uint32_t)row_of_position(g, row0 + its_row);
        queue->useful[at] = entry;
      }
      n = __popcll(some);
    }
    if (n == 0) return;
    for (int step = 1; step < 64; step *= 2) width = max(width, __shfl_xor(width, step));
    const LaneGroups slot(lane, __builtin_amdgcn_readfirstlane(width));
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    // look-ups of a row, one iteration ahead of their use
    double now_b, now_p, now_post, now_pp;
    uint32_t counts, place;
    auto look = [&](int r) {
      counts = exact->counts[r];
      place = queue->useful[r];
      const int nb = (int)(counts & 0x7fff), npre = (int)(counts >> 15 & 0x7fff);
      const double *mine = best + (int64_t)(place & 63u) * n_slots * S + min((int)(place >> 12 & 31u) + slot.offset, S - 1);
      now_b = mine[max(nb - 1, 0) * S];
      now_p = mine[(P + max(npre - 1, 0)) * S];
      now_post = mine[2 * P * S];
      now_pp = mine[(2 * P + 1) * S];
    };
    look(min(slot.item, n - 1));
    for (int r0 = 0; r0 < n; r0 += slot.n) {
      const int r = min(r0 + slot.item, n - 1), its_pair = (int)(place & 63u), first = (int)(place >> 12 & 31u);
      const int sample = min(first + slot.offset, S - 1);
      const bool on = slot.item < slot.n && r0 + slot.item < n && first + slot.offset < S;
      const double its_ratio = __shfl(ratio, sample);
      const uint32_t cn = counts;
      const double nb_now = now_b, np_now = now_p, post_now = now_post, pp_now = now_pp;
      if (r0 + slot.n < n) look(min(r0 + slot.n + slot.item, n - 1));
      const uint32_t number = exact->number[r];
      const int nb = (int)(cn & 0x7fff), npre = (int)(cn >> 15 & 0x7fff);
      const int64_t to = (tile_cell + its_pair * n_slots) * S + sample;
      double cost[4];
      uint32_t cells[4], hit = 0;
      auto offer = [&](bool ok, int variant, int own, double now) {
        const double2 xy = exact->xy[variant][r];
        const double its = its_ratio * xy.x + xy.y;
        cost[variant] = its;
        cells[variant] = (uint32_t)to + (uint32_t)(own * S);
        if (!(on && ok && its <= now && its < INFINITY)) return;
        hit |= 1u << variant;
        if (kResolve) atomicMin(tabs.row + to + own * S, number);
        else if (its < now) lower_minimum(tabs.best + to + own * S, its);
      };
      offer(nb > 0, 0, nb - 1, nb_now);
      offer(npre > 0, 1, P + npre - 1, np_now);
      offer((cn >> 30 & 1u) != 0, 2, 2 * P, post_now);
      offer((cn >> 31) != 0, 3, 2 * P + 1, pp_now);
      if (!kResolve) log.put(tabs, hit, cost, cells, number);
    }
  };

  int waiting = 0;
  // A pair's rows; `thr_post` of sample `lane & 31`, `samples` that may pass.
  auto visit = [&](int pl, double thr, double thr_post, int half, uint32_t samples) {
    const int its_lc = from_lane(lc, pl);
    const LinearPair p(its_lc & 0x7fff, its_lc >> 15);
    const double low_x = stable.at(p.n_ck, p.n_nock, p.all_ck, p.none), low_y = delta.at(p.n_ck, p.n_nock, p.all_ck, p.none);
    uint64_t found = 0;
    for (uint32_t left = samples; left != 0; left &= left - 1) {
      const int s = __ffs(left) - 1;
      found |= __ballot(__builtin_fma(from_lane(ratio, s), low_x, low_y) <= from_lane(thr, half + s));
    }
    found &= live;
    if (found == 0) return;
    LinearMemory mem;
#pragma unroll
    for (int i = 0; i < kLinearMemoryTerms; ++i) reinterpret_cast<double *>(&mem)[i] = queue->mem[i][lane];
    const LinearReach reach = linear_reach(mem, p, m, p.c == p.l - 1 ? min(P, 1) : P, cap_and_room);
    const bool post = p.c != p.l - 1 && post_may_fit(reach, mem, p, L, m, cap_and_room);
    found &= __ballot(reach.count_b > 0 || reach.count_p > 0 || post);
    if (found == 0) return;
    const int n_found = __popcll(found);
    __builtin_amdgcn_wave_barrier();
    if (found >> lane & 1ull) {
      const int at = __popcll(found & ((1ull << lane) - 1ull));
      queue->low[at] = double2{low_x, low_y};
      const double2 post_terms = queue->post_terms[lane];
      queue->post[at] = double2{low_x + post_terms.x, low_y + post_terms.y};
      queue->counts[at] = (uint32_t)reach.count_b | (uint32_t)reach.count_p << 15 | (post ? 1u << 30 : 0u);
      queue->row[at] = (uint8_t)lane;
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    // ---- lane = (row, sample) ----
    const int first = __ffs(samples) - 1;
    const LaneGroups slot(lane, 32 - __clz(samples) - first);
    const int sample = min(first + slot.offset, S - 1);
    const double its_ratio = __shfl(ratio, sample), its_post = __shfl(thr_post, half + sample),
                 its_pre = __shfl(off.pre, sample);
    const bool on = slot.item < slot.n && first + slot.offset < S;
    const double *mine = best + (int64_t)pl * n_slots * S + sample;
    uint64_t may = 0;
    for (int r0 = 0; r0 < n_found; r0 += kRowLooks * slot.n) {
      double now_b[kRowLooks], now_p[kRowLooks];
      uint32_t counts[kRowLooks];
#pragma unroll
      for (int u = 0; u < kRowLooks; ++u) {
        counts[u] = queue->counts[min(r0 + u * slot.n + slot.item, n_found - 1)];
        now_b[u] = mine[max((int)(counts[u] & 0x7fff) - 1, 0) * S];
        now_p[u] = mine[(P + max((int)(counts[u] >> 15 & 0x7fff) - 1, 0)) * S];
      }
#pragma unroll
      for (int u = 0; u < kRowLooks; ++u) {
        const int first_row = r0 + u * slot.n, r = min(first_row + slot.item, n_found - 1);
        if (first_row >= n_found) break;
        const double2 xy = queue->low[r], post_xy = queue->post[r];
        const double low = __builtin_fma(its_ratio, xy.x, xy.y);
        const bool reached = ((low <= now_b[u]) & ((counts[u] & 0x7fff) != 0)) |
                             ((low <= now_p[u] - its_pre) & ((counts[u] >> 15 & 0x7fff) != 0)) |
                             ((__builtin_fma(its_ratio, post_xy.x, post_xy.y) <= its_post) & ((counts[u] >> 30 & 1u) != 0));
        const uint64_t some = __ballot(reached && on);
        if (some == 0) continue;
        const uint64_t its = __ballot(lane < slot.n && first_row + lane < n_found && slot.bits(some, lane) != 0);
        may |= its << first_row;
      }
    }
    if (may == 0) return;
    if (may >> lane & 1ull)
      queue->entry[waiting + __popcll(may & ((1ull << lane) - 1ull))] =
          (uint32_t)pl | (uint32_t)queue->row[lane] << 6 | (uint32_t)first << 12 | (uint32_t)slot.width << 17;
    waiting += __popcll(may);
  };
  double thr, thr_post;
  uint64_t may = 0;  // samples of the two pairs
  int pair_a = 0, pair_b = 0;
  for (uint64_t rest = pairs; rest != 0 || may != 0 || waiting > 0;) {
    if (may != 0) {
      const int half = (uint32_t)may != 0 ? 0 : 32;
      const uint32_t samples = (uint32_t)(may >> half);
      may &= ~(0xffffffffull << half);
      visit(half == 0 ? pair_a : pair_b, thr, thr_post, half, samples);
    } else if (rest != 0) {
      pair_a = __ffsll((unsigned long long)rest) - 1;
      rest &= rest - 1;
      const uint64_t second = rest != 0 ? ~0ull : 0xffffffffull;
      pair_b = rest != 0 ? __ffsll((unsigned long long)rest) - 1 : pair_a;
      rest &= rest - 1;
      // ---- lane = (pair, sample): thresholds ----
      const int pl = lane < 32 ? pair_a : pair_b;
      const uint32_t its_parts = (uint32_t)__shfl(parts, pl);
      const Threshold its(loosest_minima(true, best + (int64_t)pl * n_slots * S + my_sample, S, P, (int)(its_parts & 0x7fff),
                                         (int)(its_parts >> 15 & 0x7fff), (its_parts >> 30 & 1u) != 0, its_parts >> 31 != 0,
                                         INFINITY), off);
      thr = its.at(post_layer);
      thr_post = its.post;
      const double low = m.bound(ratio, __shfl(floor_x, pl), __shfl(floor_d, pl));
      may = second & __ballot((lane & 31) < S && low <= thr);
    }
    if (waiting < 64 && (waiting == 0 || rest != 0 || may != 0)) continue;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    settle_candidates(min(waiting, 64));
    waiting = max(waiting - 64, 0);
    const uint32_t moved = queue->entry[64 + lane];
    __builtin_amdgcn_wave_barrier();
    queue->entry[lane] = moved;
  }
}

// Every 2^k-th pair from the first on.
__device__ __forceinline__ uint64_t every_pair(int k) {
  return k == 0 ? ~0ull : k == 1 ? 0x5555555555555555ull : k == 2 ? 0x1111111111111111ull : k == 3 ? 0x0101010101010101ull
                                                                                     : 0x0001000100010001ull;
}

// A unit of work is an opened item with every 2^split-th of its pairs: an item has 1 to 64 open
// pairs at 1 - 3 us each, and a wavefront that drew several full ones was the launch's length (7B
// on 4x8, whole items handed out in turn: 0.53 ms at one wavefront per SIMD on average).  The list
// is in tile order; each XCD draws from its eighth of it, then from the next ones', and the next
// draw is on its way while a unit is worked on.
template <bool kResolve, bool kSamples, bool kInLds>
__global__ __launch_bounds__(kReduceThreads, 3) void reduce_kernel(
    const MistProblem prob, const MistGroupDesc *__restrict__ groups, const double *__restrict__ row_terms,
    const double *__restrict__ stage_floor, const RatioList ratios, const ReduceTables tabs, int wave_pitch) {
  extern __shared__ double lds_rows[];
  constexpr int kWaves = kReduceThreads / 64;
  const int local_wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
  const uint32_t n_waves = gridDim.x * kWaves;
  if (kResolve && tabs.counter[kLogFull * kCounterPitch] == 0) return;
  HitLog log;
  auto work = [&](uint64_t word, uint64_t pairs) {
    const Item item(word);
    const int gi = item.group, tile_rel = item.tile, stage = item.stage;
    const MistGroupDesc *g = groups + gi;
    if constexpr (kSamples) {
      __shared__ SampleQueue lds_queues[kWaves];
      reduce_item_samples<kResolve>(prob, g, gi, tile_rel, stage, row_terms, stage_floor, ratios, tabs, pairs,
                                    &lds_queues[local_wave], log);
    } else
      reduce_item<kResolve, kInLds>(prob, g, gi, tile_rel, stage, row_terms, stage_floor, ratios.r[0], tabs, pairs,
                                    lds_rows + local_wave * wave_pitch, log);
  };
  const FlatQueue queue = flat_queue(tabs, 1);
  // Units enough for every wavefront, and not too long ones; a pair of several samples takes longer (30 samples
  // of one tensor-parallel size of the 7B plan: 64 pairs a unit 2.36 ms, 32 2.12, 16 2.09).  A unit costs some
  // 8 us of loads that wait for each other before its first pair, so that splits beyond what fills the chip cost:
  // 3700 items of 9 pairs (7B on 4x8) 1, 2, 3 and 4 halvings 68, 73, 111 and 189 us, 14800 of 10 (13B on 8x8) none to
  // three 180, 190, 267 and 386; 6200 of 26 (uniform-pp of 7B on 2x8), where a few long units would be the launch's
  // end, none to four 279, 207, 190, 195 and 273.  (The pairs' sum may wrap: any split is right.)
  uint32_t n_pairs = tabs.counter[(kQueueShards + lane) * kCounterPitch + kOpenPairs];
  for (int k = 32; k > 0; k >>= 1) n_pairs += (uint32_t)__shfl_xor((int)n_pairs, k);
  n_pairs = (uint32_t)from_lane((int)n_pairs, 0);
  int split = kSamples ? 2 : 0;
  for (uint64_t units; split < 4; ++split) {
    units = (uint64_t)queue.total << split;
    if (units >= n_waves * 2 && (units >= n_waves * 8 || n_pairs <= 12 * units)) break;
  }
  const uint64_t units = (uint64_t)queue.total << split;
  if (kResolve) {  // handed out in turn
    for (uint64_t u = (uint64_t)blockIdx.x * kWaves + local_wave; u < units; u += n_waves) {
      const int64_t at = queue.at((uint32_t)(u >> split), tabs.capacity);
      const uint64_t pairs = from_lane((uint64_t)tabs.open_pairs[at], 0) & (every_pair(split) << (u & ((1u << split) - 1u)));
      if (pairs != 0) work(from_lane((uint64_t)tabs.opened[at], 0), pairs);
    }
    return;
  }
  for (int k = 0; k < kNumXcd; ++k) {
    const int part = ((int)blockIdx.x + k) % kNumXcd;
    const uint32_t first = (uint32_t)(units * part / kNumXcd), n = (uint32_t)(units * (part + 1) / kNumXcd) - first;
    uint32_t *drawn = tabs.counter + (3 * kQueueShards + part) * kCounterPitch;
    if (k > 0 && *drawn >= n) continue;
    auto draw = [&]() {
      uint32_t u = 0;
      if (lane == 0) u = atomicAdd(drawn, 1u);
      return u;
    };
    uint32_t ahead = draw();
    for (;;) {
      const uint32_t u = (uint32_t)from_lane((int)ahead, 0);
      if (u >= n) break;
      ahead = draw();
      const int64_t at = queue.at((first + u) >> split, tabs.capacity);
      const uint64_t pairs = tabs.open_pairs[at] & every_pair(split) << ((first + u) & ((1u << split) - 1u));
      const uint64_t word = tabs.opened[at];
      if (from_lane(pairs, 0) != 0) work(from_lane(word, 0), from_lane(pairs, 0));
    }
  }
  log.close(tabs);
}

// ---- resolve ----
// The lowest row of every minimum, from the log; a wavefront a chunk at a time, its four loads in flight together.
// Bound by the scattered reads of minima and atomics on rows.  (The items in which a row had reached a minimum gone
// through again, where the pair's minima had changed: 30 samples of one tensor-parallel size of the 7B plan 0.58 ms
// with the list of those items, now 0.08; of 7B on 1x8 0.15 and 0.012; one sample, 70B on 32x8 0.53 and 0.05, 13B on
// 4x8 0.12 and 0.017.  By the registers of the reduce kernel, three wavefronts a SIMD and two loads: 0.38 instead of
// 0.08.  What the log costs the reduce launch is within its spread.)
__global__ __launch_bounds__(kReduceThreads) void resolve_kernel(const ReduceTables tabs) {
  constexpr int kWaves = kReduceThreads / 64, kAtOnce = kLogChunk / 64;
  if (tabs.counter[kLogFull * kCounterPitch] != 0) return;  // reduce_kernel<true, ..> goes through everything
  const uint32_t n_chunks = tabs.counter[kLogTaken * kCounterPitch];
  const int lane = threadIdx.x & 63;
  for (uint32_t chunk = (uint32_t)__builtin_amdgcn_readfirstlane((int)(blockIdx.x * kWaves + (threadIdx.x >> 6)));
       chunk < n_chunks; chunk += gridDim.x * kWaves) {
    const int n = (int)tabs.log_count[chunk];
    const Hit *__restrict__ log = tabs.log + (int64_t)chunk * kLogChunk;
    Hit hit[kAtOnce];
    double best[kAtOnce];
#pragma unroll
    for (int i = 0; i < kAtOnce; ++i) hit[i] = log[min(i * 64 + lane, n - 1)];
#pragma unroll
    for (int i = 0; i < kAtOnce; ++i) best[i] = tabs.best[hit[i].cell];
#pragma unroll
    for (int i = 0; i < kAtOnce; ++i)
      if (i * 64 + lane < n && best[i] == hit[i].cost) atomicMin(tabs.row + hit[i].cell, hit[i].row);
  }
}

// Rows offered in ascending order: the first of equal costs stays (pareto.py:134-142 as written).
__device__ __forceinline__ void take_first(double &best, int32_t &best_row, bool feasible,
                                           double cost, int32_t row) {
  const bool better = feasible && cost < best;
  best = better ? cost : best;
  best_row = better ? row : best_row;
}

// ------------------------------------------------------------------------------------------
// Kernel 2x: the same reduction with every cell evaluated.  No seeds, no summaries, no bounds: each
// (row, l, c) goes through the latency model and the memory model, and each of its p values
// through the reference's feasibility test and the (cost, row) comparison.  This is the work the
// reference's formulas describe cell by cell; the pruned launches above must produce the same
// tables (tests) and are measured against it.  Workgroup = (row chunk, tile, p tile) of the
// filter launch's decomposition; it leaves its minima in a slab of its own, and
// combine_slabs_kernel takes the slabs into the table of minima, which finalize_kernel reads.
// ------------------------------------------------------------------------------------------
constexpr int kLdsRowStride = MIST_ROW_TERMS + 1;  // odd number of doubles: lanes reading the
                                                   // same term of different rows hit different banks
template <bool kFirstTile>
__device__ __forceinline__ void exhaustive_block(
    const MistProblem &prob, const MistGroupDesc *__restrict__ g, int64_t row_begin,
    int64_t row_end, int p_tile, int lc_tile, const double *__restrict__ row_terms, double ratio,
    double *lds_terms, int32_t *lds_row, double *__restrict__ out_cost,
    int32_t *__restrict__ out_index) {
  const int L = prob.num_layers;
  const int n_pairs = L * (L + 1) / 2 + L;
  const int pair_idx = lc_tile * MIST_LC_TILE + threadIdx.x;
  const bool active = pair_idx < n_pairs;
  const PairIndex pc = decode_pair(active ? pair_idx : 0);
  const int l = pc.l, c = pc.c;
  const int p0 = p_tile * MIST_P_TILE;
  const int n_tile = active ? min(MIST_P_TILE, g->num_p - p0) : 0;
  const GroupConsts k = group_consts(g);
  const double cap = prob.mem_cap_mb;
  const double G64 = (double)g->grad_accum;
  const float G32 = (float)g->grad_accum;
  const double pre_saved = g->pre_saved, pre_sas = g->pre_states_and_saved;

  double best_b[MIST_P_TILE], best_p[MIST_P_TILE];
  int32_t row_b[MIST_P_TILE], row_p[MIST_P_TILE];
  double best_post = INFINITY, best_pp = INFINITY;
  int32_t row_post = -1, row_pp = -1;
#pragma unroll
  for (int j = 0; j < MIST_P_TILE; ++j) {
    best_b[j] = best_p[j] = INFINITY;
    row_b[j] = row_p[j] = -1;
  }
  const double *__restrict__ src = row_terms + g->row_offset * MIST_ROW_TERMS;
  for (int64_t base = row_begin; base < row_end; base += kStageRows) {
    const int n_stage = (int)min((int64_t)kStageRows, row_end - base);
    __syncthreads();
    // Rows are visited in the REFERENCE's order (the chunk is a range of row numbers, gathered
    // from wherever the workspace order put them; lane = row for the index arithmetic), so that
    // within a chunk a strict "<" keeps the first of equal costs like the reference's scan does.
    lds_row[threadIdx.x] = (int32_t)position_of_row(g, min(base + threadIdx.x, row_end - 1));
    __syncthreads();
    const double2 *__restrict__ src2 = reinterpret_cast<const double2 *>(src);
    for (int i = threadIdx.x; i < n_stage * (MIST_ROW_TERMS / 2); i += MIST_LC_TILE) {
      const int r = i / (MIST_ROW_TERMS / 2), c2 = i % (MIST_ROW_TERMS / 2);
      const double2 v = src2[(int64_t)lds_row[r] * (MIST_ROW_TERMS / 2) + c2];
      lds_terms[r * kLdsRowStride + 2 * c2] = v.x;
      lds_terms[r * kLdsRowStride + 2 * c2 + 1] = v.y;
    }
    __syncthreads();
    if (!active) continue;
    for (int r = 0; r < n_stage; ++r) {
      const double *t = lds_terms + r * kLdsRowStride;
      const int32_t row = (int32_t)(base + r);
      const CellLatency lat = cell_latency<kFirstTile>(t, l, c, k);
      const LaneMemory mem = cell_memory(t, l, c);
      // objectives r * x + y (pareto.py:138): base with y = float32 delta / G in float32
      // (batched_module_analyzer.py:2815), the others in float64 (:2898-2903, 3002-3007, 3084-3089)
      const double cost_base = ratio * (double)lat.x + (double)(lat.d / G32);
      const double cost_pre = ratio * lat.sp + lat.dpre / G64;
      // Every slot through both feasibility tests (:2805-2812, 2893-2897), straight-line: the two
      // tests share the peaks of their p, and nothing is skipped by a branch (a lane whose tile
      // ends early only masks the update).
#pragma unroll
      for (int j = 0; j < MIST_P_TILE; ++j) {
        double peak_f, peak_b;
        mem.peaks(p0 + j, peak_f, peak_b);
        const bool fits_base = fmax(peak_f, peak_b) * mem.mf_base <= cap;
        const double pre_p = (double)(p0 + j) * pre_saved;
        const bool fits_pre = fmax(pre_p + peak_f + pre_sas, pre_p + peak_b + pre_sas) * mem.mf_pp <= cap;
        const bool live = j < n_tile;
        take_first(best_b[j], row_b[j], live & fits_base, cost_base, row);
        take_first(best_p[j], row_p[j], live & fits_pre, cost_pre, row);
      }
      if (kFirstTile) {  // last stage / single stage, p == 0 only (:2946-3106)
        double peak_f, peak_b;
        mem.peaks(0, peak_f, peak_b);
        const double f_in = mem.fwd_states + g->post_states + mem.mod_saved + g->post_fwd_peak + mem.gcb;
        const double b_in = mem.bwd_states + g->post_states + mem.mod_saved + g->post_bwd_peak +
                            (c == 0 ? t[MIST_T_RD] : 0.0) + mem.gcb;
        const double pf_post = fmax(f_in, peak_f + g->post_states);
        const double pb_post = fmax(b_in, peak_b - mem.out + g->post_states) + g->post_output;
        const bool ok_post = fmax(pf_post, pb_post) * mem.mf_pp <= cap;
        const double pf_pp = pf_post + g->pre_states + g->pre_saved;
        const double pb_pp = pb_post + g->pre_states + g->pre_saved;
        const bool ok_pp = fmax(pf_pp, pb_pp) * t[MIST_T_MF] <= cap;
        take_first(best_post, row_post, ok_post, ratio * lat.spost + lat.dpost / G64, row);
        take_first(best_pp, row_pp, ok_pp, ratio * lat.spp + lat.dpp / G64, row);
      }
    }
  }
#pragma unroll
  for (int j = 0; j < MIST_P_TILE; ++j) {
    out_cost[j * MIST_LC_TILE + threadIdx.x] = best_b[j];
    out_index[j * MIST_LC_TILE + threadIdx.x] = row_b[j];
    out_cost[(MIST_P_TILE + j) * MIST_LC_TILE + threadIdx.x] = best_p[j];
    out_index[(MIST_P_TILE + j) * MIST_LC_TILE + threadIdx.x] = row_p[j];
  }
  out_cost[(2 * MIST_P_TILE) * MIST_LC_TILE + threadIdx.x] = best_post;
  out_index[(2 * MIST_P_TILE) * MIST_LC_TILE + threadIdx.x] = row_post;
  out_cost[(2 * MIST_P_TILE + 1) * MIST_LC_TILE + threadIdx.x] = best_pp;
  out_index[(2 * MIST_P_TILE + 1) * MIST_LC_TILE + threadIdx.x] = row_pp;
}

#ifndef MIST_EXHAUSTIVE_MIN_WAVES
#define MIST_EXHAUSTIVE_MIN_WAVES 2
#endif
__global__ __launch_bounds__(MIST_LC_TILE, MIST_EXHAUSTIVE_MIN_WAVES) void eval_reduce_exhaustive_kernel(
    const MistProblem prob, const MistGroupDesc *__restrict__ groups, int n_groups,
    const int32_t *__restrict__ block_prefix, int n_blocks, const double *__restrict__ row_terms,
    double ratio, double *__restrict__ partial_cost, int32_t *__restrict__ partial_index) {
  __shared__ double lds_terms[kStageRows * kLdsRowStride];
  __shared__ int32_t lds_row[kStageRows];
  const int block = xcd_run_block(blockIdx.x);
  if (block >= n_blocks) return;
  int local_block;
  const MistGroupDesc *g = find_group(groups, block_prefix, n_groups, block, &local_block);
  const int n_tiles = g->n_lc_tiles * g->n_p_tiles;
  const int chunk = local_block / n_tiles, tile = local_block % n_tiles;
  const int64_t row_begin = (int64_t)chunk * g->rows_per_chunk;
  const int64_t row_end = min(row_begin + (int64_t)g->rows_per_chunk, g->n_rows);
  const int p_tile = tile % g->n_p_tiles, lc_tile = g->lc_tile_begin + tile / g->n_p_tiles;
  const int64_t slab = (int64_t)kSlots * MIST_LC_TILE;
  if (p_tile == 0)
    exhaustive_block<true>(prob, g, row_begin, row_end, p_tile, lc_tile, row_terms, ratio,
                           lds_terms, lds_row, partial_cost + block * slab, partial_index + block * slab);
  else
    exhaustive_block<false>(prob, g, row_begin, row_end, p_tile, lc_tile, row_terms, ratio,
                            lds_terms, lds_row, partial_cost + block * slab, partial_index + block * slab);
}

// The pipeline a group offers to the stage-cost estimates: S stages of L / S layers on the group's
// mesh (PipelineLayers where the layers do not divide), or 0 when the devices do not, the group has too few
// pre-saved micro-batch values, or the caller's search does not go that deep.  A power of two of devices has a
// pipeline that divides its layers, one stage on all of them, and the others seldom say more (8 of 189 such calls
// got a lower estimate, 0.8 % of their time): those are not gone through.
__device__ __forceinline__ int incumbent_stage_count(const MistProblem &prob,
                                                     const MistGroupDesc *__restrict__ g) {
  const int L = prob.num_layers, D = prob.incumbent_num_devices;
  const int nm = g->num_nodes * g->num_gpus_per_node;
  if (nm <= 0 || D % nm != 0) return 0;
  const int S = D / nm;
  if (S < 1 || S > L || S - 1 >= g->num_p) return 0;
  if (L % S != 0 && (D & (D - 1)) == 0 && prob.incumbent_close != kCloseAssignment) return 0;
  // (the per-mesh search goes up to min(devices, layers) / 2 stages, inter_tuning.py:279-281)
  if (prob.incumbent_ckpt_rule == 0 && S > (D < L ? D : L) / 2) return 0;
  return S;
}

// Its layers: the first L % S stages behind the first one, which holds the pre layer and the most micro-batches,
// have one more.  (Of 14 nodes and 57 layers or 5 and 23, no mesh has stages that divide both; such searches
// ran without an estimate, 39 of 232 calls: 70B, 57 layers on 14x8 10164 -> 2598 us, 13B, 23 on 5x8 1784 -> 1050.)
struct PipelineLayers {
  int each, extra;
  __device__ __forceinline__ PipelineLayers(int layers, int stages) : each(layers / stages), extra(layers % stages) {}
  __device__ __forceinline__ int of(int stage) const { return each + (stage >= 1 && stage <= extra ? 1 : 0); }
  __device__ __forceinline__ int end(int stage) const { return (stage + 1) * each + min(stage, extra) - 1; }  // last layer
};

// What a group's stage costs can be used for, from the bounds of its rows and of the other meshes' of its table
// row (neighbours in the list).  The search that reads the tables looks for pipelines of D devices and L layers
// whose stages cost no more than bound(G).
//  - A stage of l layers on d devices leaves L - l layers to D - d devices.  Some stage among those has at least
//    its share of them, and no mesh takes more than `load` layers a device at a cost up to bound(G): what leaves
//    more is in no such pipeline, and no stage of the table row is if all layers are more than D devices take.
//  - The most expensive stage of every pipeline costs at least what the cheapest mesh takes for its share of all
//    layers.  That search reads stage costs as threshold candidates from kExactMargins below the smallest largest
//    cost on: of what is in no pipeline, a minimum below that is as good as any other value below it.
// So a pair of fewer than `first` layers is left alone once its minimum is below `low`: 70 - 80 % of the pairs with
// a minimum up to bound(G) on clusters of a power of two of nodes, 33 - 65 % on others (a mesh of all devices is
// used with all layers only, one of half of them with close to half).  Calls, us: 7B on 4x8 1180 -> 1065, 13B on
// 8x8 1920 -> 1615, 22B on 16x8 9000 -> 7190, 70B on 32x8 5720 -> 4290, 1.3B on 1x2 the same.  (Closed in the seeds
// already, by about the same from the first estimate: they spend their time on the first rows of a pair; 70B 4290
// -> 4230, 13B uniform-device-pp 1470 -> 1600.)
// (Where a row may cost less the more layers it has - a negative share of the first micro-batch - nothing is closed,
// and neither is without an estimate: bound(G) is infinite then, but `low` would not be.)
// The workgroup `reach` is formed by; all its threads.
struct ReachBounds {
  double per_layer, rest;
  int row, devices;
};
__device__ __forceinline__ void form_reach(const MistProblem &prob, const MistGroupDesc *__restrict__ groups, int n_groups,
                                           ReachBounds *bounds, GroupReach *reach) {
  const double L = (double)prob.num_layers, D = (double)prob.incumbent_num_devices;
  const double incumbent = load_at_agent(prob.stage_cost_incumbent);
  for (int i = threadIdx.x; i < n_groups; i += blockDim.x)
    bounds[i] = ReachBounds{load_at_agent(&reach[i].per_layer), load_at_agent(&reach[i].rest), groups[i].g_index,
                            groups[i].num_nodes * groups[i].num_gpus_per_node};
  __syncthreads();
  for (int gi = threadIdx.x; gi < n_groups; gi += blockDim.x) {
    const double bound = incumbent * (1.0 / (double)groups[gi].grad_accum) * (1.0 + kIncumbentSlack);
    double load = 0.0, cheapest = INFINITY;  // layers a device takes at most, the smallest largest stage cost
    auto add = [&](const ReachBounds &r) {
      const double d = (double)r.devices, share = ceil(L * d / D - 1e-9);
      if (!(r.per_layer > 0.0)) {
        load = L;
        cheapest = -INFINITY;
        return;
      }
      if (r.rest <= bound) load = fmax(load, fmin(L, floor((bound - r.rest) / r.per_layer * (1.0 + 1e-9)) + 2.0) / d);
      cheapest = fmin(cheapest, r.rest + fmax(share - 2.0, 0.0) * r.per_layer);
    };
    const int row = bounds[gi].row;
    for (int i = gi; i >= 0 && bounds[i].row == row; --i) add(bounds[i]);
    for (int i = gi + 1; i < n_groups && bounds[i].row == row; ++i) add(bounds[i]);
    reach[gi].cutoff = load * D * (1.0 + 1e-9) < L ? -INFINITY : bound;
    reach[gi].first = (int)fmax(ceil(L - load * (D - (double)bounds[gi].devices) * (1.0 + 1e-9)), 0.0);
    reach[gi].low = cheapest * (1.0 - 1e-6) - mist::kExactMargins * mist::window_margin(cheapest);
    if (!(incumbent < INFINITY)) {  // (no estimate: what reads the tables takes them for complete)
      reach[gi].first = 0;
      reach[gi].low = -INFINITY;
    }
  }
}

// Cost of the best pipeline of equal stages on equal meshes that the seeds allow
// (sample 0 of a call with one sample, whose objective is the stage cost): group (G, mesh (n, m))
// offers S = devices / (n m) stages of about L / S layers each, the first one from the with_pre table
// at S - 1 pre-saved micro-batches, the last one from the with_post table, those between from
// the base table, a single one from the no_pp table, each at its cheapest admissible ckpt count
// (rule of the caller's search, MistProblem.incumbent_ckpt_rule); the cost is the sum of the
// stage costs + (G - 1) x the largest, as the search forms it (inter_tuning.py:342).  Seeds are
// minima over some rows, so the finished tables hold no larger values; the search that reads
// them returns no more than this unless its scan never tries the thresholds of that pipeline
// (a single-stage cost is no threshold candidate of the reference, and its gap rule drops
// some), which is why the caller checks its result against the bound that was used.
// Workgroup = group, its wavefronts take the stages in turn; lowers *incumbent.  With MistProblem.incumbent_close
// the last workgroup to end forms the records of all groups.
constexpr int kIncumbentWaves = 4;
__global__ __launch_bounds__(64 * kIncumbentWaves) void incumbent_kernel(
    const MistProblem prob, const MistGroupDesc *__restrict__ groups, const ReduceTables tabs) {
  const MistGroupDesc *g = groups + blockIdx.x;
  const int L = prob.num_layers, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const bool close = prob.incumbent_close == kCloseSearch;
  if (close && wave == 0) {
    static_assert(kSuperBlocks == 64, "a lane per workgroup of the summaries");
    const double *parts = tabs.reach_parts + ((int64_t)blockIdx.x * kSuperBlocks + lane) * 2;
    double per_layer = parts[0], rest = parts[1];
    for (int step = 32; step > 0; step >>= 1) {
      per_layer = fmin(per_layer, __shfl_xor(per_layer, step));
      rest = fmin(rest, __shfl_xor(rest, step));
    }
    if (lane == 0) {
      __hip_atomic_store(&tabs.reach[blockIdx.x].per_layer, per_layer, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __hip_atomic_store(&tabs.reach[blockIdx.x].rest, rest, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  }
  const int S = g->scout_stride > 0 ? incumbent_stage_count(prob, g) : 0;
  if (S == 0 && !close) return;
  const PipelineLayers layers(L, max(S, 1));
  const int P = g->num_p;
  // seed of a stage's (l, c) cell in slot `slot` (one sample; +inf where there is none)
  auto seed_of = [&](int slot, int l, int c) {
    const int pair = l * (l + 1) / 2 - 1 + c;
    const int lc_tile = pair / MIST_LC_TILE - g->lc_tile_begin;
    if (lc_tile < 0 || lc_tile >= g->n_lc_tiles) return (double)INFINITY;
    return tabs.best[g->cell_offset +
                     ((int64_t)lc_tile * MIST_LC_TILE + pair % MIST_LC_TILE) * slots_of(P) + slot];
  };
  // cheapest one over c = 0..c_last
  auto cheapest = [&](int slot, int l, int c_last) {
    double best = INFINITY;
    for (int c = threadIdx.x & 63; c <= c_last; c += 64) best = fmin(best, seed_of(slot, l, c));
    for (int step = 32; step > 0; step >>= 1) best = fmin(best, __shfl_xor(best, step));
    return best;
  };
  auto c_last_of = [&](int l, int end_layer) {
    return prob.incumbent_ckpt_rule == 0 ? min(l, L - end_layer) : l;
  };
  __shared__ double wave_sum[kIncumbentWaves], wave_largest[kIncumbentWaves];
  double sum = 0.0, largest = 0.0;
  for (int s = wave; s < S; s += kIncumbentWaves) {
    const int p = S - 1 - s, l = layers.of(s);
    int slot;
    if (S == 1) slot = 2 * P + 1;
    else if (s == 0) slot = P + p;
    else if (s == S - 1) slot = 2 * P;
    else slot = p;
    // (rule 2: every layer of the stage checkpointed)
    const double cost = prob.incumbent_ckpt_rule == 2 ? seed_of(slot, l, l) : cheapest(slot, l, c_last_of(l, layers.end(s)));
    sum += cost;
    largest = fmax(largest, cost);
  }
  if (lane == 0) {
    wave_sum[wave] = sum;
    wave_largest[wave] = largest;
  }
  __syncthreads();
  sum = 0.0;
  largest = 0.0;
  for (int w = 0; w < kIncumbentWaves; ++w) {
    sum += wave_sum[w];
    largest = fmax(largest, wave_largest[w]);
  }
  const double total = sum + (double)(g->grad_accum - 1) * largest;
  // (a pipeline's cost, unlike an objective of another alpha, is not negative: its bits order)
  if (threadIdx.x == 0 && S > 0 && total >= 0.0 && total < INFINITY)
    atomicMin(reinterpret_cast<unsigned long long *>(prob.stage_cost_incumbent),
              (unsigned long long)__double_as_longlong(total));
  if (!close) return;
  __shared__ bool last;
  __threadfence();
  if (threadIdx.x == 0)
    last = atomicAdd(tabs.counter + kGroupsDone * kCounterPitch, 1u) == gridDim.x - 1;
  __syncthreads();
  if (!last) return;
  __threadfence();
  extern __shared__ double lds_bounds[];
  form_reach(prob, groups, gridDim.x, reinterpret_cast<ReachBounds *>(lds_bounds), tabs.reach);
}

// First estimate of the same pipeline cost, formed before the seeds so that the seed launch
// can already leave out stage costs the caller's search cannot use.  Each group evaluates about
// kEstimateRows of its gathered rows - every parallelism row of every scout pair without
// activation / optimizer offloading first, then with the next ratios - for the layer count
// of its stages (two, where S does not divide L) and every ckpt count, exactly as the tables would (same latency and memory code as
// the evaluate-every-cell kernel, same cells kept: c == l - 1 only at p == 0 of the base /
// with_pre tables), and keeps per stage of the pipeline the cheapest feasible cost.  Minima over
// fewer rows than the seeds see, so the estimate is no smaller than theirs.
// Grid (kEstimateSplit, group); workgroup k writes its S minima to doubles [k S, (k + 1) S) of
// the group's minima (the seed launch fills them afterwards).
constexpr int kEstimateSplit = 16;
constexpr int kEstimateRows = 1024;
constexpr int kEstimateMaxStages = 256;
static_assert(kEstimateSplit <= MIST_LC_TILE, "S <= num_p: the partial minima of a group fit one tile of its minima");
__device__ __forceinline__ bool estimate_runs(const MistProblem &prob, const MistGroupDesc *g, int *stages) {
  if (g->scout_stride <= 0 || g->n_lc_tiles <= 0) return false;
  *stages = incumbent_stage_count(prob, g);
  return *stages > 0 && *stages <= kEstimateMaxStages;
}

// For an assignment (kAssignment) stages are chosen by stable + delta / G; the smallest float32 of that and its item
// are kept, whose latencies the combining launch forms again.
struct EstimateItem {
  int l, c;
  int64_t row;  // gathered
};
struct EstimateItems {
  int n_cells, n_tail, n_par;
  int64_t per_pair, per_tail, n_tails;
  __device__ __forceinline__ EstimateItems(const MistGroupDesc *g, const PipelineLayers &layers) {
    n_tail = g->n_oo * g->n_ao;
    n_par = g->n_par;
    per_pair = (int64_t)g->n_par * n_tail;
    per_tail = (int64_t)g->n_par * max(g->scout_stride, 1);
    n_tails = min((int64_t)n_tail, max((int64_t)1, (int64_t)kEstimateRows / per_tail));
    n_cells = layers.each + 1 + (layers.extra > 0 ? layers.each + 2 : 0);  // (layers, ckpt) of a row
  }
  __device__ __forceinline__ int64_t count() const { return per_tail * n_tails * n_cells; }
  __device__ __forceinline__ EstimateItem at(int64_t item, const PipelineLayers &layers) const {
    const int cell = (int)(item % n_cells);
    const bool longer = cell > layers.each;
    EstimateItem i;
    i.l = longer ? layers.each + 1 : layers.each;
    i.c = longer ? cell - i.l : cell;
    const int64_t q = item / n_cells, tail = q / per_tail, rest = q - tail * per_tail;
    const int64_t pair = rest / n_par, par = rest - pair * n_par;
    i.row = pair * per_pair + par * n_tail + tail;
    return i;
  }
};
template <bool kAssignment>
__global__ __launch_bounds__(256) void estimate_stage_minima_kernel(
    const MistProblem prob, const MistGroupDesc *__restrict__ groups,
    const double *__restrict__ row_terms, double ratio, double *__restrict__ partial_cost, double *gather_floor) {
  const MistGroupDesc *g = groups + blockIdx.y;
  // What the seed launch wants next, beside the estimate: it reads the gathered rows again and the seeds wait
  // for it.  (us, rows estimated alone -> with it; seeds reading every row -> by these bounds: 7B on 4x8 86 -> 97,
  // 285 -> 268; 13B on 8x8 116 -> 138, 553 -> 517; 22B on 16x8 198 -> 325, 5815 -> 4754; 70B on 32x8 239 -> 276,
  // 1972 -> 1269.  From the gathered rows to the filter that is no gain up to 7B on 4x8, 450 -> 465.)
  if (blockIdx.x >= kEstimateSplit) {
    gather_floors(prob, g, blockIdx.y, row_terms, ratio, gather_floor, blockIdx.x - kEstimateSplit, kGatherBlocks);
    return;
  }
  int S;
  if (!estimate_runs(prob, g, &S)) return;
  const int L = prob.num_layers, rule = prob.incumbent_ckpt_rule;
  const PipelineLayers layers(L, S);
  __shared__ unsigned long long stage_min[kEstimateMaxStages];
  const unsigned long long kInf = (unsigned long long)__double_as_longlong((double)INFINITY);
  for (int st = threadIdx.x; st < S; st += blockDim.x) stage_min[st] = kInf;
  __syncthreads();
  const EstimateItems items(g, layers);
  const int64_t n_items = items.count();
  const GroupConsts k = group_consts(g);
  const double cap = prob.mem_cap_mb;
  const double G64 = (double)g->grad_accum;
  const float G32 = (float)g->grad_accum;
  const double *__restrict__ src = row_terms + g->row_offset * MIST_ROW_TERMS;
  int64_t item = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  auto offer = [&](int st, bool ok, double cost) {
    // (stage costs, unlike objectives of another alpha, are not negative: their bits order)
    if (ok && cost >= 0.0 && cost < INFINITY)
      atomicMin(&stage_min[st], kAssignment ? (unsigned long long)__float_as_uint((float)cost) << 32 | (uint32_t)item
                                            : (unsigned long long)__double_as_longlong(cost));
  };
  for (; item < n_items; item += (int64_t)kEstimateSplit * blockDim.x) {
    const EstimateItem i = items.at(item, layers);
    const int l = i.l, c = i.c;
    const bool longer = l > layers.each;
    if (rule == 2 && c != l) continue;  // every layer of a stage checkpointed
    if (c == l - 1) continue;  // kept at p == 0 of base / with_pre only, which no stage below reads
    const double *__restrict__ t =
        src + gathered_position(g, (uint32_t)i.row) * MIST_ROW_TERMS;
    const CellLatency lat = cell_latency<true>(t, l, c, k);
    const LaneMemory mem = cell_memory(t, l, c);
    // largest ckpt count of the stage that ends with layer end_layer (rule of the caller's search)
    auto c_last = [&](int st) { return rule == 0 ? min(l, L - layers.end(st)) : l; };
    double peak_f, peak_b;
    mem.peaks(0, peak_f, peak_b);
    const double f_in = mem.fwd_states + g->post_states + mem.mod_saved + g->post_fwd_peak + mem.gcb;
    const double b_in = mem.bwd_states + g->post_states + mem.mod_saved + g->post_bwd_peak +
                        (c == 0 ? t[MIST_T_RD] : 0.0) + mem.gcb;
    const double pf_post = fmax(f_in, peak_f + g->post_states);
    const double pb_post = fmax(b_in, peak_b - mem.out + g->post_states) + g->post_output;
    if (S == 1) {  // single stage: the no_pp table
      const double pf_pp = pf_post + g->pre_states + g->pre_saved;
      const double pb_pp = pb_post + g->pre_states + g->pre_saved;
      offer(0, c <= c_last(0) && fmax(pf_pp, pb_pp) * t[MIST_T_MF] <= cap,
            ratio * lat.spp + lat.dpp / G64);
      continue;
    }
    // first stage: with_pre table at S - 1 pre-saved micro-batches
    offer(0, !longer && c <= c_last(0) && mem.feasible_pre(S - 1, cap, g->pre_saved, g->pre_states_and_saved),
          ratio * lat.sp + lat.dpre / G64);
    // last stage: with_post table
    offer(S - 1, l == layers.of(S - 1) && c <= c_last(S - 1) && fmax(pf_post, pb_post) * mem.mf_pp <= cap,
          ratio * lat.spost + lat.dpost / G64);
    // stages between: base table at S - 1 - st pre-saved micro-batches
    const double cost_base = ratio * (double)lat.x + (double)(lat.d / G32);
    // (of l layers: stages 1 .. extra have the extra layer)
    const int st_end = longer ? min(layers.extra + 1, S - 1) : S - 1;
    for (int st = longer ? 1 : layers.extra + 1; st < st_end; ++st)
      offer(st, c <= c_last(st) && mem.feasible_base(S - 1 - st, cap), cost_base);
  }
  __syncthreads();
  double *out = partial_cost + g->cell_offset + (int64_t)blockIdx.x * S;
  for (int st = threadIdx.x; st < S; st += blockDim.x)
    out[st] = __longlong_as_double((long long)stage_min[st]);
}

// Objective of the assignment that a group's chosen stages are (inter_tuning_mip.py:317-400) into *incumbent.
__global__ __launch_bounds__(64) void estimate_assignment_kernel(const MistProblem prob, const MistGroupDesc *__restrict__ groups,
                                                                 const double *__restrict__ row_terms,
                                                                 const double *__restrict__ partial_cost) {
  const MistGroupDesc *g = groups + blockIdx.x;
  int S;
  if (!estimate_runs(prob, g, &S)) return;
  const PipelineLayers layers(prob.num_layers, S);
  const EstimateItems items(g, layers);
  const GroupConsts k = group_consts(g);
  const unsigned long long *in = reinterpret_cast<const unsigned long long *>(partial_cost + g->cell_offset);
  __shared__ double stable[kEstimateMaxStages], delta[kEstimateMaxStages];
  for (int st = threadIdx.x; st < S; st += 64) {
    unsigned long long best = ~0ull;
    for (int part = 0; part < kEstimateSplit; ++part) best = min(best, in[(int64_t)part * S + st]);
    double x = INFINITY, d = INFINITY;
    if (best < (unsigned long long)__double_as_longlong((double)INFINITY)) {
      const EstimateItem i = items.at((int64_t)(uint32_t)best, layers);
      const double *__restrict__ t =
          row_terms + (g->row_offset + gathered_position(g, (uint32_t)i.row)) * MIST_ROW_TERMS;
      const CellLatency lat = cell_latency<true>(t, i.l, i.c, k);
      x = S == 1 ? lat.spp : st == 0 ? lat.sp : st == S - 1 ? lat.spost : (double)lat.x;
      d = S == 1 ? lat.dpp : st == 0 ? lat.dpre : st == S - 1 ? lat.dpost : (double)lat.d;
    }
    stable[st] = fmax(x, 0.0);
    delta[st] = fmax(d, 0.0);
  }
  __syncthreads();
  if (threadIdx.x != 0) return;
  double sum = 0.0, largest = 0.0, late = 0.0;
  for (int st = 0; st < S; ++st) {
    late = fmax(late, delta[st] - sum);
    sum += stable[st];
    largest = fmax(largest, stable[st]);
  }
  const double total = (double)(g->grad_accum - 1) * largest + sum + late;
  if (total >= 0.0 && total < INFINITY)
    atomicMin(reinterpret_cast<unsigned long long *>(prob.stage_cost_incumbent), (unsigned long long)__double_as_longlong(total));
}

// Layers a stage of a group may have in an assignment whose objective is no more than the estimate and some room
// ((G - 1) max T + sum T and what is not negative): with l of them one of the other stages has at least its share of
// the rest, and stable latencies are no less than the bounds of the group's rows.  Most groups keep the even number
// of layers alone, or nothing: 30 samples of 7B on 4x8 2870 -> 2190 us, on 1x8 (small cards) 1390 -> 1265, 13B on 8x8
// 2980 -> 1700.  (With the seeds of all pairs beside the summaries, as without an estimate: 7B on 4x8 2280, 1x8 1264.
// Of 190 drawn calls all had an optimum between 0.93 and 1.0000 times the estimate.)
__global__ __launch_bounds__(64) void assignment_reach_kernel(const MistProblem prob, const MistGroupDesc *__restrict__ groups,
                                                              const ReduceTables tabs) {
  static_assert(kSuperBlocks == 64, "a lane per workgroup of the summaries");
  const int gi = blockIdx.x, lane = threadIdx.x, L = prob.num_layers, D = prob.incumbent_num_devices;
  const MistGroupDesc *g = groups + gi;
  const double *parts = tabs.reach_parts + ((int64_t)gi * kSuperBlocks + lane) * 2;
  double per_layer = parts[0], rest = parts[1];
  for (int step = 32; step > 0; step >>= 1) {
    per_layer = fmin(per_layer, __shfl_xor(per_layer, step));
    rest = fmin(rest, __shfl_xor(rest, step));
  }
  const double most = *prob.stage_cost_incumbent * (1.0 + kIncumbentSlack), more = (double)(g->grad_accum - 1);
  const int nm = g->num_nodes * g->num_gpus_per_node, S = D / nm;
  const bool bounded = D % nm == 0 && per_layer > 0.0 && most < INFINITY;
  auto least = [&](int layers) { return rest + (double)max(layers - 2, 0) * per_layer; };
  int first = L + 1, last = 0;
  for (int l = 1 + lane; l <= L; l += 64) {
    bool in = true;
    if (bounded && S == 1) in = l == L && least(L) * (more + 1.0) * (1.0 - 1e-6) <= most;
    else if (bounded) {
      const int others = S - 1, left = L - l;
      const double largest = fmax(least(l), least((left + others - 1) / others));
      const double sum = least(l) + (double)others * rest + (double)max(left - 2 * others, 0) * per_layer;
      in = left >= others && (more * fmax(largest, 0.0) + sum) * (1.0 - 1e-6) <= most;
    }
    if (!in) continue;
    first = min(first, l);
    last = max(last, l);
  }
  for (int step = 32; step > 0; step >>= 1) {
    first = min(first, __shfl_xor(first, step));
    last = max(last, __shfl_xor(last, step));
  }
  if (lane != 0) return;
  tabs.reach[gi].first = first;
  tabs.reach[gi].last = last;
}

// Sum of a group's stage minima + (G - 1) x the largest (inter_tuning.py:342) into *incumbent.
__global__ __launch_bounds__(64) void estimate_combine_kernel(
    const MistProblem prob, const MistGroupDesc *__restrict__ groups,
    const double *__restrict__ partial_cost) {
  const MistGroupDesc *g = groups + blockIdx.x;
  int S;
  if (!estimate_runs(prob, g, &S)) return;
  const double *in = partial_cost + g->cell_offset;
  double sum = 0.0, largest = 0.0;
  for (int st = threadIdx.x; st < S; st += 64) {
    double best = INFINITY;
    for (int k = 0; k < kEstimateSplit; ++k) best = fmin(best, in[(int64_t)k * S + st]);
    sum += best;
    largest = fmax(largest, best);
  }
  for (int step = 32; step > 0; step >>= 1) {
    sum += __shfl_xor(sum, step);
    largest = fmax(largest, __shfl_xor(largest, step));
  }
  const double total = sum + (double)(g->grad_accum - 1) * largest;
  if (threadIdx.x == 0 && total >= 0.0 && total < INFINITY)
    atomicMin(reinterpret_cast<unsigned long long *>(prob.stage_cost_incumbent),
              (unsigned long long)__double_as_longlong(total));
}

// Combines the chunk slabs of the evaluate-every-cell kernel into the minima tables (one sample):
// thread = (pair of a tile, slot of a p tile).
__global__ __launch_bounds__(256) void combine_slabs_kernel(
    const MistGroupDesc *__restrict__ groups, const int32_t *__restrict__ block_prefix,
    const double *__restrict__ slab_cost, const int32_t *__restrict__ slab_index, const ReduceTables tabs) {
  const int gi = blockIdx.y;
  const MistGroupDesc *g = groups + gi;
  const int n_tiles = g->n_lc_tiles * g->n_p_tiles, P = g->num_p;
  const int64_t slab = (int64_t)kSlots * MIST_LC_TILE;
  for (int tile = blockIdx.x; tile < n_tiles; tile += gridDim.x) {
    const int p_tile = tile % g->n_p_tiles, tile_rel = tile / g->n_p_tiles, p0 = p_tile * MIST_P_TILE;
    for (int e = threadIdx.x; e < (int)slab; e += blockDim.x) {
      const int kslot = e / MIST_LC_TILE, lane = e % MIST_LC_TILE, p = p0 + kslot % MIST_P_TILE;
      int slot;
      if (kslot >= 2 * MIST_P_TILE) {
        if (p_tile != 0) continue;
        slot = 2 * P + (kslot - 2 * MIST_P_TILE);
      } else if (p >= P) {
        continue;
      } else {
        slot = kslot < MIST_P_TILE ? p : P + p;
      }
      double best = INFINITY;
      int32_t best_row = -1;
      for (int ch = 0; ch < g->n_chunks; ++ch) {
        const int64_t at = ((int64_t)block_prefix[gi] + (int64_t)ch * n_tiles + tile) * slab + e;
        const int32_t row = slab_index[at];
        take_min(best, best_row, row >= 0, slab_cost[at], row);
      }
      const int64_t cell = g->cell_offset + ((int64_t)tile_rel * MIST_LC_TILE + lane) * slots_of(P) + slot;
      tabs.best[cell] = best;
      tabs.row[cell] = (uint32_t)best_row;
    }
  }
}

// ------------------------------------------------------------------------------------------
// Kernel 3: recompute the winners' stable / delta, scatter into the output tables.  The reduction
// left each row's cost at the slot of its own count: a p's winner is the lexicographic minimum of
// (cost, row) over the slots from it up.  Neighbouring p mostly share it, so a thread goes down the
// slots and reads and prices a winner's terms once.
// ------------------------------------------------------------------------------------------
// One (group, pair, variant) of the output.
struct FinalCell {
  double stable, delta;
  uint32_t priced;  // row they are of
  int64_t at, plane;  // element of p == 0, elements between p
  // Cells the reference never writes (batched_module_analyzer.py:3021-3023 rebinds the layer
  // mask inside the p == 0 branch, so it also governs base / with_pre for p >= 1; :3103).
  int n_p;  // values of p written
};
__device__ __forceinline__ FinalCell final_cell(const MistProblem &prob, const MistGroupDesc *__restrict__ g, int variant,
                                                PairIndex pc, int sample_at) {
  const int L = prob.num_layers, P1 = prob.p_dim, S = prob.sample_size, l = pc.l, c = pc.c;
  const int64_t gq = (int64_t)g->g_index * prob.num_mesh + g->q_index;
  FinalCell f;
  f.stable = f.delta = INFINITY;
  f.priced = ~0u;
  f.plane = (int64_t)L * (L + 1) * S;
  f.at = (variant == 3 ? gq * (L + 1) + c : ((variant < 2 ? gq * P1 : gq) * L + (l - 1)) * (L + 1) + c) * S + sample_at;
  f.n_p = variant < 2 ? (c == l - 1 ? 1 : g->num_p) : variant == 2 ? c != l - 1 : l == L && c != L - 1;
  return f;
}
__device__ __forceinline__ void write_final(FinalCell &f, const MistGroupDesc *__restrict__ g, int variant, PairIndex pc,
                                            const GroupConsts &k, const double *__restrict__ row_terms, uint32_t row,
                                            int p, const MistOutTables &tables, bool sparse) {
  const int64_t at = f.at + p * f.plane;
  if (sparse && row == ~0u) {  // (all that is read of such a cell)
    tables.index[variant][at] = -1;
    return;
  }
  if (row == ~0u) {
    f.stable = f.delta = INFINITY;
    f.priced = row;
  } else if (row != f.priced) {
    const double *t = row_terms + (g->row_offset + position_of_row(g, (int32_t)row)) * MIST_ROW_TERMS;
    const CellLatency lat = cell_latency<true>(t, pc.l, pc.c, k);
    if (variant == 0) { f.stable = (double)lat.x; f.delta = (double)lat.d; }
    else if (variant == 1) { f.stable = lat.sp; f.delta = lat.dpre; }
    else if (variant == 2) { f.stable = lat.spost; f.delta = lat.dpost; }
    else { f.stable = lat.spp; f.delta = lat.dpp; }
    f.priced = row;
  }
  tables.stable[variant][at] = f.stable;
  tables.delta[variant][at] = f.delta;
  tables.index[variant][at] = (int32_t)row;
}
// (row as left by the reduction: ~0 none)
__device__ __forceinline__ void take_lower(double &cost, uint32_t &row, double its_cost, uint32_t its_row) {
  row = its_cost < cost ? its_row : its_cost == cost ? min(row, its_row) : row;
  cost = fmin(cost, its_cost);
}

// One sample: workgroup = (tile, variant, group).  The slots of a pair lie side by side, the tables'
// last axis is c: kFinalSlots slots at a time are read with lane = (pair parity, slot), scanned, and
// left in LDS for the wavefronts to write with lane = pair.  (A thread per pair and variant that
// walked the slots in memory: 3.6 ms for the 70B plan on 256 GPUs, a line per read.)
constexpr int kFinalSlots = 32;
__global__ __launch_bounds__(256) void finalize_kernel(
    const MistProblem prob, const MistGroupDesc *__restrict__ groups, const double *__restrict__ row_terms,
    const ReduceTables tabs, int sample_at, MistOutTables tables) {
  __shared__ uint32_t winner[MIST_LC_TILE][kFinalSlots + 1];
  __shared__ double carry_cost[MIST_LC_TILE];
  __shared__ uint32_t carry_row[MIST_LC_TILE];
  const int L = prob.num_layers, n_pairs = L * (L + 1) / 2 + L;
  const MistGroupDesc *g = groups + blockIdx.z;
  const int tile_rel = blockIdx.x, variant = blockIdx.y, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (tile_rel >= g->n_lc_tiles) return;
  const int P = variant < 2 ? g->num_p : 1, n_slots = slots_of(g->num_p);
  const int first_pair = (g->lc_tile_begin + tile_rel) * MIST_LC_TILE;
  const bool active = first_pair + lane < n_pairs;
  const PairIndex pc = decode_pair(active ? first_pair + lane : 0);
  FinalCell f = final_cell(prob, g, variant, pc, sample_at);
  if (!active) f.n_p = 0;
  const GroupConsts k = group_consts(g);
  const int64_t first = g->cell_offset + (int64_t)tile_rel * MIST_LC_TILE * n_slots +
                        (variant < 2 ? variant * P : 2 * g->num_p + variant - 2);
  if (threadIdx.x < MIST_LC_TILE) {
    carry_cost[threadIdx.x] = INFINITY;
    carry_row[threadIdx.x] = ~0u;
  }
  for (int p0 = (P - 1) / kFinalSlots * kFinalSlots; p0 >= 0; p0 -= kFinalSlots) {
    __syncthreads();
    const int j = lane % kFinalSlots, p = p0 + j;
#pragma unroll 2
    for (int pair = wave * 2 + lane / kFinalSlots; pair < MIST_LC_TILE; pair += 8) {
      const PairIndex its = decode_pair(min(first_pair + pair, n_pairs - 1));
      const int np = its.c == its.l - 1 ? 1 : P;  // (later slots hold no minima)
      const int64_t cell = first + (int64_t)pair * n_slots + p;
      double cost = INFINITY;
      uint32_t row = ~0u;
      if (p < np) row = tabs.row[cell];
      // (no row at or above these slots: a minimum without one was not looked for)
      if (!__any(row != ~0u || carry_row[pair] != ~0u)) {
        winner[pair][j] = ~0u;
        continue;
      }
      if (p < np) cost = tabs.best[cell];
      for (int step = 1; step < kFinalSlots; step <<= 1) {
        const double its_cost = __shfl_down(cost, step, kFinalSlots);
        const uint32_t its_row = __shfl_down(row, step, kFinalSlots);
        if (j + step < kFinalSlots) take_lower(cost, row, its_cost, its_row);
      }
      take_lower(cost, row, carry_cost[pair], carry_row[pair]);
      winner[pair][j] = row;
      if (j == 0) {
        carry_cost[pair] = cost;
        carry_row[pair] = row;
      }
    }
    __syncthreads();
    for (int q = kFinalSlots / 4 - 1; q >= 0; --q) {
      const int slot = wave * (kFinalSlots / 4) + q;
      if (p0 + slot < f.n_p) write_final(f, g, variant, pc, k, row_terms, winner[lane][slot], p0 + slot, tables,
                                      prob.sparse_tables != 0);
    }
  }
}

// Several samples (a slot's lie side by side, as in the tables): one thread per (group, pair,
// sample, variant, kFinalRange values of p).
constexpr int kFinalRange = 16;
__global__ __launch_bounds__(256) void finalize_samples_kernel(
    const MistProblem prob, const MistGroupDesc *__restrict__ groups, const double *__restrict__ row_terms,
    const ReduceTables tabs, const SampleSlots samples, MistOutTables tables) {
  const int L = prob.num_layers, n_pairs = L * (L + 1) / 2 + L;
  const MistGroupDesc *g = groups + blockIdx.z;
  const int P = g->num_p, n = tabs.n_samples;
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  const int s = e % n, pair_rel = e / n;
  // blockIdx.y: ranges of p of base, then of with_pre; with_post; no_pp
  const int ranges = (prob.p_dim + kFinalRange - 1) / kFinalRange, part = blockIdx.y;
  const int variant = part < ranges ? 0 : part < 2 * ranges ? 1 : 2 + (part - 2 * ranges);
  const int p_begin = variant < 2 ? part % ranges * kFinalRange : 0;
  // The group's tiles are a window of the pair list; cells outside were not evaluated.
  const int pair_idx = g->lc_tile_begin * MIST_LC_TILE + pair_rel;
  if (pair_rel >= g->n_lc_tiles * MIST_LC_TILE || pair_idx >= n_pairs) return;
  const PairIndex pc = decode_pair(pair_idx);
  FinalCell f = final_cell(prob, g, variant, pc, samples.at[s]);
  const int64_t first = (g->cell_offset + (int64_t)pair_rel * slots_of(P) +
                         (variant < 2 ? variant * P : 2 * P + variant - 2)) * n + s;
  const GroupConsts k = group_consts(g);
  double cost = INFINITY;
  uint32_t row = ~0u;
  for (int p = f.n_p - 1; p >= p_begin; --p) {
    take_lower(cost, row, tabs.best[first + (int64_t)p * n], tabs.row[first + (int64_t)p * n]);
    if (p < p_begin + kFinalRange) write_final(f, g, variant, pc, k, row_terms, row, p, tables, false);
  }
}

// ------------------------------------------------------------------------------------------
// Analysis path: the quantities batched_stage_analyze(get_best_solution=False) reports for ONE
// given strategy row and one (layers, ckpt, pre-saved micro-batches) cell
// (batched_module_analyzer.py:2788-2803, 2876-2892, 2980-2996, 3063-3079), unmasked.
// One thread per request; per variant (middle, first, last, single stage): stable latency, delta
// latency, stable + delta / G, forward peak, backward peak.
// ------------------------------------------------------------------------------------------
__device__ __forceinline__ LaneMemory cell_memory(const double *__restrict__ t, int l, int c) {
  const double lf = (double)l, lm1 = (double)max(l - 1, 0), cf = (double)c;
  const double S_ck = t[MIST_T_S_CK], S_nock = t[MIST_T_S_NOCK];
  LaneMemory mem;
  mem.fwd_states = t[MIST_T_FWD_STATES0] + lf * t[MIST_T_PWG] + lm1 * t[MIST_T_PO];  // :2150-2162
  mem.bwd_states = t[MIST_T_BWD_STATES0] + lf * t[MIST_T_PWGO];
  mem.cur_saved = c == l ? (lf - 1.0) * S_ck : cf * S_ck + (double)(l - c - 1) * S_nock;  // :2358-2385
  mem.mod_saved = S_ck * cf + S_nock * (double)(l - c);
  mem.ck_delta = c >= l - 1 ? t[MIST_T_D_CK] : t[MIST_T_D_NOCK];  // :2760-2769
  mem.fwd_pk = t[MIST_T_FWD_PEAK];
  mem.bwd_pk = t[MIST_T_BWD_PEAK];
  mem.out = t[MIST_T_OUT];
  mem.gcb = t[MIST_T_GCB];
  mem.mf_base = t[MIST_T_MF_BASE];
  mem.mf_pp = t[MIST_T_MF_PP];
  return mem;
}

__global__ __launch_bounds__(64) void analyze_kernel(
    const MistProblem prob, const MistGroupDesc *__restrict__ groups, int n_groups,
    const double *__restrict__ row_terms, const int32_t *__restrict__ requests, int n_requests,
    double *__restrict__ out) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n_requests) return;
  const int32_t *req = requests + (int64_t)i * MIST_ANALYZE_REQUEST_FIELDS;
  double *o = out + (int64_t)i * MIST_ANALYZE_FIELDS;
  const int gi = req[0], l = req[2], c = req[3], p = req[4];
  const int64_t pos = req[1];
  const bool ok = gi >= 0 && gi < n_groups && l >= 1 && l <= prob.num_layers && c >= 0 && c <= l &&
                  p >= 0 && pos >= 0 && pos < groups[min(max(gi, 0), n_groups - 1)].n_rows;
  if (!ok) {
    for (int f = 0; f < MIST_ANALYZE_FIELDS; ++f) o[f] = NAN;
    return;
  }
  const MistGroupDesc *g = groups + gi;
  const double *t = row_terms + (g->row_offset + pos) * MIST_ROW_TERMS;
  const GroupConsts k = group_consts(g);
  const CellLatency lat = cell_latency<true>(t, l, c, k);
  const LaneMemory mem = cell_memory(t, l, c);
  const double G64 = (double)g->grad_accum;
  const float G32 = (float)g->grad_accum;
  double peak_f, peak_b;
  mem.peaks(p, peak_f, peak_b);
  // middle stage: float32 stable + float32 delta / G stays float32 (:2212-2216)
  o[0] = (double)lat.x;
  o[1] = (double)lat.d;
  o[2] = (double)(lat.x + lat.d / G32);
  o[3] = peak_f;
  o[4] = peak_b;
  // first stage (:2866-2875)
  const double pre_p = (double)p * g->pre_saved;
  o[5] = lat.sp;
  o[6] = lat.dpre;
  o[7] = lat.sp + lat.dpre / G64;
  o[8] = pre_p + peak_f + g->pre_states_and_saved;
  o[9] = pre_p + peak_b + g->pre_states_and_saved;
  // last stage (:2946-2979); the reference evaluates it for p == 0 only
  const double f_in =
      mem.fwd_states + g->post_states + mem.mod_saved + g->post_fwd_peak + mem.gcb;
  const double b_in = mem.bwd_states + g->post_states + mem.mod_saved + g->post_bwd_peak +
                      (c == 0 ? t[MIST_T_RD] : 0.0) + mem.gcb;
  const double pf_post = fmax(f_in, peak_f + g->post_states);
  const double pb_post = fmax(b_in, peak_b - mem.out + g->post_states) + g->post_output;
  o[10] = lat.spost;
  o[11] = lat.dpost;
  o[12] = lat.spost + lat.dpost / G64;
  o[13] = pf_post;
  o[14] = pb_post;
  // single stage (:3057-3062)
  o[15] = lat.spp;
  o[16] = lat.dpp;
  o[17] = lat.spp + lat.dpp / G64;
  o[18] = pf_post + g->pre_states + g->pre_saved;
  o[19] = pb_post + g->pre_states + g->pre_saved;
  // module-level memory of the cell (:2150-2162, 2378-2383), reported by get_extra_info
  o[20] = mem.fwd_states;
  o[21] = mem.bwd_states;
  o[22] = mem.mod_saved;
}

// The intermediate quantities of one candidate row that the row terms fold together: what the
// reference's get_extra_info (:2401-2749) reports besides them.  Thread = request = (group,
// workspace position); the same device functions as row_terms_kernel, every row on its own.
__global__ __launch_bounds__(kTermsBlock) void row_diagnostics_kernel(
    const MistProblem prob, const MistGroupDesc *__restrict__ groups, int n_groups,
    const int32_t *__restrict__ requests, int n_requests, double *__restrict__ out) {
  __shared__ __align__(16) double lds_factor[11][kFactorPitch];
  __shared__ double lds_gpu_gpu[32];
  InterferenceModel<false> I;
  I.factors_tame = load_model_tables(prob, lds_factor, lds_gpu_gpu);
  I.table = (LdsDouble *)&lds_factor[0][0];
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int i_safe = min(i, n_requests - 1);  // no early exit: the model's wave-wide test wants every lane
  const int32_t *req = requests + (int64_t)i_safe * 2;
  const int gi = req[0];
  const int64_t pos = req[1];
  const bool ok = gi >= 0 && gi < n_groups && pos >= 0 && pos < groups[min(max(gi, 0), n_groups - 1)].n_rows;
  const MistGroupDesc *g = groups + (ok ? gi : 0);
  const RowParts parts = parts_of_position(g, ok ? pos : 0);
  const double wo = g->wo[g->pair_wo[parts.pair]], go = g->go[g->pair_go[parts.pair]];
  const double oo = g->oo[parts.oo], ao = g->ao[parts.ao];
  const double *par = g->par[parts.par];
  const double dp = par[MIST_PAR_DP], wre = par[MIST_PAR_WRE], gre = par[MIST_PAR_GRE];
  const double ore = par[MIST_PAR_ORE], W = par[MIST_PAR_W], Gr = par[MIST_PAR_G], O = par[MIST_PAR_O];
  const double wre_size = wre == 1.0 ? dp : 1.0, gre_size = gre == 1.0 ? dp : 1.0;
  const double ore_size = ore == 1.0 ? dp : 1.0;
  const KeyInputs in = key_inputs(prob, lds_gpu_gpu, g, par, wo, go, ao);
  const double so_O = host_link_latency(prob.gpu_cpu, O / ore_size * oo);
  const double si_O = host_link_latency(prob.cpu_gpu, O / ore_size * oo);
  const bool adv = prob.adv_first_block != 0;
  Family fam[8];  // forward first / later micro-batch, backward last / not last; nock, ck each
#pragma unroll
  for (int ph = 0; ph < 2; ++ph) {
    const FwdOperands op = fwd_operands(in, ph == 0, so_O, si_O);
    double first, extra_pre;
    fwd_common(I, in, op, ph == 0, adv, first, extra_pre);
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      Family &f = fam[ph * 2 + k];
      f.first = first;
      f.extra_pre = extra_pre;
      fwd_of_ckpt(I, in, op, k != 0, f.layer, f.last, f.extra_post);
    }
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) fam[4 + j] = bwd_family(I, in, (j & 2) != 0, (j & 1) != 0);
  if (i >= n_requests) return;
  double *o = out + (int64_t)i * MIST_DIAG_FIELDS;
  if (!ok) {
    for (int f = 0; f < MIST_DIAG_FIELDS; ++f) o[f] = NAN;
    return;
  }
  const bool wbuf_on = wre_size > 1.0 || g->pp_wre == 1 || wo > 0.0;
  const bool gbuf_on = gre_size > 1.0 || g->pp_gre == 1 || go > 0.0;
  const FwdOperands f0 = fwd_operands(in, true, so_O, si_O), f1 = fwd_operands(in, false, 0.0, 0.0);
  o[MIST_DG_SO_W] = in.so_W;
  o[MIST_DG_SI_W] = in.si_W;
  o[MIST_DG_SO_G] = in.so_G;
  o[MIST_DG_SI_G] = in.si_G;
  o[MIST_DG_SO_O] = so_O;
  o[MIST_DG_SI_O] = si_O;
  o[MIST_DG_SO_A_CK] = in.so_A_ck;
  o[MIST_DG_SI_A_CK] = in.si_A_ck;
  o[MIST_DG_SO_A_NOCK] = in.so_A_nock;
  o[MIST_DG_SI_A_NOCK] = in.si_A_nock;
  o[MIST_DG_AG_W] = in.AG_w;
  o[MIST_DG_RS_G] = in.RS_g;
  o[MIST_DG_AR_G] = in.AR_g;
  o[MIST_DG_WBUF] = wbuf_on ? fmax(fmax(g->pre_full_w, g->post_full_w), W) : 0.0;
  o[MIST_DG_GBUF] = gbuf_on ? fmax(fmax(g->pre_full_g, g->post_full_g), Gr) : 0.0;
  o[MIST_DG_PW] = W / wre_size * (1.0 - wo);
  o[MIST_DG_PG] = Gr / gre_size * (1.0 - go);
  o[MIST_DG_G2C_F0] = f0.g2c;
  o[MIST_DG_C2G_F0] = f0.c2g;
  o[MIST_DG_G2G_F0] = f0.g2g;
  o[MIST_DG_G2C_F1] = f1.g2c;
  o[MIST_DG_C2G_F1] = f1.c2g;
  o[MIST_DG_G2G_F1] = f1.g2g;
  o[MIST_DG_G2C_B] = in.g2c_B;
  o[MIST_DG_C2G_B] = in.c2g_B;
  o[MIST_DG_G2G_B0] = in.g2g_B[0];
  o[MIST_DG_G2G_B1] = in.g2g_B[1];
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    double *f = o + MIST_DG_FAMILIES + j * 5;
    f[0] = fam[j].layer;
    f[1] = fam[j].first;
    f[2] = fam[j].last;
    f[3] = fam[j].extra_pre;
    f[4] = fam[j].extra_post;
  }
}

int check_factors(const MistProblem *problem) {
  for (int m = 0; m < 11; ++m)
    for (int i = 0; i < 4; ++i) {
      const double f = problem->interf_factor[m][i];
      // the kernel takes 0 / f == +0 for granted
      if (!(f > 0.0) || std::isinf(f))
        return fail(MIST_E_INVALID, "interference factor [%d][%d] must be positive and finite", m, i);
    }
  return 0;
}

int check_common(const void *d_problem, const void *d_groups, int n_groups) {
  if (!d_problem || !d_groups) return fail(MIST_E_INVALID, "null problem / group pointer");
  if (n_groups <= 0) return fail(MIST_E_INVALID, "n_groups must be positive, got %d", n_groups);
  const MistProblem *problem = static_cast<const MistProblem *>(d_problem);
  if (problem->stage_cost_incumbent != nullptr) {
    if (problem->sample_size != 1 && problem->incumbent_close != kCloseAssignment)
      return fail(MIST_E_INVALID, "a stage-cost incumbent needs sample_size 1, got %d",
                  problem->sample_size);
    if (problem->incumbent_num_devices < 1 || problem->incumbent_ckpt_rule < 0 ||
        problem->incumbent_ckpt_rule > 2)
      return fail(MIST_E_INVALID, "stage-cost incumbent with %d devices, ckpt rule %d",
                  problem->incumbent_num_devices, problem->incumbent_ckpt_rule);
  }
  if (problem->incumbent_close != 0 && problem->stage_cost_incumbent == nullptr)
    return fail(MIST_E_INVALID, "incumbent_close without a stage-cost incumbent");
  if (problem->incumbent_close < 0 || problem->incumbent_close > kCloseAssignment)
    return fail(MIST_E_INVALID, "incumbent_close %d", problem->incumbent_close);
  return 0;
}

}  // namespace

extern "C" {

const char *mist_version(void) { return "mist_search 0.1 (gfx950)"; }
const char *mist_last_error(void) { return g_last_error; }
int mist_sizeof_problem(void) { return (int)sizeof(MistProblem); }
int mist_sizeof_group(void) { return (int)sizeof(MistGroupDesc); }
int mist_reduce_p_tile(void) { return MIST_P_TILE; }
double mist_incumbent_slack(void) { return kIncumbentSlack; }

static bool has_key_terms(const MistProblem *problem, int n_groups, const double *d_key_terms) {
  return d_key_terms != nullptr && problem->max_group_keys > 0 && n_groups <= 65535;
}
// (for tests MIST_STAGE_FLOOR_RUNS = 0 | 1 decides)
static bool stage_floor_runs(int n_blocks) {
  const char *decided = getenv("MIST_STAGE_FLOOR_RUNS");
  return decided == nullptr || *decided == '\0' ? n_blocks >= kFloorRunBlocks : *decided != '0';
}
static void launch_stage_floors(const MistProblem *problem, const MistGroupDesc *d_groups, int n_groups,
                                const int32_t *d_block_prefix, int n_blocks, double *d_stage_floor,
                                const double *d_key_terms, hipStream_t stream) {
  if (!stage_floor_runs(n_blocks))
    hipLaunchKernelGGL(stage_floor_kernel, dim3(n_blocks), dim3(kTermsBlock), 0, stream, *problem, d_groups, n_groups,
                       d_block_prefix, d_stage_floor, d_key_terms);
  else
    hipLaunchKernelGGL(stage_floor_runs_kernel, dim3(xcd_padded_grid((n_blocks + kFloorRun - 1) / kFloorRun)),
                       dim3(kFloorThreads), 0, stream, *problem, d_groups, n_groups, d_block_prefix, n_blocks, d_stage_floor,
                       d_key_terms);
}
// key_terms_kernel over every group when the caller gave a key-term workspace and the bound the
// grid needs; *launched tells whether the row-term kernel can read key terms.
static int launch_key_terms(const MistProblem *problem, const MistGroupDesc *d_groups, int n_groups,
                            double *d_key_terms, hipStream_t stream, bool *launched) {
  *launched = has_key_terms(problem, n_groups, d_key_terms);
  if (!*launched) return 0;
  constexpr int kKeysPerBlock = kTermsBlock / 4;
  const unsigned blocks = (unsigned)((problem->max_group_keys + kKeysPerBlock - 1) / kKeysPerBlock);
  hipLaunchKernelGGL(key_terms_kernel, dim3(blocks, n_groups), dim3(kTermsBlock), 0, stream, *problem,
                     d_groups, d_key_terms);
  MIST_HIP_CHECK(hipGetLastError());
  return 0;
}

int mist_row_terms(const MistProblem *problem, const MistGroupDesc *d_groups, int n_groups,
                   const int32_t *d_block_prefix, int n_blocks, double *d_row_terms,
                   double *d_stage_floor, double *d_key_terms, void *stream) {
  if (int rc = check_common(problem, d_groups, n_groups)) return rc;
  if (!d_block_prefix || !d_row_terms || !d_stage_floor)
    return fail(MIST_E_INVALID, "null workspace pointer");
  if (n_blocks <= 0) return fail(MIST_E_INVALID, "n_blocks must be positive, got %d", n_blocks);
  if (int rc = check_factors(problem)) return rc;
  bool from_keys = false;
  if (int rc = launch_key_terms(problem, d_groups, n_groups, d_key_terms, (hipStream_t)stream, &from_keys))
    return rc;
  if (from_keys) {
    launch_stage_floors(problem, d_groups, n_groups, d_block_prefix, n_blocks, d_stage_floor, d_key_terms, (hipStream_t)stream);
    MIST_HIP_CHECK(hipGetLastError());
    hipLaunchKernelGGL((row_terms_kernel<0, true>), dim3(n_blocks), dim3(kTermsBlock), 0,
                       (hipStream_t)stream, *problem, d_groups, n_groups, d_block_prefix, d_row_terms,
                       d_stage_floor, d_key_terms);
  } else
    hipLaunchKernelGGL((row_terms_kernel<0, false>), dim3(n_blocks), dim3(kTermsBlock), 0,
                       (hipStream_t)stream, *problem, d_groups, n_groups, d_block_prefix, d_row_terms,
                       d_stage_floor, nullptr);
  MIST_HIP_CHECK(hipGetLastError());
  return 0;
}

int64_t mist_key_terms_doubles(int64_t total_keys) {
  return total_keys < 0 ? -1 : total_keys * MIST_KEY_TERMS;
}

int mist_reduce_stage_rows(void) { return kStageRows; }
int mist_reduce_lc_tile(void) { return MIST_LC_TILE; }
int mist_terms_block_rows(void) { return kTermsBlock; }
int mist_reduce_scout_split(void) { return kScoutSplit; }
int mist_workspace_oo_tile(void) { return kOoTile; }
int mist_max_sample_batch(void) { return MIST_MAX_SAMPLE_BATCH; }
int mist_key_terms_per_key(void) { return MIST_KEY_TERMS; }
int mist_max_scout_pairs(void) { return MIST_MAX_SCOUT_PAIRS; }
int64_t mist_stage_floor_doubles(int64_t total_rows, int n_groups) {
  if (total_rows < 0 || n_groups < 0) return -1;
  return (total_rows / kStageRows + n_groups + 1) * kStageFloorPitch;
}

// Sections of the reduce workspace in `d_partial_cost` (doubles): the minima of n_samples samples,
// the second-level summaries, the four lists, their counters, a word per stage, the bounds of the gathered
// rows, a record per group, the log and its chunks' counts.
struct WorkspaceLayout {
  int64_t best, supers, items, counters, flags, gathered, reach, log, log_counts, total;
  int64_t capacity;    // items per shard
  int64_t log_chunks;
};
// `doubles`: what there is (0: all that is of use), at least total - log_chunks' share.
static WorkspaceLayout workspace_layout(int64_t cells, int64_t supers, int64_t items, int n_samples, int64_t doubles) {
  WorkspaceLayout w;
  w.capacity = (items + kQueueShards - 1) / kQueueShards + 1;
  w.best = 0;
  w.supers = cells * n_samples;
  w.items = w.supers + supers * kStageFloorPitch;
  w.counters = w.items + 4 * kQueueShards * w.capacity;
  w.flags = w.counters + kCounters * kCounterPitch / 2;
  w.gathered = w.flags + supers * kSuperStages / 2;
  w.reach = w.gathered + supers * kSuperStages * kGatherFloor;  // (a batch of samples may end with one alone)
  // (two second-level summaries a group at least)
  w.log = w.reach + supers / 2 * (int64_t)(sizeof(GroupReach) / 8 + 2 * kSuperBlocks);
  w.log += w.log % 2;
  // (a chunk of every wavefront's is as a rule not full; a log's cells are 32 bits)
  w.log_chunks = std::min(kLogPerCell * cells * n_samples, kLogEntries) / kLogChunk + kReduceWorkers * (kReduceThreads / 64);
  if (cells * n_samples > (int64_t)UINT32_MAX) w.log_chunks = 0;
  constexpr int64_t kChunkDoubles = kLogChunk * (int64_t)(sizeof(Hit) / 8);
  if (doubles > 0)  // (half a double per chunk for its count, and one more)
    w.log_chunks = std::min(w.log_chunks, std::max<int64_t>(doubles - w.log - 1, 0) * 2 / (2 * kChunkDoubles + 1));
  w.log_counts = w.log + w.log_chunks * kChunkDoubles;
  w.total = w.log_counts + w.log_chunks / 2 + 1;
  return w;
}
int64_t mist_reduce_workspace_doubles(int64_t cells, int64_t supers, int64_t items, int n_samples) {
  if (cells < 0 || supers < 0 || items < 0 || n_samples < 1) return -1;
  return workspace_layout(cells, supers, items, n_samples, 0).total;
}
int64_t mist_reduce_workspace_least_doubles(int64_t cells, int64_t supers, int64_t items, int n_samples) {
  if (cells < 0 || supers < 0 || items < 0 || n_samples < 1) return -1;
  return workspace_layout(cells, supers, items, n_samples, 1).total;
}
// (for tests MIST_REDUCE_LOG_CHUNKS is the most)
static uint32_t log_chunks(int64_t chunks) {
  const char *most = getenv("MIST_REDUCE_LOG_CHUNKS");
  return (uint32_t)(most == nullptr || *most == '\0' ? chunks : std::min(chunks, std::max<int64_t>(atoll(most), 0)));
}
// rows_present: false = only the rows the seed launch gathers are, the others follow by need
static int reduce_tables(const MistProblem *problem, int n_samples, double *d_partial_cost, int32_t *d_partial_index,
                         ReduceTables *out, bool rows_present = true) {
  if (problem->reduce_cells < 1 || problem->reduce_supers < 1 || problem->reduce_items < 1 ||
      problem->reduce_max_p < 1)
    return fail(MIST_E_INVALID, "MistProblem.reduce_* sizes of the workspace are not set");
  const WorkspaceLayout w =
      workspace_layout(problem->reduce_cells, problem->reduce_supers, problem->reduce_items, n_samples,
                       std::max<int64_t>(problem->reduce_doubles, 0));
  if (problem->reduce_doubles < 0 || (problem->reduce_doubles > 0 && problem->reduce_doubles < w.total))
    return fail(MIST_E_INVALID, "a reduce workspace of %lld doubles needs %lld", (long long)problem->reduce_doubles,
                (long long)w.total);
  if (w.capacity >= (int64_t)1 << 31) return fail(MIST_E_INVALID, "too many (tile, stage) items");
  out->best = d_partial_cost + w.best;
  out->row = reinterpret_cast<uint32_t *>(d_partial_index);
  out->super_floor = d_partial_cost + w.supers;
  out->item = reinterpret_cast<unsigned long long *>(d_partial_cost + w.items);
  out->opened = out->item + kQueueShards * w.capacity;
  out->open_pairs = out->opened + kQueueShards * w.capacity;
  out->listed = rows_present ? nullptr : out->open_pairs + kQueueShards * w.capacity;
  out->stage_flag = reinterpret_cast<uint32_t *>(d_partial_cost + w.flags);
  out->counter = reinterpret_cast<uint32_t *>(d_partial_cost + w.counters);
  out->log = reinterpret_cast<Hit *>(d_partial_cost + w.log);
  out->log_count = reinterpret_cast<uint32_t *>(d_partial_cost + w.log_counts);
  out->log_chunks = log_chunks(w.log_chunks);
  out->gather_floor = d_partial_cost + w.gathered;
  out->reach = reinterpret_cast<GroupReach *>(d_partial_cost + w.reach);
  out->reach_parts = d_partial_cost + w.reach + problem->reduce_supers / 2 * (int64_t)(sizeof(GroupReach) / 8);
  out->capacity = (uint32_t)w.capacity;
  out->n_samples = n_samples;
  return 0;
}

static int launch_first_estimate(const MistProblem *problem, const MistGroupDesc *d_groups, int n_groups,
                                 const double *d_row_terms, double ratio, double *d_partial_cost,
                                 double *gather_floor, void *stream) {
  const bool assignment = problem->incumbent_close == kCloseAssignment;
  hipLaunchKernelGGL(assignment ? estimate_stage_minima_kernel<true> : estimate_stage_minima_kernel<false>,
                     dim3(kEstimateSplit + (gather_floor ? kGatherBlocks : 0), n_groups), dim3(256), 0, (hipStream_t)stream,
                     *problem, d_groups, d_row_terms, assignment ? 1.0 : ratio, d_partial_cost, gather_floor);
  MIST_HIP_CHECK(hipGetLastError());
  if (assignment) {
    hipLaunchKernelGGL(estimate_assignment_kernel, dim3(n_groups), dim3(64), 0, (hipStream_t)stream, *problem, d_groups,
                       d_row_terms, d_partial_cost);
    MIST_HIP_CHECK(hipGetLastError());
    return 0;
  }
  hipLaunchKernelGGL(estimate_combine_kernel, dim3(n_groups), dim3(64), 0, (hipStream_t)stream,
                     *problem, d_groups, d_partial_cost);
  MIST_HIP_CHECK(hipGetLastError());
  return 0;
}

// Samples of a batch that one set of launches takes (see kMostCountedP).
static int samples_together(const MistProblem *problem, int n_samples) {
  return problem->reduce_max_p > kMostCountedP ? 1 : n_samples;
}

// More than 64 KB of LDS per workgroup needs an opt-in, once per device.
static int allow_large_lds() {
  static std::mutex lock;
  static bool done[64];
  int device = 0;
  MIST_HIP_CHECK(hipGetDevice(&device));
  if (device < 0 || device >= 64) return fail(MIST_E_INVALID, "device ordinal %d outside [0, 64)", device);
  std::lock_guard<std::mutex> guard(lock);
  if (!done[device]) {
    for (const void *kernel : {reinterpret_cast<const void *>(seed_kernel),
                               reinterpret_cast<const void *>(seed_samples_kernel),
                               reinterpret_cast<const void *>(reduce_kernel<false, false, true>),
                               reinterpret_cast<const void *>(reduce_kernel<true, false, true>)})
      MIST_HIP_CHECK(hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, kSeedLdsMost));
    done[device] = true;
  }
  return 0;
}

// The problem as the launches of one call take it: cells are closed where form_reach has room for the groups.
static MistProblem closing(const MistProblem *problem, int n_groups, int n_samples, bool assignments = true) {
  MistProblem own = *problem;
  if (own.incumbent_close == kCloseAssignment) {
    // an estimate of the assignments bounds no stage cost at one of the samples
    if (n_samples == 1 || !assignments) own.incumbent_close = 0, own.stage_cost_incumbent = nullptr;
  } else if (n_samples != 1 || n_groups > kReachGroups) {
    own.incumbent_close = 0;
  }
  return own;
}

// The estimate of the best pipeline cost that the seeds allow, and with MistProblem.incumbent_close (behind the
// second-level summaries) what it says of every group.
static int launch_incumbent(const MistProblem *problem, const MistGroupDesc *d_groups, int n_groups, const ReduceTables &tabs,
                            void *stream) {
  if (problem->incumbent_close == kCloseAssignment) {
    hipLaunchKernelGGL(assignment_reach_kernel, dim3(n_groups), dim3(64), 0, (hipStream_t)stream, *problem, d_groups, tabs);
    MIST_HIP_CHECK(hipGetLastError());
    return 0;
  }
  if (problem->stage_cost_incumbent == nullptr || tabs.n_samples != 1) return 0;
  hipLaunchKernelGGL(incumbent_kernel, dim3(n_groups), dim3(64 * kIncumbentWaves),
                     problem->incumbent_close == kCloseSearch ? n_groups * sizeof(ReachBounds) : 0, (hipStream_t)stream, *problem, d_groups,
                     tabs);
  MIST_HIP_CHECK(hipGetLastError());
  return 0;
}

// Minima tables filled with what the rows of the scout pairs give (+inf where a group has none and
// with `scouted` false), and the estimate of the best pipeline cost they allow (with MistProblem.incumbent_close that
// is left to launch_incumbent; without seeds nothing is closed).
static int launch_seeds(MistProblem *problem, const MistGroupDesc *d_groups, int n_groups,
                        const double *d_row_terms, const RatioList &ratios, bool scouted,
                        const ReduceTables &tabs, double *d_partial_cost, void *stream) {
  const int L = problem->num_layers, n_pairs = L * (L + 1) / 2 + L;
  const int tiles = (n_pairs + MIST_LC_TILE - 1) / MIST_LC_TILE;
  if (tiles > 1 << kItemTileBits)
    return fail(MIST_E_INVALID, "at most %d tiles of (l, c) pairs, got %d", 1 << kItemTileBits, tiles);
  const int64_t pair_bytes = 8 * (int64_t)slots_of(problem->reduce_max_p);
  // fewer pairs, or samples, per workgroup when the slots are many, so that several stay resident
  int pair_split = tabs.n_samples == 1 ? 16 : 1;
  while (pair_split > 1 && pair_split * pair_bytes > kSeedLdsBytes) pair_split /= 2;
  // ... and where there would be fewer than eight workgroups per CU (16, 8 and 4 pairs: stage operator of 7B on
  // 2x8, one group, 106, 65, 40 us; uniform-pp of 7B on 2x8, 56 groups, beside the summaries 125, 90 to 167 by run,
  // 168, from the gathered rows to the filter 249, 251 to 277, 267; the 7B plan on 4x8, 72 groups, 257, 255, 259;
  // 70B on 32x8, 120 groups, 1250, 1490, 1930)
  while (pair_split > 4 && (int64_t)tiles * (MIST_LC_TILE / pair_split) * n_groups < kSeedWorkgroups) pair_split /= 2;
  int sample_split = tabs.n_samples;
  while (sample_split > 1 && pair_bytes * sample_split > kSeedLdsBytes) sample_split = (sample_split + 1) / 2;
  int sample_waves = tabs.n_samples == 1 ? 0 : kSeedSampleWaves;
  while (sample_waves > 1 && pair_bytes + sample_waves * (int64_t)sizeof(SampleRows) > kSeedLdsMost) sample_waves /= 2;
  const int64_t bytes = pair_bytes * pair_split * sample_split + sample_waves * (int64_t)sizeof(SampleRows);
  const bool seeds = scouted && bytes <= kSeedLdsMost;  // (some 10000 values of p)
  const bool estimate = scouted && problem->stage_cost_incumbent != nullptr && problem->incumbent_first_estimate != 0 &&
                        tabs.n_samples == 1 && problem->sample_size == 1;
  // a first estimate from a few rows, so that the seed launch itself runs under a bound
  if (estimate)
    if (int rc = launch_first_estimate(problem, d_groups, n_groups, d_row_terms, ratios.r[0], d_partial_cost,
                                       seeds && tabs.n_samples == 1 ? tabs.gather_floor : nullptr, stream))
      return rc;
  if (!seeds) {
    if (problem->incumbent_close == kCloseSearch) problem->incumbent_close = 0;
    hipLaunchKernelGGL(empty_minima_kernel, dim3(kReduceBlocks), dim3(256), 0, (hipStream_t)stream, tabs,
                       problem->reduce_cells);
    MIST_HIP_CHECK(hipGetLastError());
    return 0;
  }
  if (bytes > 64 * 1024)
    if (int rc = allow_large_lds()) return rc;
  if (tabs.n_samples == 1 && !estimate) {
    hipLaunchKernelGGL(gather_floor_kernel, dim3(kGatherBlocks, n_groups), dim3(256), 0, (hipStream_t)stream, *problem,
                       d_groups, d_row_terms, ratios.r[0], tabs.gather_floor);
    MIST_HIP_CHECK(hipGetLastError());
  }
  const dim3 grid(tiles * (MIST_LC_TILE / pair_split), n_groups,
                  (tabs.n_samples + sample_split - 1) / sample_split);
  if (tabs.n_samples == 1)
    hipLaunchKernelGGL(seed_kernel, grid, dim3(kSeedThreads), (size_t)bytes, (hipStream_t)stream, *problem, d_groups,
                       d_row_terms, ratios.r[0], tabs, pair_split);
  else
    hipLaunchKernelGGL(seed_samples_kernel, grid, dim3(64 * sample_waves), (size_t)bytes, (hipStream_t)stream, *problem, d_groups,
                       d_row_terms, ratios, tabs, sample_split);
  MIST_HIP_CHECK(hipGetLastError());
  return problem->incumbent_close != 0 ? 0 : launch_incumbent(problem, d_groups, n_groups, tabs, stream);
}

static int launch_super_floors(const MistProblem *problem, const MistGroupDesc *d_groups, int n_groups,
                               const double *d_stage_floor, double ratio, const ReduceTables &tabs, void *stream) {
  hipLaunchKernelGGL(super_floor_kernel, dim3(kSuperBlocks, n_groups), dim3(256), 0, (hipStream_t)stream, d_groups,
                     n_groups, d_stage_floor, problem->incumbent_close == kCloseAssignment ? 1.0 : ratio, problem->incumbent_close, tabs);
  MIST_HIP_CHECK(hipGetLastError());
  return 0;
}

// filter + open + reduce + resolve on seeded tables.
static int launch_reduce(const MistProblem *problem, const MistGroupDesc *d_groups, int n_groups,
                         const int32_t *d_block_prefix, int n_blocks, const double *d_row_terms,
                         const double *d_stage_floor, const double *d_key_terms, const RatioList &ratios,
                         const ReduceTables &tabs, void *stream) {
  const bool one = tabs.n_samples == 1;
  hipLaunchKernelGGL(one ? filter_kernel<false> : filter_kernel<true>, dim3(xcd_padded_grid(n_blocks)),
                     dim3(one ? 64 : kFilterShares * 64), one ? 0 : tabs.n_samples * 2 * kFilterPitch * sizeof(double),
                     (hipStream_t)stream, *problem, d_groups, n_groups, d_block_prefix, n_blocks, d_stage_floor,
                     tabs.super_floor, ratios, tabs);
  MIST_HIP_CHECK(hipGetLastError());
  const bool buffered = one && slots_of(problem->reduce_max_p) <= kMostBufferedSlots;
  hipLaunchKernelGGL(one ? open_kernel<false> : open_kernel<true>, dim3(kReduceBlocks), dim3(kReduceThreads), 0,
                     (hipStream_t)stream, *problem, d_groups, d_stage_floor, ratios, tabs);
  MIST_HIP_CHECK(hipGetLastError());
  if (tabs.listed != nullptr) {
    hipLaunchKernelGGL(stage_rows_kernel, dim3(kStageRowsBlocks), dim3(kTermsBlock), 0, (hipStream_t)stream, *problem,
                       d_groups, const_cast<double *>(d_row_terms), d_key_terms, tabs);
    MIST_HIP_CHECK(hipGetLastError());
  }
  const int wave_pitch = one ? kCandidateDoubles + (buffered ? slots_of(problem->reduce_max_p) : 0) : 0;
  const size_t lds = sizeof(double) * wave_pitch * (kReduceThreads / 64);
  if (lds > 64 * 1024)
    if (int rc = allow_large_lds()) return rc;
#define MIST_REDUCE(RESOLVE, SAMPLES, IN_LDS)                                                               \
  hipLaunchKernelGGL((reduce_kernel<RESOLVE, SAMPLES, IN_LDS>), dim3(RESOLVE ? kAgainBlocks : kReduceWorkers),    \
                     dim3(kReduceThreads), lds, (hipStream_t)stream, *problem, d_groups, d_row_terms, d_stage_floor, ratios, tabs, wave_pitch)
  if (!one) MIST_REDUCE(false, true, false);
  else if (buffered) MIST_REDUCE(false, false, true);
  else MIST_REDUCE(false, false, false);
  MIST_HIP_CHECK(hipGetLastError());
  hipLaunchKernelGGL(resolve_kernel, dim3(kReduceBlocks), dim3(kReduceThreads), 0, (hipStream_t)stream, tabs);
  MIST_HIP_CHECK(hipGetLastError());
  // (returns at once unless the log ran full)
  if (!one) MIST_REDUCE(true, true, false);
  else if (buffered) MIST_REDUCE(true, false, true);
  else MIST_REDUCE(true, false, false);
#undef MIST_REDUCE
  MIST_HIP_CHECK(hipGetLastError());
  return 0;
}

static int check_reduce_arguments(const MistProblem *problem, const MistGroupDesc *d_groups,
                                  int n_groups, const int32_t *d_block_prefix, int n_blocks,
                                  const int32_t *d_scout_prefix, int n_scout_blocks,
                                  const double *d_row_terms, const double *d_stage_floor,
                                  const double *d_partial_cost, const int32_t *d_partial_index) {
  if (int rc = check_common(problem, d_groups, n_groups)) return rc;
  if (!d_block_prefix || !d_row_terms || !d_stage_floor || !d_partial_cost || !d_partial_index)
    return fail(MIST_E_INVALID, "null workspace pointer");
  if (n_blocks <= 0) return fail(MIST_E_INVALID, "n_blocks must be positive, got %d", n_blocks);
  if (n_scout_blocks < 0 || (n_scout_blocks > 0 && !d_scout_prefix))
    return fail(MIST_E_INVALID, "scout blocks need a scout prefix (n_scout_blocks=%d)",
                n_scout_blocks);
  if (n_groups > 65535) return fail(MIST_E_INVALID, "at most 65535 groups per call, got %d", n_groups);
  return 0;
}

int mist_eval_reduce(const MistProblem *problem, const MistGroupDesc *d_groups, int n_groups,
                     const int32_t *d_block_prefix, int n_blocks,
                     const int32_t *d_scout_prefix, int n_scout_blocks,
                     const double *d_row_terms, const double *d_stage_floor, double ratio,
                     double *d_partial_cost, int32_t *d_partial_index, void *stream) {
  if (int rc = check_reduce_arguments(problem, d_groups, n_groups, d_block_prefix, n_blocks,
                                      d_scout_prefix, n_scout_blocks, d_row_terms, d_stage_floor,
                                      d_partial_cost, d_partial_index))
    return rc;
  if (!(ratio >= 0.0)) return fail(MIST_E_INVALID, "ratio must be non-negative");
  RatioList ratios = {};
  ratios.r[0] = ratio;
  ReduceTables tabs;
  if (int rc = reduce_tables(problem, 1, d_partial_cost, d_partial_index, &tabs)) return rc;
  MistProblem own = closing(problem, n_groups, 1);
  if (int rc = launch_seeds(&own, d_groups, n_groups, d_row_terms, ratios, n_scout_blocks > 0, tabs, d_partial_cost,
                            stream))
    return rc;
  if (int rc = launch_super_floors(&own, d_groups, n_groups, d_stage_floor, ratio, tabs, stream)) return rc;
  if (own.incumbent_close != 0)
    if (int rc = launch_incumbent(&own, d_groups, n_groups, tabs, stream)) return rc;
  return launch_reduce(&own, d_groups, n_groups, d_block_prefix, n_blocks, d_row_terms, d_stage_floor, nullptr, ratios, tabs,
                       stream);
}

int mist_stage_cost_first_estimate(const MistProblem *problem, const MistGroupDesc *d_groups,
                                   int n_groups, const int32_t *d_scout_prefix, int n_blocks,
                                   const double *d_row_terms, double ratio, double *d_partial_cost,
                                   void *stream) {
  if (int rc = check_common(problem, d_groups, n_groups)) return rc;
  if (!d_scout_prefix || !d_row_terms || !d_partial_cost)
    return fail(MIST_E_INVALID, "null workspace pointer");
  if (n_blocks < 0) return fail(MIST_E_INVALID, "n_blocks must not be negative, got %d", n_blocks);
  if (problem->stage_cost_incumbent == nullptr)
    return fail(MIST_E_INVALID, "no stage-cost incumbent to lower");
  if (n_groups > 65535) return fail(MIST_E_INVALID, "at most 65535 groups per call, got %d", n_groups);
  if (!(ratio >= 0.0)) return fail(MIST_E_INVALID, "ratio must be non-negative");
  return launch_first_estimate(problem, d_groups, n_groups, d_row_terms, ratio, d_partial_cost, nullptr, stream);
}

static int launch_finalize(const MistProblem *problem, const MistGroupDesc *d_groups, int n_groups,
                           const double *d_row_terms, const ReduceTables &tabs, const int32_t *sample_index,
                           const MistOutTables *tables, void *stream) {
  if (!d_row_terms || !tables) return fail(MIST_E_INVALID, "null pointer argument");
  for (int v = 0; v < 4; ++v)
    if (!tables->stable[v] || !tables->delta[v] || !tables->index[v])
      return fail(MIST_E_INVALID, "output table %d is null", v);
  const MistProblem &prob = *problem;
  const int L = prob.num_layers, P1 = prob.p_dim, n_samples = tabs.n_samples;
  if (L <= 0 || P1 <= 0 || prob.sample_size <= 0)
    return fail(MIST_E_INVALID, "bad problem extents L=%d P+1=%d S=%d", L, P1, prob.sample_size);
  SampleSlots slots = {};
  for (int i = 0; i < n_samples; ++i) {
    if (sample_index[i] < 0 || sample_index[i] >= prob.sample_size)
      return fail(MIST_E_INVALID, "sample_index %d outside [0, %d)", sample_index[i], prob.sample_size);
    slots.at[i] = sample_index[i];
  }
  if (n_groups > 65535) return fail(MIST_E_INVALID, "too many groups for one launch: %d", n_groups);
  const int64_t n_pairs = (int64_t)L * (L + 1) / 2 + L + MIST_LC_TILE;
  if (n_samples == 1)
    hipLaunchKernelGGL(finalize_kernel, dim3((unsigned)(n_pairs / MIST_LC_TILE), 4, n_groups), dim3(256), 0,
                       (hipStream_t)stream, prob, d_groups, d_row_terms, tabs, slots.at[0], *tables);
  else
    hipLaunchKernelGGL(finalize_samples_kernel,
                       dim3((unsigned)((n_pairs * n_samples + 255) / 256),
                            2 * ((P1 + kFinalRange - 1) / kFinalRange) + 2, n_groups),
                       dim3(256), 0, (hipStream_t)stream, prob, d_groups, d_row_terms, tabs, slots, *tables);
  MIST_HIP_CHECK(hipGetLastError());
  return 0;
}

int mist_eval_reduce_samples(const MistProblem *problem, const MistGroupDesc *d_groups,
                             int n_groups, const int32_t *d_block_prefix, int n_blocks,
                             const int32_t *d_scout_prefix, int n_scout_blocks,
                             const double *d_row_terms, const double *d_stage_floor,
                             const double *ratios, const int32_t *sample_index, int n_samples,
                             int main_batch, double *d_partial_cost, int32_t *d_partial_index,
                             const MistOutTables *tables, void *stream) {
  if (int rc = check_reduce_arguments(problem, d_groups, n_groups, d_block_prefix, n_blocks,
                                      d_scout_prefix, n_scout_blocks, d_row_terms, d_stage_floor,
                                      d_partial_cost, d_partial_index))
    return rc;
  if (!ratios || !sample_index || n_samples < 1 || n_samples > MIST_MAX_SAMPLE_BATCH)
    return fail(MIST_E_INVALID, "n_samples %d outside [1, %d] or null sample lists", n_samples,
                MIST_MAX_SAMPLE_BATCH);
  if (main_batch < 1 || main_batch > n_samples)
    return fail(MIST_E_INVALID, "main_batch %d outside [1, n_samples = %d]", main_batch, n_samples);
  for (int i = 0; i < n_samples; ++i)
    if (!(ratios[i] >= 0.0)) return fail(MIST_E_INVALID, "ratio %d must be non-negative", i);
  const int batch = samples_together(problem, n_samples);
  for (int first = 0; first < n_samples; first += batch) {
    const int count = std::min(batch, n_samples - first);
    RatioList list = {};
    for (int i = 0; i < count; ++i) list.r[i] = ratios[first + i];
    ReduceTables tabs;
    if (int rc = reduce_tables(problem, count, d_partial_cost, d_partial_index, &tabs)) return rc;
    MistProblem own = closing(problem, n_groups, count, false);
    if (int rc = launch_seeds(&own, d_groups, n_groups, d_row_terms, list, n_scout_blocks > 0, tabs, d_partial_cost,
                              stream))
      return rc;
    if (int rc = launch_super_floors(&own, d_groups, n_groups, d_stage_floor, list.r[0], tabs, stream)) return rc;
    if (own.incumbent_close != 0)
      if (int rc = launch_incumbent(&own, d_groups, n_groups, tabs, stream)) return rc;
    if (int rc = launch_reduce(&own, d_groups, n_groups, d_block_prefix, n_blocks, d_row_terms, d_stage_floor, nullptr,
                               list, tabs, stream))
      return rc;
    if (int rc = launch_finalize(problem, d_groups, n_groups, d_row_terms, tabs, sample_index + first, tables, stream))
      return rc;
  }
  return 0;
}

int mist_eval_reduce_exhaustive(const MistProblem *problem, const MistGroupDesc *d_groups,
                                int n_groups, const int32_t *d_block_prefix, int n_blocks,
                                const double *d_row_terms, double ratio, double *d_partial_cost,
                                int32_t *d_partial_index, void *stream) {
  if (int rc = check_common(problem, d_groups, n_groups)) return rc;
  if (!d_block_prefix || !d_row_terms || !d_partial_cost || !d_partial_index)
    return fail(MIST_E_INVALID, "null workspace pointer");
  if (n_blocks <= 0) return fail(MIST_E_INVALID, "n_blocks must be positive, got %d", n_blocks);
  if (!(ratio >= 0.0)) return fail(MIST_E_INVALID, "ratio must be non-negative");
  if (n_groups > 65535) return fail(MIST_E_INVALID, "at most 65535 groups per call, got %d", n_groups);
  ReduceTables tabs;
  if (int rc = reduce_tables(problem, 1, d_partial_cost, d_partial_index, &tabs)) return rc;
  // the chunks' slabs lie behind the minima
  double *slab_cost = d_partial_cost + problem->reduce_cells;
  int32_t *slab_index = d_partial_index + problem->reduce_cells;
  hipLaunchKernelGGL(eval_reduce_exhaustive_kernel, dim3(xcd_padded_grid(n_blocks)),
                     dim3(MIST_LC_TILE), 0, (hipStream_t)stream, *problem, d_groups, n_groups,
                     d_block_prefix, n_blocks, d_row_terms, ratio, slab_cost, slab_index);
  MIST_HIP_CHECK(hipGetLastError());
  hipLaunchKernelGGL(combine_slabs_kernel, dim3(64, n_groups), dim3(256), 0, (hipStream_t)stream, d_groups,
                     d_block_prefix, slab_cost, slab_index, tabs);
  MIST_HIP_CHECK(hipGetLastError());
  return 0;
}

int mist_finalize(const MistProblem *problem, const MistGroupDesc *d_groups, int n_groups,
                  const int32_t *d_block_prefix, const double *d_row_terms,
                  const double *d_partial_cost, const int32_t *d_partial_index,
                  int sample_index, const MistOutTables *tables, void *stream) {
  if (int rc = check_common(problem, d_groups, n_groups)) return rc;
  if (!d_block_prefix || !d_partial_cost || !d_partial_index) return fail(MIST_E_INVALID, "null pointer argument");
  ReduceTables tabs;
  if (int rc = reduce_tables(problem, 1, const_cast<double *>(d_partial_cost),
                             const_cast<int32_t *>(d_partial_index), &tabs))
    return rc;
  return launch_finalize(problem, d_groups, n_groups, d_row_terms, tabs, &sample_index, tables, stream);
}

// Second stream and events of mist_intra_stage_eval, one set per device, kept for the life of
// the process.
namespace {
struct OverlapStreams {
  hipStream_t side = nullptr;
  hipEvent_t rows_ready = nullptr, seeds_done = nullptr;
};
std::mutex g_enqueue_lock;  // one call's records and waits on the shared events are a unit
int overlap_streams(OverlapStreams **out) {
  static std::mutex lock;
  static OverlapStreams known[64];
  int device = 0;
  MIST_HIP_CHECK(hipGetDevice(&device));
  if (device < 0 || device >= 64) return fail(MIST_E_INVALID, "device ordinal %d outside [0, 64)", device);
  std::lock_guard<std::mutex> guard(lock);
  OverlapStreams &s = known[device];
  if (s.side == nullptr) {
    MIST_HIP_CHECK(hipStreamCreateWithFlags(&s.side, hipStreamNonBlocking));  // default priority
    MIST_HIP_CHECK(hipEventCreateWithFlags(&s.rows_ready, hipEventDisableTiming));
    MIST_HIP_CHECK(hipEventCreateWithFlags(&s.seeds_done, hipEventDisableTiming));
  }
  *out = &s;
  return 0;
}
}  // namespace

int mist_intra_stage_eval_samples(const MistProblem *problem, const MistGroupDesc *d_groups,
                                  int n_groups, const int32_t *d_terms_block_prefix,
                                  int n_terms_blocks, const int32_t *d_reduce_block_prefix,
                                  int n_reduce_blocks, const int32_t *d_scout_prefix,
                                  int n_scout_blocks, double *d_row_terms, double *d_stage_floor,
                                  double *d_key_terms, double *d_partial_cost,
                                  int32_t *d_partial_index, const double *ratios,
                                  const int32_t *sample_index, int n_samples, int sample_batch,
                                  int main_batch, const MistOutTables *tables, void *stream) {
  if (!ratios || !sample_index || n_samples < 1)
    return fail(MIST_E_INVALID, "n_samples %d < 1 or null sample lists", n_samples);
  if (sample_batch < 1 || sample_batch > MIST_MAX_SAMPLE_BATCH)
    return fail(MIST_E_INVALID, "sample_batch %d outside [1, %d]", sample_batch, MIST_MAX_SAMPLE_BATCH);
  if (main_batch < 1 || main_batch > sample_batch)
    return fail(MIST_E_INVALID, "main_batch %d outside [1, sample_batch = %d]", main_batch, sample_batch);
  if (int rc = check_reduce_arguments(problem, d_groups, n_groups, d_reduce_block_prefix,
                                      n_reduce_blocks, d_scout_prefix, n_scout_blocks,
                                      d_row_terms, d_stage_floor, d_partial_cost, d_partial_index))
    return rc;
  if (!d_terms_block_prefix || n_terms_blocks <= 0)
    return fail(MIST_E_INVALID, "null / empty row-term decomposition");
  if (int rc = check_factors(problem)) return rc;
  for (int i = 0; i < n_samples; ++i)
    if (!(ratios[i] >= 0.0)) return fail(MIST_E_INVALID, "ratio %d must be non-negative", i);
  hipStream_t main_stream = (hipStream_t)stream;
  // The seeds read a few hundred rows per group and leave most of the GPU idle; the stage summaries
  // are computed beside them.  Stream order: [terms of the gathered rows] -> side stream: seeds of
  // the first batch of samples || this stream: key terms, summaries -> filter, open, rows of the
  // opened stages, reduce, resolve, finalize; further batches one after the other.
  const bool overlap = n_scout_blocks > 0 && problem->max_scout_rows > 0 && has_key_terms(problem, n_groups, d_key_terms);
  const bool by_need = overlap;
  OverlapStreams *os = nullptr;
  std::unique_lock<std::mutex> enqueue_guard;
  if (overlap) {
    if (int rc = overlap_streams(&os)) return rc;
    // the second stream and its events are shared by all callers: one call's records and waits
    // are enqueued as a unit
    enqueue_guard = std::unique_lock<std::mutex>(g_enqueue_lock);
    const unsigned scout_term_blocks = (unsigned)((problem->max_scout_rows + kTermsBlock - 1) / kTermsBlock);
    hipLaunchKernelGGL((row_terms_kernel<1, false>), dim3(scout_term_blocks, n_groups),
                       dim3(kTermsBlock), 0, main_stream, *problem, d_groups, n_groups,
                       d_terms_block_prefix, d_row_terms, d_stage_floor, nullptr);
    MIST_HIP_CHECK(hipGetLastError());
    MIST_HIP_CHECK(hipEventRecord(os->rows_ready, main_stream));
    MIST_HIP_CHECK(hipStreamWaitEvent(os->side, os->rows_ready, 0));
    // (the summaries are queued first: the seeds are several launches, and this stream would idle
    // while they are made)
    bool from_keys = false;
    if (int rc = launch_key_terms(problem, d_groups, n_groups, d_key_terms, main_stream, &from_keys))
      return rc;
    launch_stage_floors(problem, d_groups, n_groups, d_terms_block_prefix, n_terms_blocks, d_stage_floor, d_key_terms,
                        main_stream);
    MIST_HIP_CHECK(hipGetLastError());
  } else {
    if (int rc = mist_row_terms(problem, d_groups, n_groups, d_terms_block_prefix, n_terms_blocks,
                                d_row_terms, d_stage_floor, d_key_terms, stream))
      return rc;
  }
  const int batch = samples_together(problem, sample_batch);
  for (int first = 0; first < n_samples; first += batch) {
    const int count = std::min(batch, n_samples - first);
    ReduceTables tabs;
    if (int rc = reduce_tables(problem, count, d_partial_cost, d_partial_index, &tabs, !by_need)) return rc;
    RatioList list = {};
    for (int i = 0; i < count; ++i) list.r[i] = ratios[first + i];
    const bool aside = overlap && first == 0;
    MistProblem own = closing(problem, n_groups, count);
    // for an assignment only the estimate is formed beside the summaries: they leave few pairs to seed
    const bool assignment = own.incumbent_close == kCloseAssignment;
    void *const beside = aside ? (void *)os->side : stream;
    if (assignment) {
      if (first == 0 && n_scout_blocks > 0 && own.incumbent_first_estimate != 0)
        if (int rc = launch_first_estimate(&own, d_groups, n_groups, d_row_terms, 1.0, d_partial_cost, nullptr, beside)) return rc;
      own.incumbent_first_estimate = 0;
    } else if (int rc = launch_seeds(&own, d_groups, n_groups, d_row_terms, list, n_scout_blocks > 0, tabs, d_partial_cost,
                                     beside)) {
      return rc;
    }
    if (aside) MIST_HIP_CHECK(hipEventRecord(os->seeds_done, os->side));
    // (the summaries' place depends on the number of samples)
    if (int rc = launch_super_floors(&own, d_groups, n_groups, d_stage_floor, list.r[0], tabs, stream)) return rc;
    if (aside) MIST_HIP_CHECK(hipStreamWaitEvent(main_stream, os->seeds_done, 0));
    if (own.incumbent_close != 0)
      if (int rc = launch_incumbent(&own, d_groups, n_groups, tabs, stream)) return rc;
    if (assignment)
      if (int rc = launch_seeds(&own, d_groups, n_groups, d_row_terms, list, n_scout_blocks > 0, tabs, d_partial_cost, stream))
        return rc;
    if (int rc = launch_reduce(&own, d_groups, n_groups, d_reduce_block_prefix, n_reduce_blocks, d_row_terms,
                               d_stage_floor, d_key_terms, list, tabs, stream))
      return rc;
    if (int rc = launch_finalize(problem, d_groups, n_groups, d_row_terms, tabs, sample_index + first, tables, stream))
      return rc;
  }
  return 0;
}

int mist_intra_stage_eval(const MistProblem *problem, const MistGroupDesc *d_groups,
                          int n_groups, const int32_t *d_terms_block_prefix, int n_terms_blocks,
                          const int32_t *d_reduce_block_prefix, int n_reduce_blocks,
                          const int32_t *d_scout_prefix, int n_scout_blocks, double *d_row_terms,
                          double *d_stage_floor, double *d_key_terms, double *d_partial_cost,
                          int32_t *d_partial_index, double ratio, int sample_index,
                          int compute_terms, const MistOutTables *tables, void *stream) {
  if (compute_terms)
    return mist_intra_stage_eval_samples(problem, d_groups, n_groups, d_terms_block_prefix, n_terms_blocks,
                                         d_reduce_block_prefix, n_reduce_blocks, d_scout_prefix, n_scout_blocks,
                                         d_row_terms, d_stage_floor, d_key_terms, d_partial_cost, d_partial_index,
                                         &ratio, &sample_index, 1, 1, 1, tables, stream);
  if (int rc = mist_eval_reduce(problem, d_groups, n_groups, d_reduce_block_prefix,
                                n_reduce_blocks, d_scout_prefix, n_scout_blocks, d_row_terms,
                                d_stage_floor, ratio, d_partial_cost, d_partial_index, stream))
    return rc;
  return mist_finalize(problem, d_groups, n_groups, d_reduce_block_prefix, d_row_terms,
                       d_partial_cost, d_partial_index, sample_index, tables, stream);
}

int mist_row_diagnostics(const MistProblem *problem, const MistGroupDesc *d_groups, int n_groups,
                         const int32_t *d_requests, int n_requests, double *d_out, void *stream) {
  if (int rc = check_common(problem, d_groups, n_groups)) return rc;
  if (!d_requests || !d_out) return fail(MIST_E_INVALID, "null pointer");
  if (n_requests <= 0) return fail(MIST_E_INVALID, "n_requests must be positive, got %d", n_requests);
  if (int rc = check_factors(problem)) return rc;
  hipLaunchKernelGGL(row_diagnostics_kernel, dim3((n_requests + kTermsBlock - 1) / kTermsBlock),
                     dim3(kTermsBlock), 0, (hipStream_t)stream, *problem, d_groups, n_groups,
                     d_requests, n_requests, d_out);
  MIST_HIP_CHECK(hipGetLastError());
  return 0;
}

int mist_stage_analyze(const MistProblem *problem, const MistGroupDesc *d_groups, int n_groups,
                       const double *d_row_terms, const int32_t *d_requests, int n_requests,
                       double *d_out, void *stream) {
  if (int rc = check_common(problem, d_groups, n_groups)) return rc;
  if (!d_row_terms || !d_requests || !d_out) return fail(MIST_E_INVALID, "null pointer");
  if (n_requests <= 0) return fail(MIST_E_INVALID, "n_requests must be positive, got %d", n_requests);
  hipLaunchKernelGGL(analyze_kernel, dim3((n_requests + 63) / 64), dim3(64), 0, (hipStream_t)stream,
                     *problem, d_groups, n_groups, d_row_terms, d_requests, n_requests, d_out);
  MIST_HIP_CHECK(hipGetLastError());
  return 0;
}

}  // extern "C"
