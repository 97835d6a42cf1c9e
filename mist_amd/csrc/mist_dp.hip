// Inter-stage pipeline-partition DP on MI355X (gfx950).
//
// The stage index s is the sequential axis.  The (threshold, start layer k, devices d) states
// of one s are independent; each is scanned by one thread (or a team of lanes) that walks its
// (mesh, end layer, ckpt) candidates in the reference's order with float32 adds and strict "<",
// so ties resolve exactly as in the reference loop nest (mist/analyzer/inter_tuning.py:298-333).
// Schedules: one launch per s with the states of all instances spread over the GPU
// (dp_step_kernel); one workgroup per instance that loops over s itself, with its state planes in
// LDS (dp_fused_kernel) or only the one it reads at random (dp_plane_kernel); and, where no
// back-pointers are asked for, dp_history_kernel, which finds winners on the answer's path alone.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <cstdlib>
#include <map>
#include <tuple>
#include <mutex>
#include <set>
#include <type_traits>
#include <utility>

#include "mist_common.h"
#include "mist_dp.h"
#include "mist_dp_rates.h"

namespace {

using mist::fail;

constexpr int kDpThreads = 64;  // one wavefront per workgroup
constexpr int kDpWideTeam = 8;  // lanes that share one DP state in small batches
constexpr size_t kDpLdsPerCu = 160 * 1024;  // LDS of a gfx950 compute unit
constexpr int kDpFusedThreads = 1024;  // largest workgroup of the one-launch kernel
constexpr int kDpFusedMinInstances = 64;  // threshold batches of at least this size use it
constexpr int kDpFusedSmallPlane = 2048;  // (L + 1)(D + 1) up to which every batch uses it
constexpr int kDpStageBatch = 8;   // row minima a lane copies together in the one-launch kernel
constexpr int kSelectBatch = 8;  // table values a lane of the candidate selection reads together
constexpr int kSelectSegments = 3 * MIST_MAX_MESH;  // runs of neighbouring values it reads
constexpr int kSelectBuffer = 4096;  // selected values a workgroup holds before it appends them
constexpr float kDpNoThreshold = 3.402823466e+38f;  // FLT_MAX: admits every finite stage cost
constexpr int kDpBatch = 4;  // end layers whose reads a lane of the one-lane-per-state kernel overlaps

// ------------------------------------------------------------------------------------------
// Adapter: float64 (stable, delta) tables -> float32 DP cost tables for every g.
// ------------------------------------------------------------------------------------------
// Table rows (fixed g, mesh, p, layers) hold the L+1 ckpt entries: cost = (float)stable +
// (float)delta / G, and alongside its running minimum pmin[j] = min(cost[0..j]).  A workgroup
// takes sets of whole rows, so that loads and stores are contiguous; the running minimum is a
// segmented scan (lane shifts, LDS between the wavefronts a row spans).
// Most cells of a plan hold no strategy (no group for that (g, mesh), or nothing fits): their
// row index is -1 and their costs +inf, so with the index table (may be null) the 16 bytes of
// such a cell's costs are not read.
// The four tables of a call (base, with_pre, with_post, no_pp) go through one launch: table v
// owns the workgroups first_block[v] .. first_block[v + 1] - 1.  A workgroup takes up to kCostRuns sets
// of rows one after the other: with one each, its own start and a division per lane were the bound.
// Small tables, whose workgroups are all resident, take fewer (1.3B on 1x2: eight 14.4 us, one 5.3).
// Bound: 12 bytes a cell and 16 more where it holds a row.
constexpr int kCostRuns = 8;
constexpr int kCostResident = 2048;  // workgroups at a time, eight per CU
struct CostTableJob {
  const double *stable[4], *delta[4];
  const int32_t *index[4];
  float *out[4], *pmin[4];
  int64_t n_rows[4], rows_per_g[4];
  unsigned first_block[5];
  int runs;  // sets of rows per workgroup
};
// `run` of the lane `control` names, where it is `distance` back in the same row of the table;
// a lane without a source keeps its own
#define MIST_RUN_DPP(run, back, control, rows, distance)                                          \
  {                                                                                               \
    const int other = __builtin_amdgcn_update_dpp(__float_as_int(run), __float_as_int(run),       \
                                                  control, rows, 0xf, false);                     \
    run = (back) >= (distance) ? fminf(run, __int_as_float(other)) : run;                         \
  }
// running minimum over the lanes of a wavefront; `back`: lanes since the row's first
__device__ __forceinline__ float running_minimum(float run, int back) {
  const int lane = threadIdx.x & 63;
  MIST_RUN_DPP(run, back, 0x111, 0xf, 1)  // row_shr:1
  MIST_RUN_DPP(run, back, 0x112, 0xf, 2)
  MIST_RUN_DPP(run, back, 0x114, 0xf, 4)
  MIST_RUN_DPP(run, back, 0x118, 0xf, 8)
  MIST_RUN_DPP(run, back, 0x142, 0xa, (lane & 15) + 1)  // row_bcast:15 into the odd rows of 16 lanes
  MIST_RUN_DPP(run, back, 0x143, 0xc, lane - 31)        // row_bcast:31 into the upper half
  return run;
}
#undef MIST_RUN_DPP

// Four neighbouring cells per lane, in as many rows (a multiple of four, so that each set begins at
// 16 bytes) as 1024 cells hold; one sample, rows of up to 256 cells: a row lies in two wavefronts at
// most.  (A cell per lane: 95 vector instructions for 64 cells and the stores of 4 bytes, 70B on 32x8
// with its 4.5e8 cells 2.03 ms; now 1.06, 5.1 TB/s; 7B on 4x8 0.084 -> 0.047.)
constexpr int kCostCells = 1024;
// (a table may begin at any of its elements; loads and stores of 16 bytes need 4)
typedef int AnyInt4 __attribute__((ext_vector_type(4), aligned(4)));
typedef float AnyFloat4 __attribute__((ext_vector_type(4), aligned(4)));
typedef double AnyDouble2 __attribute__((ext_vector_type(2), aligned(8)));
// A lane's four cells of a set of rows.
struct CostLane {
  int cell0, row[4], j[4];
  int back;     // lanes to where the last cell's row begins
  bool spills;  // the first cell's begins in an earlier wavefront
  __device__ __forceinline__ explicit CostLane(int row_len) : cell0((int)threadIdx.x * 4) {
    row[0] = cell0 / row_len;
    j[0] = cell0 - row[0] * row_len;
#pragma unroll
    for (int u = 1; u < 4; ++u) {
      const bool next = j[u - 1] + 1 == row_len;
      row[u] = row[u - 1] + next;
      j[u] = next ? 0 : j[u - 1] + 1;
    }
    back = min((int)threadIdx.x - ((cell0 + 3 - j[3]) >> 2), (int)(threadIdx.x & 63));
    spills = cell0 - j[0] < (int)(threadIdx.x >> 6) * 256;
  }
};
// Costs of a set and their running minima, by the whole workgroup; `ends`: four floats that the set before
// does not use.
__device__ __forceinline__ void store_costs(const CostLane &at, const float (&c)[4], int n_mine, float *__restrict__ out,
                                            float *__restrict__ pmin, float *ends) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  float run = INFINITY;
#pragma unroll
  for (int u = 0; u < 4; ++u) run = fminf(c[u], at.j[u] == 0 ? INFINITY : run);
  run = running_minimum(run, at.back);
  if (lane == 63) ends[wave] = run;
  __syncthreads();
  run = __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(INFINITY), __float_as_int(run), 0x138, 0xf, 0xf,
                                                   false));  // wave_shr:1
  if (at.spills) run = fminf(run, ends[wave - 1]);
  float m[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) m[u] = run = fminf(c[u], at.j[u] == 0 ? INFINITY : run);
  if (n_mine == 4) {
    *reinterpret_cast<AnyFloat4 *>(out) = AnyFloat4{c[0], c[1], c[2], c[3]};
    *reinterpret_cast<AnyFloat4 *>(pmin) = AnyFloat4{m[0], m[1], m[2], m[3]};
  } else {
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (u < n_mine) {
        out[u] = c[u];
        pmin[u] = m[u];
      }
  }
}
__global__ __launch_bounds__(256) void cost_rows_kernel(const CostTableJob job, const int32_t *__restrict__ grad_accum,
                                                        int row_len) {
  __shared__ float ends[2][4];
  const int v = (blockIdx.x >= job.first_block[1]) + (blockIdx.x >= job.first_block[2]) +
                (blockIdx.x >= job.first_block[3]);
  const double *__restrict__ stable = job.stable[v], *__restrict__ delta = job.delta[v];
  const int32_t *__restrict__ index = job.index[v];
  float *__restrict__ out = job.out[v], *__restrict__ pmin = job.pmin[v];
  const int64_t n_rows = job.n_rows[v], per_g = job.rows_per_g[v];
  const int rows_here = (kCostCells / row_len) & ~3, cells_here = rows_here * row_len;
  const CostLane at_lane(row_len);
  const int cell0 = at_lane.cell0;
  const int(&its_row)[4] = at_lane.row;
  const int64_t row0 = (int64_t)(blockIdx.x - job.first_block[v]) * rows_here * job.runs;
  int64_t g = row0 / per_g, in_g = row0 - g * per_g;
  for (int turn = 0; turn < job.runs; ++turn) {
    const int64_t row = row0 + turn * rows_here;
    if (row >= n_rows) break;
    const int n_cells = (int)min((int64_t)cells_here, (n_rows - row) * row_len);
    const int n_mine = min(n_cells - cell0, 4);
    const int64_t i = row * row_len + cell0;
    const int until = (int)min(per_g - in_g, (int64_t)rows_here);  // rows of g
    float c[4];
    bool holds[4];
    if (n_mine == 4) {
      const AnyInt4 at = index == nullptr ? AnyInt4{0, 0, 0, 0} : *reinterpret_cast<const AnyInt4 *>(index + i);
      holds[0] = at.x >= 0;
      holds[1] = at.y >= 0;
      holds[2] = at.z >= 0;
      holds[3] = at.w >= 0;
    } else {
#pragma unroll
      for (int u = 0; u < 4; ++u) holds[u] = u < n_mine && (index == nullptr || index[i + u] >= 0);
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) c[u] = INFINITY;
    if (holds[0] || holds[1] || holds[2] || holds[3]) {
      double its_stable[4], its_delta[4];
      if (n_mine == 4) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const AnyDouble2 s = reinterpret_cast<const AnyDouble2 *>(stable + i)[h];
          const AnyDouble2 d = reinterpret_cast<const AnyDouble2 *>(delta + i)[h];
          its_stable[2 * h] = s.x;
          its_stable[2 * h + 1] = s.y;
          its_delta[2 * h] = d.x;
          its_delta[2 * h + 1] = d.y;
        }
      } else {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          its_stable[u] = holds[u] ? stable[i + u] : 0.0;
          its_delta[u] = holds[u] ? delta[i + u] : 0.0;
        }
      }
      const float first_G = (float)grad_accum[g];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        float G = first_G;
        if (holds[u] && its_row[u] >= until) {
          int64_t its_g = g + 1;
          for (int64_t past = its_row[u] - until; past >= per_g; past -= per_g) ++its_g;
          G = (float)grad_accum[its_g];
        }
        const float cost = (float)its_stable[u] + (float)its_delta[u] / G;
        c[u] = holds[u] ? cost : INFINITY;
      }
    }
    for (in_g += rows_here; in_g >= per_g; in_g -= per_g) ++g;
    store_costs(at_lane, c, n_mine, out + i, pmin + i, ends[turn & 1]);
  }
}

// Only the planes of the p axis that hold something (MistDpCosts.planes): workgroups of a (g, mesh) take its
// sets of rows in turn, table after table.  The cells of a row that the reference never writes are known by
// their place, so that no fill of the row indices comes before: c > l, and c == l - 1 except at p == 0 of base /
// with_pre.  Bound: 12 bytes a cell of the planes, and latency: a set is two dependent reads and a barrier.
// (70B on 32x8, where 21 % of the planes hold something: fill 254 us and every cell 1063 -> 243; 13B on 8x8 26 and
// 98 -> 41; 7B on 4x8 12 and 46 -> 22.)
constexpr int64_t kCostPlaneBlocks = 16384;
struct CostPlanesJob {
  const double *stable[4], *delta[4];
  const int32_t *index[4];
  float *out[4], *pmin[4];
  const int32_t *planes, *grad_accum;
  int L, P1;
};
__global__ __launch_bounds__(256) void cost_planes_kernel(const CostPlanesJob job) {
  __shared__ float ends[2][4];
  const int L = job.L, P1 = job.P1, row_len = L + 1, q = blockIdx.y, Q = gridDim.y;
  const int64_t gq = (int64_t)blockIdx.z * Q + q;
  const int planes = min(job.planes[gq], P1);
  if (planes <= 0) return;
  const float G = (float)job.grad_accum[blockIdx.z];
  const int rows_here = (kCostCells / row_len) & ~3;
  const CostLane at_lane(row_len);
  const int wide_sets = (planes * L + rows_here - 1) / rows_here, post_sets = (L + rows_here - 1) / rows_here;
  const int n_sets = 2 * wide_sets + post_sets + 1;
  for (int set = blockIdx.x, turn = 0; set < n_sets; set += gridDim.x, ++turn) {
    const int v = set < wide_sets ? 0 : set < 2 * wide_sets ? 1 : set < 2 * wide_sets + post_sets ? 2 : 3;
    const int row0 = (v == 3 ? 0 : set - (v == 0 ? 0 : v * wide_sets)) * rows_here;
    const int n_rows = v < 2 ? planes * L : v == 2 ? L : 1;
    const int64_t first = (v < 2 ? gq * P1 * L : v == 2 ? gq * L : gq) * row_len;  // cell of the (g, mesh)'s row 0
    const int n_cells = min(rows_here, n_rows - row0) * row_len, n_mine = min(n_cells - at_lane.cell0, 4);
    const int64_t i = first + (int64_t)row0 * row_len + at_lane.cell0;
    float c[4] = {INFINITY, INFINITY, INFINITY, INFINITY};
    if (n_mine > 0) {
      int32_t index[4] = {-1, -1, -1, -1};
      if (n_mine == 4) {
        const AnyInt4 four = *reinterpret_cast<const AnyInt4 *>(job.index[v] + i);
        index[0] = four.x, index[1] = four.y, index[2] = four.z, index[3] = four.w;
      } else {
#pragma unroll
        for (int u = 0; u < 4; ++u)
          if (u < n_mine) index[u] = job.index[v][i + u];
      }
      int p = (row0 + at_lane.row[0]) / L, l = v == 3 ? L : row0 + at_lane.row[0] - p * L + 1;
      bool holds[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        if (u > 0 && at_lane.j[u] == 0) {  // the next row
          const bool wraps = l == L;
          p += wraps;
          l = wraps ? 1 : l + 1;
        }
        const bool written = at_lane.j[u] <= l && (at_lane.j[u] != l - 1 || (v < 2 && p == 0));
        holds[u] = u < n_mine && written && index[u] >= 0;
      }
      if (holds[0] || holds[1] || holds[2] || holds[3]) {
        double its_stable[4], its_delta[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          its_stable[u] = u < n_mine ? job.stable[v][i + u] : 0.0;
          its_delta[u] = u < n_mine ? job.delta[v][i + u] : 0.0;
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const float cost = (float)its_stable[u] + (float)its_delta[u] / G;
          c[u] = holds[u] ? cost : INFINITY;
        }
      }
    }
    store_costs(at_lane, c, n_mine, job.out[v] + i, job.pmin[v] + i, ends[turn & 1]);
  }
}

// Any row length and sample position: a cell per lane.
__global__ __launch_bounds__(256) void cost_table_kernel(const CostTableJob job,
                                                         const int32_t *__restrict__ grad_accum,
                                                         int row_len, int sample_size, int slot) {
  __shared__ float lds[256];
  const int v = (blockIdx.x >= job.first_block[1]) + (blockIdx.x >= job.first_block[2]) +
                (blockIdx.x >= job.first_block[3]);
  const double *__restrict__ stable = job.stable[v], *__restrict__ delta = job.delta[v];
  const int32_t *__restrict__ index = job.index[v];
  float *__restrict__ out = job.out[v], *__restrict__ pmin = job.pmin[v];
  const int64_t n_rows = job.n_rows[v], rows_per_g = job.rows_per_g[v];
  const int seg = min(row_len, 256);  // entries of a row per pass
  const int rows_here = 256 / seg;
  const int local_row = threadIdx.x / seg, j0 = threadIdx.x % seg;
  // (rows_per_g is the size of one g: 32 bits)
  const uint32_t per_g = (uint32_t)rows_per_g;
  const int64_t row0 = (int64_t)(blockIdx.x - job.first_block[v]) * rows_here * job.runs;
  const int64_t g0 = row0 >> 32 == 0 ? (int64_t)((uint32_t)row0 / per_g) : row0 / rows_per_g;
  const uint32_t in_g0 = (uint32_t)(row0 - g0 * rows_per_g);
  for (int turn = 0; turn < job.runs; ++turn) {
    const uint32_t ahead = (uint32_t)(turn * rows_here + local_row);
    const int64_t r = row0 + ahead;
    if (row0 + turn * rows_here >= n_rows) break;
    const bool live_row = local_row < rows_here && r < n_rows;
    const float G = live_row ? (float)grad_accum[g0 + (in_g0 + ahead) / per_g] : 1.0f;
    float carry = INFINITY;
    for (int base = 0; base < row_len; base += seg) {
      const int j = base + j0;
      const bool live = live_row && j < row_len;
      const int64_t i = r * row_len + j;
      float c = INFINITY;
      if (live) {
        if (index == nullptr || index[i * sample_size + slot] >= 0) {
          const float s = (float)stable[i * sample_size + slot];
          const float d = (float)delta[i * sample_size + slot];
          c = s + d / G;
        }
        out[i] = c;
      }
      // running minimum over the row's lanes of this pass: inside a wavefront by lane shifts that stop
      // at the row's first lane, then the part of the row that lies in earlier wavefronts (their
      // last lanes hold it)
      float run = running_minimum(c, j0);
      lds[threadIdx.x] = run;
      __syncthreads();
      const int row_first = (int)threadIdx.x - j0;
      for (int at = (int)(threadIdx.x & ~63u) - 1; at >= row_first; at -= 64) run = fminf(run, lds[at]);
      if (live) pmin[i] = fminf(run, carry);
      if (base + seg < row_len)  // only rows longer than one pass: then the row is the workgroup
        carry = fminf(carry, fminf(fminf(lds[63], lds[127]), fminf(lds[191], lds[255])));
      __syncthreads();
    }
  }
}

// Counters and instance slots of a first batch before it: one launch (two fills of the runtime take three, 5 us
// of the chain each).
__global__ __launch_bounds__(256) void window_clear_kernel(int32_t *__restrict__ counts, int n_counts,
                                                           int32_t *__restrict__ inst_row, int n_inst) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < n_counts) counts[i] = 0;
  if (i < n_inst) inst_row[i] = -1;
}

// ------------------------------------------------------------------------------------------
// t_max candidates of a value window: one pass over the three cost tables of a table row g
// (costs, with_pre, with_post; inter_tuning.py:180-186).  Request r selects the finite values v
// of row rows[r] with lo[r] < v <= hi[r]; they are appended, unordered, to one output list as
// (value, request) pairs; counts[0] = pairs wanted in total (may exceed the capacity, then the
// caller retries with a larger list), counts[1 + r] = finite values of request r above hi[r].
// ------------------------------------------------------------------------------------------
// With `per_request` every request appends to a list of its own instead, out_values[r][capacity],
// counted in counts[1 + n_requests + r] (then counts[0] and out_request are not touched).
__global__ __launch_bounds__(256) void select_candidates_kernel(
    const MistDpCosts tabs, const int32_t *__restrict__ rows, const float *__restrict__ lo,
    const float *__restrict__ hi, float *__restrict__ out_values, int32_t *__restrict__ out_request,
    int capacity, int32_t *__restrict__ counts, bool per_request) {
  // Selected values collect in LDS and leave in one piece: appends to the one output list go
  // through a single counter, and an atomic per wavefront round (thousands per launch) made
  // that counter the bottleneck of the kernel.
  __shared__ float kept[kSelectBuffer];
  __shared__ int n_kept, flush_at;
  __shared__ int above_of_wave[4];
  const int r = blockIdx.y;
  const int64_t g = rows[r];
  const int64_t n0 = tabs.g_stride[0], n1 = tabs.g_stride[1], n2 = tabs.g_stride[2];
  const float lo_r = lo[r], hi_r = hi[r];
  if (lo_r == INFINITY && hi_r == INFINITY) return;  // (nothing is feasible there)
  const int lane = threadIdx.x & 63;
  int above = 0;
  if (threadIdx.x == 0) n_kept = 0;
  __syncthreads();
  int32_t *list_count = per_request ? &counts[1 + gridDim.y + r] : &counts[0];
  float *list = per_request ? out_values + (int64_t)r * capacity : out_values;
  auto flush = [&]() {  // called by the whole workgroup
    if (threadIdx.x == 0) flush_at = n_kept > 0 ? atomicAdd(list_count, n_kept) : 0;
    __syncthreads();
    for (int i = threadIdx.x; i < n_kept; i += blockDim.x) {
      const int at = flush_at + i;
      if (at < capacity) {
        list[at] = kept[i];
        if (!per_request) out_request[at] = r;
      }
    }
    __syncthreads();
    if (threadIdx.x == 0) n_kept = 0;
    __syncthreads();
  };
  // Batches of kSelectBatch values per lane, the next one on its way while one is tried, from segments of
  // neighbouring values: the three tables, or per table and mesh the planes that hold something.  (Every value
  // of the tables, the reads of a batch behind its barriers: 70B on 32x8 318 us, 7B on 4x8 21; the planes alone
  // 200, and 80 and 16 with the next batch on its way.)
  constexpr int kBatch = kSelectBatch * 256;
  __shared__ const float *segment_from[kSelectSegments];
  __shared__ int64_t segment_cells[kSelectSegments], segment_end[kSelectSegments];  // (the latter in batches)
  const int meshes = tabs.planes == nullptr ? 1 : (int)tabs.planes_g_stride, n_segments = 3 * meshes;
  if (threadIdx.x < 64) {  // lane = segment
    const int v = lane / meshes, q = lane - v * meshes;
    const int64_t of_mesh = (v == 0 ? n0 : v == 1 ? n1 : n2) / meshes;
    int64_t cells = 0;
    if (lane < n_segments) {
      cells = of_mesh;
      if (tabs.planes != nullptr) {
        const int held = tabs.planes[g * meshes + q];
        // (n2: one plane of every mesh; never more than the p axis, as in cost_planes_kernel)
        cells = v < 2 ? min(max(held, 0) * (n2 / meshes), of_mesh) : held > 0 ? of_mesh : 0;
      }
    }
    int64_t end = (cells + kBatch - 1) / kBatch;
    for (int step = 1; step < 64; step <<= 1) {
      const int64_t before = __shfl_up((long long)end, step);
      if (lane >= step) end += before;
    }
    if (lane < n_segments) {
      segment_from[lane] = (v == 0 ? tabs.costs + g * n0 : v == 1 ? tabs.costs_pre + g * n1 : tabs.costs_post + g * n2) +
                           q * of_mesh;
      segment_cells[lane] = cells;
      segment_end[lane] = end;
    }
  }
  __syncthreads();
  int segment = 0;
  auto read = [&](int64_t batch, float (&value)[kSelectBatch]) {
    while (segment < n_segments && segment_end[segment] <= batch) ++segment;
    if (segment >= n_segments) return false;
    const int64_t at = (batch - (segment > 0 ? segment_end[segment - 1] : 0)) * kBatch;
    const float *__restrict__ from = segment_from[segment] + at;
    const int left = (int)min(segment_cells[segment] - at, (int64_t)kBatch);
#pragma unroll
    for (int u = 0; u < kSelectBatch; ++u) {
      const int in_batch = u * 256 + (int)threadIdx.x;
      const float v = from[min(in_batch, left - 1)];
      value[u] = in_batch < left ? v : INFINITY;
    }
    return true;
  };
  float value[kSelectBatch], ahead[kSelectBatch];
  bool more = read(blockIdx.x, value);
  for (int64_t batch = blockIdx.x; more;) {
    more = read(batch += gridDim.x, ahead);
#pragma unroll
    for (int u = 0; u < kSelectBatch; ++u) {
      const float v = value[u];
      const bool finite = v < INFINITY;  // +inf (nothing feasible) and NaN are not candidates
      above += finite && v > hi_r;
      const bool take = finite && v > lo_r && v <= hi_r;
      // one LDS atomic per wavefront reserves the slots of all its selected values
      const unsigned long long takers = __ballot(take);
      if (takers != 0) {
        const int leader = __ffsll(takers) - 1;
        int first = 0;
        if (lane == leader) first = atomicAdd(&n_kept, __popcll(takers));
        first = __shfl(first, leader);
        if (take) kept[first + __popcll(takers & ((1ull << lane) - 1))] = v;
      }
    }
    __syncthreads();
    // Room for another round of kSelectBatch values per thread?  Every wave reads the count
    // before any wave adds to it again (second barrier), so the whole workgroup takes the
    // same branch and flush()'s barriers are reached by all of its waves.
    const int kept_now = n_kept;
    __syncthreads();
    if (kept_now > kSelectBuffer - kSelectBatch * 256) flush();
#pragma unroll
    for (int u = 0; u < kSelectBatch; ++u) value[u] = ahead[u];
  }
  flush();
  // one atomic per workgroup for the "above" count
  for (int step = 32; step >= 1; step >>= 1) above += __shfl_xor(above, step);
  if (lane == 0) above_of_wave[threadIdx.x >> 6] = above;
  __syncthreads();
  if (threadIdx.x == 0) {
    const int total = above_of_wave[0] + above_of_wave[1] + above_of_wave[2] + above_of_wave[3];
    if (total > 0) atomicAdd(&counts[1 + r], total);
  }
}

// ------------------------------------------------------------------------------------------
// The reference's gap rule (inter_tuning.py:198) and the start of a walk that does not begin at
// the bottom of the candidate list (see mist_dp_window_begin in mist_dp.h): the same code for
// the host entry points and for the kernel that walks the windows on the device.
// ------------------------------------------------------------------------------------------
// "t - last < 1e-6" as the reference evaluates it: float32 difference, float64 comparison
__host__ __device__ inline bool gap_below(float t, float last, double gap) {
  const float diff = t - last;
  return (double)diff < gap;
}
// Index the walk over `ascending` starts at, or -1 when the fetched part holds no certain start.
__host__ __device__ inline int window_walk_start(const float *ascending, int n, float lo,
                                                 bool open_below, float start_value, double gap) {
  // A candidate whose predecessor is at least the gap below it is kept whatever the walk did
  // before; the predecessor of the first fetched candidate is unknown unless the fetch was open
  // below.
  int first = -1;
  for (int i = 0; i < n && ascending[i] <= start_value; ++i) {
    const float prev = i == 0 ? (open_below ? 0.0f : lo) : ascending[i - 1];
    const bool certain = !gap_below(ascending[i], prev, gap) || (i == 0 && open_below);
    if (certain) first = i;
  }
  if (first < 0) {
    const bool certain0 = !gap_below(ascending[0], open_below ? 0.0f : lo, gap) || open_below;
    if (ascending[0] > start_value && certain0) first = 0;
  }
  return first;
}

// Which kept threshold (counted from the first one at or above the smallest feasible threshold)
// instance k of a window's first scan batch runs, when n_avail of them are there: all of them if
// they fit the batch; else the first `first_lead` ones, then the rest of the batch spread evenly
// up to the window's last one (probes: the stage-cost sum at a later threshold bounds the sums at
// every earlier one from below, which lets the scan pass thresholds that cannot improve its best).
__host__ __device__ __forceinline__ int dp_first_batch_index(int k, int n_avail, int first_chunk,
                                                             int first_lead) {
  if (n_avail <= first_chunk || k < first_lead || first_lead >= first_chunk) return k;
  const int spread = first_chunk - first_lead;
  return first_lead + (int)(((int64_t)(k - first_lead + 1) * (n_avail - first_lead)) / spread) - 1;
}

constexpr int kWindowThreads = 1024;
constexpr int kWindowMost = 32768;      // values of a window that is walked on the device ...
constexpr int kWindowDistinct = 16384;  // ... and different ones among them
constexpr int kWindowHeld = kWindowMost / kWindowThreads, kWindowOwn = kWindowDistinct / kWindowThreads;
constexpr int kWindowProbes = 256;      // slots of the hash table (about half full at most) that a value tries
constexpr int kWindowBuckets = 4096;
constexpr int kWindowBucketMost = 32;  // values in one bucket; where there are more the bitonic sort takes over
// LDS: a hash table of at least twice the values (as many, of the most), then in its place the different values,
// buckets, followers and marks
__host__ __device__ constexpr int window_distinct(int capacity) { return capacity < kWindowDistinct ? capacity : kWindowDistinct; }
__host__ __device__ constexpr int window_slots(int capacity) { return capacity < kWindowMost ? 2 * capacity : kWindowMost; }
inline size_t window_lds(int capacity) {
  const size_t walk = (size_t)window_distinct(capacity) * (sizeof(float) + sizeof(uint16_t) + sizeof(uint8_t)) +
                      kWindowBuckets * sizeof(int32_t);
  return std::max(walk, (size_t)window_slots(capacity) * sizeof(float));
}
// status of a window walked on the device (meta[r][2])
constexpr int kWindowOk = 0, kWindowNone = 1, kWindowOverflow = 2, kWindowNoStart = 3,
              kWindowNoBound = 4, kWindowKeptOverflow = 5;

// Most values of a window come several times (a stage costs the same for every number of pre-saved
// micro-batches that fits): the different ones of `n` through a hash table in the LDS of `v` and behind it, then in
// any order in `v`, by the whole workgroup.  Returns how many there are, -1 if they are more than `most` or one found
// no slot within kWindowProbes.  (Launches of a window of 32768 different values, which is given up: 550 us when they
// were counted behind the last one, now 118; 24000 119, now 95.  16384, which are walked, 156 either way; 32768 of
// 1000, 74.5 and 75.5.)
__device__ __forceinline__ int window_distinct_values(const float *__restrict__ in, int n, int slots, int most, float *v) {
  __shared__ int32_t found, inserted;
  uint32_t *table = reinterpret_cast<uint32_t *>(v);
  float held[kWindowHeld];
  const int tid = threadIdx.x, lane = tid & 63;
  constexpr uint32_t kEmpty = 0x7f800000u;  // (+inf: the values are finite)
  int bits = 7;
  while ((1 << bits) < slots && (1 << bits) < 2 * n) ++bits;
  const uint32_t mask = (1u << bits) - 1u;
  for (int i = tid; i <= (int)mask; i += kWindowThreads) table[i] = kEmpty;
  if (tid == 0) found = inserted = 0;
#pragma unroll
  for (int u = 0; u < kWindowHeld; ++u) {
    if (u * kWindowThreads >= n) break;
    held[u] = in[min(u * kWindowThreads + tid, n - 1)];
  }
  __syncthreads();
  uint32_t first = 0;  // bit u: value u is the first of its kind
  int counted = 0;
  bool lost = false;
#pragma unroll
  for (int u = 0; u < kWindowHeld; ++u) {
    if (u * kWindowThreads >= n) break;
    // given up when that is certain: the fuller the table, the longer the probing
    if (u == kWindowOwn + 1 || u == kWindowOwn + 8) {
      int own = __popc(first) - counted;
      counted += own;
      for (int step = 1; step < 64; step <<= 1) own += __shfl_xor(own, step);
      if (lane == 0) atomicAdd(&inserted, own);
    } else if (u > kWindowOwn + 1) {
      if (__any(lost || __hip_atomic_load(&inserted, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) > most)) break;
    }
    if (u * kWindowThreads + tid >= n) continue;
    const uint32_t key = __float_as_uint(held[u]);
    uint32_t at = key * 2654435761u >> (32 - bits);
    int probes = 0;
    for (; probes < kWindowProbes; ++probes, at = (at + 1) & mask) {
      const uint32_t there = atomicCAS(table + at, kEmpty, key);
      if (there == kEmpty) first |= 1u << u;
      if (there == kEmpty || there == key) break;
    }
    lost = lost || probes == kWindowProbes;
  }
  int end = __popc(first), base = 0;
  const int mine = end;
  for (int step = 1; step < 64; step <<= 1) {
    const int o = __shfl_up(end, step);
    if (lane >= step) end += o;
  }
  if (lane == 63) base = atomicAdd(&found, end);
  int at = __shfl(base, 63) + end - mine;
  if (__syncthreads_or(lost) || found > most) return -1;
#pragma unroll
  for (int u = 0; u < kWindowHeld; ++u) {
    if (u * kWindowThreads >= n) break;
    if (first >> u & 1u) v[at++] = held[u];
  }
  __syncthreads();
  return found;
}

// Sorts the `n` different values in `v` (LDS), by the whole workgroup.  They are finite and lie in a narrow range:
// equal-width buckets, whose number does not decrease with the value, and an insertion sort of what lands in each;
// where a bucket holds too many, or no width can be given, a bitonic sort.
__device__ __forceinline__ void window_sort(float *v, int n, int32_t *buckets) {
  __shared__ float low_of_wave[kWindowThreads / 64], high_of_wave[kWindowThreads / 64];
  __shared__ int32_t wave_total[kWindowThreads / 64];
  float held[kWindowOwn];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  float low = INFINITY, high = -INFINITY;
#pragma unroll
  for (int u = 0; u < kWindowOwn; ++u) {
    if (u * kWindowThreads >= n) break;
    held[u] = v[min(u * kWindowThreads + tid, n - 1)];
    low = fminf(low, held[u]);
    high = fmaxf(high, held[u]);
  }
  for (int step = 1; step < 64; step <<= 1) {
    low = fminf(low, __shfl_xor(low, step));
    high = fmaxf(high, __shfl_xor(high, step));
  }
  if (lane == 0) {
    low_of_wave[wave] = low;
    high_of_wave[wave] = high;
  }
  constexpr int kOwn = kWindowBuckets / kWindowThreads;  // buckets of a thread
#pragma unroll
  for (int u = 0; u < kOwn; ++u) buckets[u * kWindowThreads + tid] = 0;
  __syncthreads();
  for (int w = 0; w < kWindowThreads / 64; ++w) {
    low = fminf(low, low_of_wave[w]);
    high = fmaxf(high, high_of_wave[w]);
  }
  const float span = high - low, scale = (float)(kWindowBuckets - 1) / span;
  const bool fits = span < INFINITY && scale < INFINITY;
  auto bucket_of = [&](float value) { return min((int)((value - low) * scale), kWindowBuckets - 1); };
  bool crowded = !fits;
  int place[kWindowOwn];  // number inside the bucket
#pragma unroll
  for (int u = 0; u < kWindowOwn; ++u) {
    if (!fits || u * kWindowThreads >= n) break;
    if (u * kWindowThreads + tid >= n) continue;
    place[u] = atomicAdd(buckets + bucket_of(held[u]), 1);
    crowded = crowded || place[u] >= kWindowBucketMost;
  }
  if (__syncthreads_or(crowded)) {
    // One compare-exchange per thread and step, thread x holds the pair (i, i + j) with i = 2 j (x / j) + x % j.
    // For j <= 32 the 64 pairs of a wavefront lie in its own 128 consecutive values, and so do those of the
    // following smaller j: those steps need no barrier between them (a wavefront's LDS accesses complete in order).
    int m = 128;
    while (m < n) m <<= 1;  // (at most the power of two that `v` holds)
    for (int i = n + tid; i < m; i += kWindowThreads) v[i] = INFINITY;
    __syncthreads();
    for (int k = 2; k <= m; k <<= 1) {
      for (int j = k >> 1; j > 0; j >>= 1) {
        for (int x = tid; x < m / 2; x += kWindowThreads) {
          const int i = 2 * (x & ~(j - 1)) + (x & (j - 1)), other = i + j;
          const float a = v[i], b = v[other];
          const bool ascending = (i & k) == 0;
          if ((a > b) == ascending) {
            v[i] = b;
            v[other] = a;
          }
        }
        if (j > 32) __syncthreads();
        else __builtin_amdgcn_wave_barrier();
      }
      if (k >= 64) __syncthreads();  // the next k starts with j = k: other wavefronts' values
    }
    __syncthreads();
    return;
  }
  // first value of every bucket: an exclusive scan, kOwn neighbouring buckets a thread
  int count[kOwn], own = 0;
#pragma unroll
  for (int u = 0; u < kOwn; ++u) own += count[u] = buckets[tid * kOwn + u];
  int end = own;
  for (int step = 1; step < 64; step <<= 1) {
    const int o = __shfl_up(end, step);
    if (lane >= step) end += o;
  }
  if (lane == 63) wave_total[wave] = end;
  __syncthreads();
  int begin = end - own;
  for (int w = 0; w < wave; ++w) begin += wave_total[w];
  int next = begin;
#pragma unroll
  for (int u = 0; u < kOwn; ++u) {
    buckets[tid * kOwn + u] = next;
    next += count[u];
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < kWindowOwn; ++u) {
    if (u * kWindowThreads >= n) break;
    if (u * kWindowThreads + tid < n) v[buckets[bucket_of(held[u])] + place[u]] = held[u];
  }
  __syncthreads();
  // a thread's buckets are neighbours, and in order: values move a few places
  for (int i = begin + 1; i < next; ++i) {
    const float x = v[i];
    int j = i;
    for (; j > begin && v[j - 1] > x; --j) v[j] = v[j - 1];
    v[j] = x;
  }
  __syncthreads();
}

// The walk over `n` > 0 ascending values from `first` on (mist_dp_window_begin's), by the whole workgroup.  A
// value is followed by the first one that is not within the gap above it (float32 differences do not decrease
// along the list), whatever was kept before it, and the walk is what the first kept value leads to: every
// value's follower, then twice, four times .. as far, and each time what the kept ones lead to is kept too.
__device__ __forceinline__ void window_walk(const float *v, int first, int n, double gap, uint16_t *follow, uint8_t *keep) {
  const int tid = threadIdx.x;
  int mine[kWindowOwn];
#pragma unroll
  for (int u = 0; u < kWindowOwn; ++u) {
    const int i = u * kWindowThreads + tid;
    if (u * kWindowThreads >= n) break;
    if (i >= n) continue;
    const float x = v[i];
    int step = 1, below = i;  // (the last one known to be within the gap)
    while (below + step < n && gap_below(v[below + step], x, gap)) {
      below += step;
      step *= 2;
    }
    for (; step > 0; step /= 2)
      if (below + step < n && gap_below(v[below + step], x, gap)) below += step;
    mine[u] = below + 1;
    follow[i] = (uint16_t)mine[u];
  }
  // the first one starts with nothing kept (mist_dp_filter_tmax)
  if (tid == 0) {
    while (first < n && gap_below(v[first], 0.0f, gap)) ++first;
    if (first < n) keep[first] = 1;
  }
  __syncthreads();
  for (bool more = true; more;) {
    more = false;
    int further[kWindowOwn];
#pragma unroll
    for (int u = 0; u < kWindowOwn; ++u) {
      if (u * kWindowThreads >= n) break;
      further[u] = n;
      if (u * kWindowThreads + tid >= n || mine[u] >= n) continue;
      if (keep[u * kWindowThreads + tid] != 0) keep[mine[u]] = 1;
      further[u] = follow[mine[u]];
      more = true;
    }
    more = __syncthreads_or(more) != 0;
#pragma unroll
    for (int u = 0; u < kWindowOwn; ++u) {
      if (u * kWindowThreads >= n) break;
      if (u * kWindowThreads + tid >= n || mine[u] >= n) continue;
      follow[u * kWindowThreads + tid] = (uint16_t)further[u];
      mine[u] = further[u];
    }
    __syncthreads();
  }
}

// (Bound: instruction issue of 16 wavefronts and the barriers between its passes; 14 us for one value, 24 for 2000
// different ones or 8000 of 400, 50 for 8000, 90 for 16000.  All values, repeated ones too, through a bitonic sort with
// a division per compare-exchange, and pieces between certain values walked by a thread each: GPT-7B 43 us, now 20;
// LLaMA-70B 117, now 64; GPT-22B 105, now 52.)
// One workgroup per request of a per-request candidate selection: sorts the request's different values
// (in LDS), walks them with the gap rule from the certain start below `start[r]` (the
// smallest feasible threshold; +inf = nothing feasible, the request is skipped), appends the kept
// thresholds to one list (kept_out, cursor in counts[0]) and lays out the first scan batch: up to
// `first_chunk` kept thresholds at or above start[r] (dp_first_batch_index) as DP instances,
// appended to inst_tmax / inst_row (cursor in counts[1 + 2 n_requests]; the caller pre-fills inst_row with
// -1, so that the live instances are the first workgroups of the DP launch and the empty slots
// its tail).
// meta[r][8] = (selected, above hi, status, kept, offset in kept_out, kept below start, instances,
// offset of the instances).
__global__ __launch_bounds__(kWindowThreads) void window_walk_kernel(
    const float *__restrict__ values, int capacity, int32_t *__restrict__ counts,
    const int32_t *__restrict__ rows, const float *__restrict__ lo,
    const float *__restrict__ start, double gap, int first_chunk, int first_lead,
    float *__restrict__ kept_out, int kept_capacity, int32_t *__restrict__ meta,
    float *__restrict__ inst_tmax, int32_t *__restrict__ inst_row) {
  extern __shared__ float win_lds[];
  float *v = win_lds;  // [most]
  const int most = window_distinct(capacity);
  int32_t *buckets = reinterpret_cast<int32_t *>(win_lds + most);             // [kWindowBuckets]
  uint16_t *follow = reinterpret_cast<uint16_t *>(buckets + kWindowBuckets);  // [most]
  uint8_t *keep = reinterpret_cast<uint8_t *>(follow + most);                 // [most]
  __shared__ int32_t wave_kept[kWindowThreads / 64], wave_below[kWindowThreads / 64];
  __shared__ int32_t walk_first, kept_base, kept_overflow, inst_base;
  const int r = blockIdx.x, n_requests = gridDim.x, tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6, n_waves = blockDim.x >> 6;
  const int n_sel = counts[1 + n_requests + r];
  const float start_r = start[r], lo_r = lo[r];
  int status = kWindowOk;
  if (!(start_r < INFINITY)) status = kWindowNone;
  else if (n_sel > capacity) status = kWindowOverflow;
  int n = 0;
  if (status == kWindowOk && n_sel > 0) {  // (the same for the whole workgroup)
    n = window_distinct_values(values + (int64_t)r * capacity, n_sel, window_slots(capacity), most, v);
    if (n < 0) {
      status = kWindowOverflow;
      n = 0;
    } else {
      window_sort(v, n, buckets);
    }
  }
  for (int i = tid; i < n; i += blockDim.x) keep[i] = 0;
  if (tid == 0) {
    walk_first = -1;
    kept_overflow = 0;
  }
  __syncthreads();
  // start of the walk (window_walk_start with a fetch that is not open below): the last
  // candidate <= start_r whose predecessor is at least the gap below, else the first candidate
  // if it lies above start_r and is certain itself
  // (an odd number of values a thread: neighbouring threads' lie in different LDS banks)
  const int per = ((n + (int)blockDim.x - 1) / (int)blockDim.x) | 1;
  const int i0 = min(tid * per, n), i1 = min(i0 + per, n);
  {
    int mine = -1;
    for (int i = i0; i < i1; ++i)
      if (v[i] <= start_r && !gap_below(v[i], i == 0 ? lo_r : v[i - 1], gap)) mine = i;
    if (mine >= 0) atomicMax(&walk_first, mine);
  }
  __syncthreads();
  int first = walk_first;
  if (status == kWindowOk && n > 0 && first < 0) {
    if (v[0] > start_r && !gap_below(v[0], lo_r, gap)) first = 0;
    else status = kWindowNoStart;
  }
  // the walk
  if (status == kWindowOk && n > 0) window_walk(v, first, n, gap, follow, keep);
  __syncthreads();
  // kept values per thread (consecutive elements), those below the start among them
  int mine = 0, below = 0;
  if (status == kWindowOk)
    for (int i = i0; i < i1; ++i) {
      mine += keep[i];
      below += keep[i] && v[i] < start_r;
    }
  int scan_kept = mine, scan_below = below;  // inclusive scans over the wavefront
  for (int step = 1; step < 64; step <<= 1) {
    const int a = __shfl_up(scan_kept, step), b = __shfl_up(scan_below, step);
    if (lane >= step) {
      scan_kept += a;
      scan_below += b;
    }
  }
  if (lane == 63) {
    wave_kept[wave] = scan_kept;
    wave_below[wave] = scan_below;
  }
  __syncthreads();
  int before = 0, n_kept = 0, pos = 0;
  for (int w = 0; w < n_waves; ++w) {
    if (w < wave) before += wave_kept[w];
    n_kept += wave_kept[w];
    pos += wave_below[w];
  }
  if (status == kWindowOk && pos >= n_kept) status = kWindowNoBound;  // nothing kept at or above the start
  const int n_inst = status == kWindowOk ? min(first_chunk, n_kept - pos) : 0;
  if (tid == 0) {
    kept_base = inst_base = 0;
    if (status == kWindowOk) {
      kept_base = atomicAdd(&counts[0], n_kept);
      if (kept_base + n_kept > kept_capacity) kept_overflow = 1;
      else inst_base = atomicAdd(&counts[1 + 2 * n_requests], n_inst);  // <= n_requests * first_chunk
    }
  }
  __syncthreads();
  if (status == kWindowOk && kept_overflow) status = kWindowKeptOverflow;
  if (status == kWindowOk) {
    int at = before + scan_kept - mine;  // kept values in front of this thread's elements
    for (int i = i0; i < i1; ++i) {
      if (!keep[i]) continue;
      kept_out[kept_base + at] = v[i];
      ++at;
    }
  }
  __syncthreads();  // (the workgroup's own writes to kept_out are visible to it behind the barrier)
  if (status == kWindowOk) {
    for (int k = tid; k < n_inst; k += blockDim.x) {
      inst_tmax[inst_base + k] =
          kept_out[kept_base + pos + dp_first_batch_index(k, n_kept - pos, first_chunk, first_lead)];
      inst_row[inst_base + k] = rows[r];
    }
  }
  if (tid == 0) {
    int32_t *out = meta + 8 * r;
    out[0] = n_sel;
    out[1] = counts[1 + r];
    out[2] = status;
    out[3] = status == kWindowOk ? n_kept : 0;
    out[4] = kept_base;
    out[5] = pos;
    out[6] = status == kWindowOk ? n_inst : 0;
    out[7] = inst_base;
  }
}

// ------------------------------------------------------------------------------------------
// DP kernels.  The stage index s is the sequential axis: one launch per s.  Within a launch
// every (threshold, start layer k, devices d) state is one thread; workgroups are single
// wavefronts so that even a handful of thresholds spreads over many CUs.  F(s-1) / F(s) and
// the running stage maxima ping-pong between two planes per threshold in a global scratch slab
// (L2 resident: 4 * (L+1) * (D+1) floats per threshold).
// ------------------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void dp_init_kernel(const MistDpShape shape, int n_tmax,
                                                      float *__restrict__ scratch,
                                                      int32_t *__restrict__ ranges,
                                                      int32_t *__restrict__ best_s,
                                                      float *__restrict__ best_sum,
                                                      float *__restrict__ stage_max) {
  const int W = shape.num_devices + 1;
  const int plane = (shape.num_layers + 1) * W;
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < (int64_t)n_tmax * W) {
    // Reachable start layers [first, last] per instance and device column, three buffers used
    // in rotation by the steps.  F(0) is reachable at (k = L, d = 0) only.
    const int64_t stride = (int64_t)n_tmax * W * 2;
    const bool origin = i % W == 0;
    ranges[2 * i] = origin ? shape.num_layers : shape.num_layers + 1;
    ranges[2 * i + 1] = origin ? shape.num_layers : -1;
    for (int b = 1; b < 3; ++b) {
      ranges[b * stride + 2 * i] = shape.num_layers + 1;
      ranges[b * stride + 2 * i + 1] = -1;
    }
  }
  if (i >= (int64_t)n_tmax * plane) return;
  const int t = (int)(i / plane), e = (int)(i % plane);
  float *state = scratch + (int64_t)t * 4 * plane;
  // plane 0 holds F(0, ., .): 0 at (k = L, d = 0), +inf elsewhere; maxima start at 0.
  state[e] = e == shape.num_layers * W ? 0.0f : INFINITY;
  state[2 * plane + e] = 0.0f;
  if (e == 0) {
    best_s[t] = -1;
    best_sum[t] = INFINITY;
    stage_max[t] = 0.0f;
  }
}

// Where the ckpt row of (variant, mesh q, pre-saved micro-batches p, layers k..i) starts and which
// table holds it.
struct DpRowRef {
  int v;
  int64_t at;
};
__device__ __forceinline__ DpRowRef dp_row_ref(const MistDpShape &shape, const int64_t (&off)[4],
                                               int p, int k, int q, int i) {
  const int L = shape.num_layers, P1 = shape.p_dim, C = L + 1;
  const int l = i - k + 1;
  DpRowRef r;
  if (k == 0 && i == L - 1) { r.v = 3; r.at = (int64_t)q * C; }
  else if (k == 0) { r.v = 1; r.at = (((int64_t)q * P1 + p) * L + (l - 1)) * C; }
  else if (i == L - 1) { r.v = 2; r.at = ((int64_t)q * L + (l - 1)) * C; }
  else { r.v = 0; r.at = (((int64_t)q * P1 + p) * L + (l - 1)) * C; }
  r.at += off[r.v];
  return r;
}
__device__ __forceinline__ const float *dp_table(const MistDpCosts &tabs, int v, bool running_min) {
  if (running_min)
    return v == 0 ? tabs.pmin : v == 1 ? tabs.pmin_pre : v == 2 ? tabs.pmin_post : tabs.pmin_nopp;
  return v == 0 ? tabs.costs : v == 1 ? tabs.costs_pre : v == 2 ? tabs.costs_post : tabs.costs_nopp;
}
// ckpt candidates j_begin..j_end of a stage k..i: 0..L-i (inter_tuning.py:315), or 0..l / only l
// (inter_tuning_uniform_device.py:400-404)
__device__ __forceinline__ int dp_j_last(const MistDpShape &shape, int k, int i) {
  return shape.ckpt_rule == MIST_DP_CKPT_TAIL ? shape.num_layers - i : i - k + 1;
}
// What dp_row_min reads of a g.  By value: a table that is picked through a reference to the kernel's arguments
// puts those into scratch, 176 bytes a lane of dp_free_kernel and 136 of dp_step_kernel, which then read them there for
// every row.  (1024 instances of 32 stages: 128 layers by dp_step_kernel 2990 us, now 2645; 110 by dp_free_kernel
// 449 -> 372, 91 250 -> 217.)
struct DpRows {
  const float *inner, *pre, *post, *nopp;  // costs where only the last ckpt candidate counts, else running minima
  const int32_t *planes;                   // per mesh (MistDpCosts.planes), NULL = all
  int L, P1, ckpt_rule;
};
__device__ __forceinline__ DpRows dp_rows(const MistDpShape &shape, const MistDpCosts &tabs, int64_t g) {
  DpRows r;
  if (shape.ckpt_rule == MIST_DP_CKPT_ALL) {
    r.inner = tabs.costs, r.pre = tabs.costs_pre, r.post = tabs.costs_post, r.nopp = tabs.costs_nopp;
  } else {
    r.inner = tabs.pmin, r.pre = tabs.pmin_pre, r.post = tabs.pmin_post, r.nopp = tabs.pmin_nopp;
  }
  r.inner += g * tabs.g_stride[0];
  r.pre += g * tabs.g_stride[1];
  r.post += g * tabs.g_stride[2];
  r.nopp += g * tabs.g_stride[3];
  r.planes = tabs.planes == nullptr ? nullptr : tabs.planes + g * tabs.planes_g_stride;
  r.L = shape.num_layers;
  r.P1 = shape.p_dim;
  r.ckpt_rule = shape.ckpt_rule;
  return r;
}
// The reference walks j = j_begin..j_end with "cost <= t_max and cost + prev < best".  "+ prev" is
// monotone, so the smallest reachable sum is (smallest admissible cost) + prev, and the smallest
// admissible cost is the row's running minimum if that is <= t_max (else nothing is admissible).
__device__ __forceinline__ float dp_row_min(const DpRows rows, int p, int k, int q, int i) {
  if (rows.planes != nullptr && p >= rows.planes[q]) return INFINITY;
  const int L = rows.L, l = i - k + 1;
  const bool first = k == 0, last = i == L - 1;
  const float *__restrict__ table = first ? (last ? rows.nopp : rows.pre) : last ? rows.post : rows.inner;
  const int64_t row = first && last ? q : (last ? (int64_t)q : (int64_t)q * rows.P1 + p) * L + (l - 1);
  return table[row * (L + 1) + (rows.ckpt_rule == MIST_DP_CKPT_TAIL ? L - i : l)];
}

// Re-laid row minima (mist_dp_stage_minima): per (g, p, mesh) a triangle over (k, i >= k), row k
// at dp_triangle_row(L, k), entry i - k.
__device__ __host__ __forceinline__ int dp_triangle(int L) { return L * (L + 1) / 2; }
__device__ __host__ __forceinline__ int dp_triangle_row(int L, int k) {
  return k * L - k * (k - 1) / 2;
}

// Running winner of one state's scan.  The reference visits (q, i) in ascending order and
// replaces on a strict "<".  A state reachable only through an unreachable successor cannot
// improve (inf + c is never < best); skipping it changes nothing.
constexpr int kDpNoCandidate = 0x7fffffff;
struct DpBest {
  float best = INFINITY, best_m = 0.0f, best_rmin = 0.0f;
  int order = kDpNoCandidate;  // q * L + i of the candidate that set `best`: its place in the visit
  int arg_i = -1, arg_q = -1, arg_j = -1;
  // mesh and end layer of the winner, once the scan is over
  __device__ __forceinline__ void resolve(int L) {
    arg_q = order == kDpNoCandidate ? -1 : order / L;
    arg_i = order == kDpNoCandidate ? -1 : order % L;
  }
};
// One candidate, without a branch: an unreachable successor (+inf) gives a target of +inf, which
// is never below the winner's.
template <bool kBottleneck>
__device__ __forceinline__ void dp_consider(DpBest &w, float t_max, int order, float prev,
                                            float rmin) {
  const float target = kBottleneck ? fmaxf(rmin, prev) : rmin + prev;
  const bool better = rmin <= t_max && target < w.best;
  w.best = better ? target : w.best;
  w.best_rmin = better ? rmin : w.best_rmin;
  w.order = better ? order : w.order;
}

// The winner's ckpt count and stage maximum: the first j attaining the sum is the entry the
// reference's strict "<" keeps.  Only the final winner matters, so the row is walked once.
template <bool kBottleneck>
__device__ __forceinline__ void dp_finish_winner(DpBest &w, const MistDpShape &shape,
                                                 const MistDpCosts &tabs, const int64_t (&off)[4],
                                                 float t_max, int p, int k, int d,
                                                 const float *f_prev, const float *m_prev) {
  if (w.arg_i < 0) return;
  const int W = shape.num_devices + 1;
  const int nm = shape.free_devices != 0 ? 0 : shape.mesh_n[w.arg_q] * shape.mesh_m[w.arg_q];
  const int from = (w.arg_i + 1) * W + (d - nm);
  if (kBottleneck) {
    // the maxima plane carries the SUM of the stage costs along the min-max path: a partition
    // that is admissible at the returned threshold, with its float32 sum accumulated in the
    // threshold DP's order
    w.best_m = w.best_rmin + m_prev[from];
    return;
  }
  const DpRowRef r = dp_row_ref(shape, off, p, k, w.arg_q, w.arg_i);
  const float *__restrict__ row = dp_table(tabs, r.v, false) + r.at;
  const float prev = f_prev[from];
  const int j_begin = shape.ckpt_rule == MIST_DP_CKPT_ALL ? w.arg_i - k + 1 : 0;
  const int j_end = dp_j_last(shape, k, w.arg_i);
  // kDpBatch entries are read together and tested in order
  for (int j0 = j_begin; j0 <= j_end; j0 += kDpBatch) {
    float stage_cost[kDpBatch];
#pragma unroll
    for (int u = 0; u < kDpBatch; ++u) stage_cost[u] = j0 + u <= j_end ? row[j0 + u] : INFINITY;
#pragma unroll
    for (int u = 0; u < kDpBatch; ++u) {
      if (j0 + u <= j_end && stage_cost[u] <= t_max && stage_cost[u] + prev == w.best) {
        w.arg_j = j0 + u;
        w.best_m = fmaxf(m_prev[from], stage_cost[u]);
        return;
      }
    }
  }
}

// Upper bound of the smallest feasible threshold, for the bottleneck DP of one instance: the
// largest stage cost of any partition bounds the min-max optimum from above, and a stage that
// costs more than such a bound is on no min-max partition, so the bottleneck DP may treat it as
// inadmissible (same value, same first-wins path: every candidate it drops has a target above
// the optimum).  The bound is the min-max optimum over the partitions that put every stage on
// the same mesh q (n m s = D stages, or any s <= max_stages when stages do not consume devices)
// with the layers split freely: a recurrence over (stage count, start layer) alone,
//   B(s, k) = min over i >= k of max(cost(s, k, i, q), B(s - 1, i + 1)),
// one wavefront per mesh, its two rows of B in `rows` (LDS, 2 (L + 1) of its `n_rows` floats per
// wavefront), kDpBoundLoads costs of a lane in flight (one at a time: 34 us of a bottleneck instance
// of the 7B plan, 364 of 70B on 32x8; 16 at a time about half of it).  Called by the whole workgroup; `slot` is one int of LDS.  +inf when no such
// partition is feasible (or L > 128: a lane holds two start layers; or `rows` is too small).
constexpr int kDpBoundLoads = 16;
__device__ __forceinline__ float dp_uniform_mesh_bound(const MistDpShape &shape,
                                                       const float *__restrict__ relaid,
                                                       float *rows, int n_rows, int32_t *slot) {
  const int L = shape.num_layers, D = shape.num_devices, Q = shape.num_mesh;
  const int tri = dp_triangle(L);
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n_waves = (blockDim.x + 63) >> 6;
  if (threadIdx.x == 0) *slot = __float_as_int(INFINITY);
  __syncthreads();
  if (L <= 128 && n_waves * 2 * (L + 1) <= n_rows) {
    float *prev = rows + wave * 2 * (L + 1), *cur = prev + (L + 1);
    for (int q = wave; q < Q; q += n_waves) {
      int s_last = shape.max_stages;
      if (shape.free_devices == 0) {
        const int nm = shape.mesh_n[q] * shape.mesh_m[q];
        if (nm <= 0 || D % nm != 0 || D / nm > shape.max_stages) continue;
        s_last = D / nm;
      }
      if (s_last > L) continue;
      for (int k = lane; k <= L; k += 64) prev[k] = k == L ? 0.0f : INFINITY;
      __builtin_amdgcn_wave_barrier();
      float bound = INFINITY;
      for (int s = 1; s <= s_last; ++s) {
        const float *__restrict__ block = relaid + ((int64_t)(s - 1) * Q + q) * tri;
        for (int k = lane; k <= L; k += 64) {
          float best = INFINITY;
          if (k <= L - s) {
            const float *__restrict__ row = block + dp_triangle_row(L, k) - k;  // row[i]
            // the s - 1 stages behind this one take a layer each at least
            for (int i0 = k; i0 <= L - s; i0 += kDpBoundLoads) {
              float cost[kDpBoundLoads];
#pragma unroll
              for (int u = 0; u < kDpBoundLoads; ++u) cost[u] = row[min(i0 + u, L - s)];
#pragma unroll
              for (int u = 0; u < kDpBoundLoads; ++u)
                best = fminf(best, fmaxf(cost[u], prev[min(i0 + u, L - s) + 1]));
            }
          }
          cur[k] = best;
        }
        __builtin_amdgcn_wave_barrier();
        if (shape.free_devices != 0 || s == s_last) bound = fminf(bound, cur[0]);
        float *swap = prev;
        prev = cur;
        cur = swap;
        __builtin_amdgcn_wave_barrier();
      }
      // stage costs are not negative, and non-negative floats order like their bit patterns
      if (lane == 0 && bound >= 0.0f && bound < INFINITY) atomicMin(slot, __float_as_int(bound));
    }
  }
  __syncthreads();
  return __int_as_float(*slot);
}

// Scan of one state (start layer k, devices d) by one lane (member 0 of 1) or by its share of a
// team: meshes q and end layers i in the reachable range of the successor column.
// `row_min(q, i)` returns dp_row_min of the stage k..i on mesh q; `narrow(q, i_first, i_last)`
// may shrink the range of end layers to one that still holds every i with row_min <= t_max.
struct DpKeepRange {
  __device__ __forceinline__ void operator()(int, int &, int &) const {}
};
template <bool kBottleneck, int kDpTeam, typename RowMin, typename Narrow = DpKeepRange>
__device__ __forceinline__ void dp_scan_state(DpBest &w, const MistDpShape &shape, float t_max,
                                              int k, int d, int member, const float *f_prev,
                                              const int32_t *range_prev, RowMin row_min,
                                              Narrow narrow = Narrow()) {
  const int L = shape.num_layers, W = shape.num_devices + 1;
  const bool free_devices = shape.free_devices != 0;
  for (int q = 0; q < shape.num_mesh; ++q) {
    const int nm = free_devices ? 0 : shape.mesh_n[q] * shape.mesh_m[q];
    if (nm > d) continue;
    // reachable start layers i + 1 of the remaining stages on d - nm devices
    const int32_t *reach = range_prev + 2 * (d - nm);
    int i_first = max(k, reach[0] - 1), i_last = min(L - 1, reach[1] - 1);
    narrow(q, i_first, i_last);
    if constexpr (kDpTeam == 1) {
      // One lane per state: the scan is a chain of reads.  kDpBatch end layers at a time, first
      // all their successor values, then the row minima of the reachable ones, so that the reads
      // of a batch are in flight together; the comparisons keep the order.
      for (int i0 = i_first; i0 <= i_last; i0 += kDpBatch) {
        float prev[kDpBatch], rmin[kDpBatch];
#pragma unroll
        for (int u = 0; u < kDpBatch; ++u)
          prev[u] = i0 + u <= i_last ? f_prev[(i0 + u + 1) * W + (d - nm)] : INFINITY;
#pragma unroll
        for (int u = 0; u < kDpBatch; ++u)
          rmin[u] = prev[u] == INFINITY ? INFINITY : row_min(q, i0 + u);
#pragma unroll
        for (int u = 0; u < kDpBatch; ++u)
          dp_consider<kBottleneck>(w, t_max, q * L + i0 + u, prev[u], rmin[u]);
      }
    } else {
      for (int i = i_first + member; i <= i_last; i += kDpTeam) {
        const float prev = f_prev[(i + 1) * W + (d - nm)];
        if (prev == INFINITY) continue;
        dp_consider<kBottleneck>(w, t_max, q * L + i, prev, row_min(q, i));
      }
    }
  }
}

template <bool kBottleneck, int kDpTeam>
__global__ __launch_bounds__(kDpThreads) void dp_step_kernel(
    const MistDpShape shape, const MistDpCosts tabs, const float *__restrict__ tmax_list,
    const int32_t *__restrict__ g_list, int s, float *__restrict__ scratch,
    int32_t *__restrict__ ranges, int32_t *__restrict__ best_s_out,
    float *__restrict__ best_sum_out, float *__restrict__ stage_max_out,
    int32_t *__restrict__ argmin) {
  const int L = shape.num_layers, D = shape.num_devices;
  const int W = D + 1;            // row pitch of a state plane
  const int plane = (L + 1) * W;  // states per s
  // kDpTeam consecutive lanes share one state and split its end layers between them.  The scan
  // of a state is a chain of dependent L2 reads: in a small batch its latency, not the
  // arithmetic, sets the time of a launch (team of 8); a batch that fills the GPU anyway runs
  // one lane per state, which prunes better.
  const int member = threadIdx.x % kDpTeam;
  const int e_raw = (blockIdx.x * kDpThreads + threadIdx.x) / kDpTeam;
  const bool real = e_raw < plane;  // the last team of a plane may be a dummy (kept for shuffles)
  if constexpr (kDpTeam == 1) {
    if (!real) return;
  }
  const int e = real ? e_raw : plane - 1;
  const int t = blockIdx.y;
  float *state = scratch + (int64_t)t * 4 * plane;
  const int cur = s & 1, prv = cur ^ 1;
  const float *__restrict__ f_prev = state + prv * plane;
  const float *__restrict__ m_prev = state + (2 + prv) * plane;
  float *__restrict__ f_cur = state + cur * plane;
  float *__restrict__ m_cur = state + (2 + cur) * plane;
  // bottleneck mode has no threshold; the largest finite value skips the +inf entries, which
  // improve no state (inf is never < best)
  const float t_max = kBottleneck ? kDpNoThreshold : tmax_list[t];
  const int64_t g = g_list[t];
  if (g < 0) return;  // an empty slot of the batch (the whole workgroup: blockIdx.y is the instance)
  const int64_t off[4] = {g * tabs.g_stride[0], g * tabs.g_stride[1], g * tabs.g_stride[2],
                          g * tabs.g_stride[3]};
  const DpRows rows_of_g = dp_rows(shape, tabs, g);
  const int k = e / W, d = e % W;
  const int p = s - 1;
  // Most states are unreachable.  Every step records, per instance and device column, the first
  // and last start layer it reached (buffer s % 3); the next step scans only that range.  The
  // buffer after that one is reset here: its last readers ran in the step before this one.
  const int64_t range_stride = (int64_t)gridDim.y * W * 2;
  const int32_t *range_prev = ranges + ((s + 2) % 3) * range_stride + (int64_t)t * W * 2;
  int32_t *range_cur = ranges + (s % 3) * range_stride + (int64_t)t * W * 2;
  int32_t *range_next = ranges + ((s + 1) % 3) * range_stride + (int64_t)t * W * 2;

  // the row minima of this stage count in (mesh, k, i) order, if the caller prepared them
  const int tri = dp_triangle(L);
  const float *__restrict__ relaid =
      tabs.stage_min == nullptr
          ? nullptr
          : tabs.stage_min + g * tabs.stage_min_g_stride + (int64_t)p * shape.num_mesh * tri +
                dp_triangle_row(L, k) - k;
  DpBest w;
  const bool live = k <= L - s && (d >= 1 || shape.free_devices != 0);
  if (live) {
    dp_scan_state<kBottleneck, kDpTeam>(
        w, shape, t_max, k, d, member, f_prev, range_prev,
        [&](int q, int i) {
          return relaid != nullptr ? relaid[q * tri + i] : dp_row_min(rows_of_g, p, k, q, i);
        });
    if constexpr (kDpTeam == 1) {
      w.resolve(L);
      dp_finish_winner<kBottleneck>(w, shape, tabs, off, t_max, p, k, d, f_prev, m_prev);
    }
  }
  // Team reduction: the winner is the first candidate that attains the minimum, i.e. the
  // lexicographic minimum of (target, q, i).  Each lane holds that minimum over its own
  // candidates.
  if constexpr (kDpTeam > 1) {
#pragma unroll
    for (int step = 1; step < kDpTeam; step <<= 1) {
      const float o_best = __shfl_xor(w.best, step);
      const float o_rmin = __shfl_xor(w.best_rmin, step);
      const int o_order = __shfl_xor(w.order, step);
      const bool take = o_best < w.best || (o_best == w.best && o_order < w.order);
      w.best = take ? o_best : w.best;
      w.best_rmin = take ? o_rmin : w.best_rmin;
      w.order = take ? o_order : w.order;
    }
    w.resolve(L);
    if (!real || member != 0) return;
    if (live) dp_finish_winner<kBottleneck>(w, shape, tabs, off, t_max, p, k, d, f_prev, m_prev);
  }
  f_cur[e] = w.best;
  m_cur[e] = w.best_m;
  if (w.best < INFINITY) {
    atomicMin(&range_cur[2 * d], k);
    atomicMax(&range_cur[2 * d + 1], k);
  }
  if (k == 0) {
    range_next[2 * d] = L + 1;
    range_next[2 * d + 1] = -1;
  }
  if (argmin != nullptr && w.arg_i >= 0) {
    int32_t *a = argmin + (((int64_t)t * (shape.max_stages + 1) + s) * plane + e) * 4;
    a[0] = w.arg_i;
    a[1] = shape.mesh_n[w.arg_q];
    a[2] = shape.mesh_m[w.arg_q];
    a[3] = w.arg_j;
  }
  // The state (k = 0, d = D) is the answer of this stage count; first s wins ties
  // (inter_tuning.py:335-340).  The same thread handles it in every launch.
  if (k == 0 && d == D && w.best < best_sum_out[t]) {
    best_sum_out[t] = w.best;
    best_s_out[t] = s;
    stage_max_out[t] = w.best_m;
  }
}

// ------------------------------------------------------------------------------------------
// The same recurrence with the whole instance in one workgroup: the four state planes and the
// reachable ranges live in LDS, the stage counts are a loop with a barrier between them, and one
// launch replaces init + max_stages step launches.  Used whenever the planes fit (16 bytes per
// state); the arithmetic per state is the code above.
// ------------------------------------------------------------------------------------------
template <bool kBottleneck>
__global__ __launch_bounds__(kDpFusedThreads) void dp_fused_kernel(
    const MistDpShape shape, const MistDpCosts tabs, const float *__restrict__ tmax_list,
    const int32_t *__restrict__ g_list, int32_t *__restrict__ best_s_out,
    float *__restrict__ best_sum_out, float *__restrict__ stage_max_out,
    int32_t *__restrict__ argmin) {
  extern __shared__ float dp_lds[];
  const int L = shape.num_layers, D = shape.num_devices;
  const int W = D + 1, plane = (L + 1) * W;
  float *f_plane = dp_lds;              // [2][plane]
  float *m_plane = dp_lds + 2 * plane;  // [2][plane]
  int32_t *range = reinterpret_cast<int32_t *>(dp_lds + 4 * plane);  // [3][W][2]
  // row minima of the current stage count: per mesh a triangle (k, i >= k)
  float *stage_min = dp_lds + 4 * plane + 6 * W;
  const int tri = dp_triangle(L), n_stage = shape.num_mesh * tri;
  // first and last end layer of a stage on mesh q from layer k whose row minimum is <= t_max
  int32_t *admissible = reinterpret_cast<int32_t *>(stage_min + n_stage);  // [Q][L][2]
  const int t = blockIdx.x;
  const int64_t g = g_list[t];
  if (g < 0) {  // an empty slot of the batch
    if (threadIdx.x == 0) {
      best_s_out[t] = -1;
      best_sum_out[t] = INFINITY;
      stage_max_out[t] = 0.0f;
    }
    return;
  }
  const int64_t off[4] = {g * tabs.g_stride[0], g * tabs.g_stride[1], g * tabs.g_stride[2],
                          g * tabs.g_stride[3]};
  const float *__restrict__ relaid = tabs.stage_min + g * tabs.stage_min_g_stride;
  // the bottleneck DP has no threshold of its own: an upper bound of its answer serves as one
  // (not with back-pointers: then every state gets the entry the unbounded recurrence gives it)
  const float t_max = !kBottleneck       ? tmax_list[t]
                      : argmin != nullptr
                          ? kDpNoThreshold
                          : fminf(kDpNoThreshold,
                                  dp_uniform_mesh_bound(shape, relaid, stage_min, n_stage, admissible));
  // F(0, ., .): 0 at (k = L, d = 0), +inf elsewhere; maxima start at 0; only that state is
  // reachable.
  for (int e = threadIdx.x; e < plane; e += blockDim.x) {
    f_plane[e] = e == L * W ? 0.0f : INFINITY;
    m_plane[e] = 0.0f;
  }
  for (int col = threadIdx.x; col < W; col += blockDim.x) {
    range[2 * col] = col == 0 ? L : L + 1;
    range[2 * col + 1] = col == 0 ? L : -1;
    for (int b = 1; b < 3; ++b) {
      range[(b * W + col) * 2] = L + 1;
      range[(b * W + col) * 2 + 1] = -1;
    }
  }
  // a thread's states are blockDim.x apart: (k, d) advance by fixed steps
  const int k_first = threadIdx.x / W, d_first = threadIdx.x % W;
  const int k_step = blockDim.x / W, d_step = blockDim.x % W;
  // the answer state (k = 0, d = D) belongs to the same thread in every step
  float answer_sum = INFINITY, answer_max = 0.0f;
  int answer_s = -1;
  __syncthreads();
  for (int s = 1; s <= shape.max_stages; ++s) {
    const int cur = s & 1, prv = cur ^ 1, p = s - 1;
    const float *f_prev = f_plane + prv * plane, *m_prev = m_plane + prv * plane;
    float *f_cur = f_plane + cur * plane, *m_cur = m_plane + cur * plane;
    const int32_t *range_prev = range + ((s + 2) % 3) * W * 2;
    int32_t *range_cur = range + (s % 3) * W * 2;
    int32_t *range_next = range + ((s + 1) % 3) * W * 2;
    // Every state with start layer k reads the same row minima: copy the block of this stage
    // count (contiguous in the re-laid table) once per workgroup, kDpStageBatch loads per lane
    // in flight, so that the scans below touch LDS only.  (The previous step's scans ended at
    // the barrier that closed it.)
    const float *__restrict__ block = relaid + (int64_t)p * n_stage;
    for (int x0 = threadIdx.x; x0 < n_stage; x0 += kDpStageBatch * blockDim.x) {
      float value[kDpStageBatch];
#pragma unroll
      for (int u = 0; u < kDpStageBatch; ++u) {
        const int x = x0 + u * blockDim.x;
        if (x < n_stage) value[u] = block[x];
      }
#pragma unroll
      for (int u = 0; u < kDpStageBatch; ++u) {
        const int x = x0 + u * blockDim.x;
        if (x < n_stage) stage_min[x] = value[u];
      }
    }
    __syncthreads();
    // Near the smallest feasible threshold only short stages are admissible: the end layers
    // outside [first, last] fail "cost <= t_max" for every device count, so the scans of all
    // states with this start layer skip them (what lies inside is still tested one by one).
    {
      for (int x = threadIdx.x; x < shape.num_mesh * L; x += blockDim.x) {
        const int q = x / L, k0 = x % L;
        const float *row = stage_min + q * tri + dp_triangle_row(L, k0) - k0;
        int first = L, last = -1;
        for (int i = k0; i < L; ++i) {
          if (row[i] <= t_max) {
            first = min(first, i);
            last = i;
          }
        }
        admissible[2 * x] = first;
        admissible[2 * x + 1] = last;
      }
      __syncthreads();
    }
    int k = k_first, d = d_first;
    for (int e = threadIdx.x; e < plane; e += blockDim.x) {
      DpBest w;
      if (k <= L - s && (d >= 1 || shape.free_devices != 0)) {
        const float *mine = stage_min + dp_triangle_row(L, k) - k;
        dp_scan_state<kBottleneck, 1>(w, shape, t_max, k, d, 0, f_prev, range_prev,
                                      [&](int q, int i) { return mine[q * tri + i]; },
                                      [&](int q, int &i_first, int &i_last) {
                                        const int32_t *a = admissible + 2 * (q * L + k);
                                        i_first = max(i_first, a[0]);
                                        i_last = min(i_last, a[1]);
                                      });
        w.resolve(L);
        dp_finish_winner<kBottleneck>(w, shape, tabs, off, t_max, p, k, d, f_prev, m_prev);
      }
      f_cur[e] = w.best;
      m_cur[e] = w.best_m;
      if (w.best < INFINITY) {
        atomicMin(&range_cur[2 * d], k);
        atomicMax(&range_cur[2 * d + 1], k);
      }
      if (k == 0) {
        range_next[2 * d] = L + 1;
        range_next[2 * d + 1] = -1;
      }
      if (argmin != nullptr && w.arg_i >= 0) {
        int32_t *a = argmin + (((int64_t)t * (shape.max_stages + 1) + s) * plane + e) * 4;
        a[0] = w.arg_i;
        a[1] = shape.mesh_n[w.arg_q];
        a[2] = shape.mesh_m[w.arg_q];
        a[3] = w.arg_j;
      }
      if (e == D && w.best < answer_sum) {  // first s wins ties (inter_tuning.py:335-340)
        answer_sum = w.best;
        answer_s = s;
        answer_max = w.best_m;
      }
      k += k_step;  // state e + blockDim.x
      d += d_step;
      if (d >= W) {
        d -= W;
        ++k;
      }
    }
    __syncthreads();
  }
  if ((int)threadIdx.x == D % (int)blockDim.x) {
    best_s_out[t] = answer_s;
    best_sum_out[t] = answer_sum;
    stage_max_out[t] = answer_max;
  }
}

// ------------------------------------------------------------------------------------------
// The recurrence for shapes whose four state planes do not fit the LDS of a compute unit (80
// layers x 256 devices: 333 KB).  One workgroup per instance keeps ONE plane in LDS, F(s - 1),
// the only one the scans read at random; F(s) and the maxima planes go through the instance's
// global scratch (one coalesced copy of F(s) into LDS per stage count), the row minima are read
// from the re-laid table.  A wavefront owns (start layer k, 64 consecutive device counts d): the
// loop over (mesh, end layer) is the same for all its lanes, so the row minimum is one uniform
// read, the test against t_max a scalar branch that skips the step for the whole wavefront, and
// the LDS reads of F(s - 1) are 64 consecutive floats.  Per state the candidates are still
// visited in the reference's (mesh, end layer) order with a strict "<": same winner, same ties.
// ------------------------------------------------------------------------------------------
constexpr int kDpPlaneThreads = 1024;
constexpr int kDpPlaneCols = 4;    // device counts per lane: d = 1 + lane + 64 j, so D <= 256
constexpr int kDpPlaneLoads = 20;  // row minima a lane fetches per start layer: Q * L <= 1280
#ifndef MIST_DP_PLANE_MIN_INSTANCES
#define MIST_DP_PLANE_MIN_INSTANCES 16
#endif
// smaller batches stay on the per-stage-count launches, which spread one instance over the GPU
constexpr int kDpPlaneMinInstances = MIST_DP_PLANE_MIN_INSTANCES;

template <bool kBottleneck>
__global__ __launch_bounds__(kDpPlaneThreads) void dp_plane_kernel(
    const MistDpShape shape, const MistDpCosts tabs, const float *__restrict__ tmax_list,
    const int32_t *__restrict__ g_list, float *__restrict__ scratch,
    int32_t *__restrict__ best_s_out, float *__restrict__ best_sum_out,
    float *__restrict__ stage_max_out, int32_t *__restrict__ argmin) {
  extern __shared__ float dp_lds[];
  const int L = shape.num_layers, D = shape.num_devices, Q = shape.num_mesh;
  const int W = D + 1, plane = (L + 1) * W;
  float *f_lds = dp_lds;                                        // F(s - 1)
  int32_t *range = reinterpret_cast<int32_t *>(dp_lds + plane);  // [3][W][2] reachable rows per column
  int32_t *reach_q = range + 6 * W;                              // [Q][2] the same per mesh, all columns
  float *wave_rows = reinterpret_cast<float *>(reach_q + 2 * Q);  // [n_waves][Q][L] row minima of a task
  const int t = blockIdx.x;
  const int64_t g = g_list[t];
  if (g < 0) {  // an empty slot of the batch
    if (threadIdx.x == 0) {
      best_s_out[t] = -1;
      best_sum_out[t] = INFINITY;
      stage_max_out[t] = 0.0f;
    }
    return;
  }
  const int64_t off[4] = {g * tabs.g_stride[0], g * tabs.g_stride[1], g * tabs.g_stride[2],
                          g * tabs.g_stride[3]};
  const int tri = dp_triangle(L);
  const float *__restrict__ relaid = tabs.stage_min + g * tabs.stage_min_g_stride;
  // the bottleneck DP has no threshold of its own: an upper bound of its answer serves as one
  // (reach_q is free until the first stage count)
  // (not with back-pointers: then every state gets the entry the unbounded recurrence gives it)
  const float t_max = !kBottleneck       ? tmax_list[t]
                      : argmin != nullptr
                          ? kDpNoThreshold
                          : fminf(kDpNoThreshold,
                                  dp_uniform_mesh_bound(shape, relaid, wave_rows,
                                                        (int)(blockDim.x >> 6) * Q * L, reach_q));
  float *state = scratch + (int64_t)t * 4 * plane;
  float *__restrict__ f_cur = state;  // F(s) on its way into LDS
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n_waves = blockDim.x >> 6;
  float *my_rows = wave_rows + wave * Q * L;
  int d_of[kDpPlaneCols];
  bool col_ok[kDpPlaneCols];
#pragma unroll
  for (int j = 0; j < kDpPlaneCols; ++j) {
    d_of[j] = 1 + lane + 64 * j;
    col_ok[j] = d_of[j] <= D;
  }

  for (int e = threadIdx.x; e < plane; e += blockDim.x) f_lds[e] = e == L * W ? 0.0f : INFINITY;
  for (int col = threadIdx.x; col < W; col += blockDim.x) {
    range[2 * col] = col == 0 ? L : L + 1;
    range[2 * col + 1] = col == 0 ? L : -1;
    for (int b = 1; b < 3; ++b) {
      range[(b * W + col) * 2] = L + 1;
      range[(b * W + col) * 2 + 1] = -1;
    }
  }
  if (threadIdx.x == 0) state[2 * plane + L * W] = 0.0f;  // maximum of the empty partition
  float answer_sum = INFINITY, answer_max = 0.0f;
  int answer_s = -1;
  __syncthreads();
  for (int s = 1; s <= shape.max_stages; ++s) {
    const int cur = s & 1, prv = cur ^ 1, p = s - 1;
    const float *m_prev = state + (2 + prv) * plane;
    float *__restrict__ m_cur = state + (2 + cur) * plane;
    const int32_t *range_prev = range + ((s + 2) % 3) * W * 2;
    int32_t *range_cur = range + (s % 3) * W * 2;
    int32_t *range_next = range + ((s + 1) % 3) * W * 2;
    // reachable successor rows per mesh (over all columns): bounds of the uniform loop
    if (wave < Q) {
      const int q = wave;
      const int nm = shape.mesh_n[q] * shape.mesh_m[q];
      int first = L + 1, last = -1;
      for (int c = lane; c + nm <= D; c += 64) {  // successor column c = d - nm of some d <= D
        first = min(first, range_prev[2 * c]);
        last = max(last, range_prev[2 * c + 1]);
      }
#pragma unroll
      for (int step = 32; step >= 1; step >>= 1) {
        first = min(first, __shfl_xor(first, step));
        last = max(last, __shfl_xor(last, step));
      }
      if (lane == 0) {
        reach_q[2 * q] = first;
        reach_q[2 * q + 1] = last;
      }
    }
    for (int q = n_waves + wave; q < Q; q += n_waves) {  // (more meshes than wavefronts)
      if (lane == 0) {
        reach_q[2 * q] = 0;
        reach_q[2 * q + 1] = L;
      }
    }
    if (threadIdx.x == 0) {  // column 0 holds the origin only: unreachable from here on
      range_next[0] = L + 1;
      range_next[1] = -1;
    }
    __syncthreads();
    const float *__restrict__ block = relaid + (int64_t)p * Q * tri;
    // One task = one start layer k with all its device counts.  Tasks go to the wavefronts in
    // snake order (their cost falls with k).  A task's row minima, [Q][L - k] floats, are fetched
    // one task ahead into registers and laid into this wavefront's LDS buffer, so the loops
    // below have no global read in their dependence chain.
    const int n_tasks = L - s + 1;  // start layers 0 .. L - s
    auto task_k = [&](int round) {
      const int at = round * n_waves + ((round & 1) ? n_waves - 1 - wave : wave);
      return at < n_tasks ? at : -1;
    };
    float fetched[kDpPlaneLoads];
    auto fetch = [&](int k) {
      const int width = L - k;
#pragma unroll
      for (int u = 0; u < kDpPlaneLoads; ++u) {
        const int x = lane + 64 * u;
        if (k >= 0 && x < Q * width) {
          const int q = x / width, di = x - q * width;
          fetched[u] = block[q * tri + dp_triangle_row(L, k) + di];
        }
      }
    };
    fetch(task_k(0));
    for (int round = 0; task_k(round) >= 0; ++round) {
      const int k = task_k(round);
      const int width = L - k;
#pragma unroll
      for (int u = 0; u < kDpPlaneLoads; ++u) {
        const int x = lane + 64 * u;
        if (x < Q * width) my_rows[x] = fetched[u];
      }
      fetch(task_k(round + 1));
      __builtin_amdgcn_wave_barrier();
      // Running winner per column, lean: the value and (mesh << 8 | end layer) of the candidate
      // that set it; an unreachable successor (+inf) never compares below the winner, and the
      // admissibility of the candidate is the same for every lane (tested once, below).
      float best[kDpPlaneCols];
      int best_at[kDpPlaneCols];
#pragma unroll
      for (int j = 0; j < kDpPlaneCols; ++j) {
        best[j] = INFINITY;
        best_at[j] = -1;
      }
      for (int q = 0; q < Q; ++q) {
        const int nm = shape.mesh_n[q] * shape.mesh_m[q];
        const int i_first = max(k, reach_q[2 * q] - 1);
        const int i_last = min(L - 1, reach_q[2 * q + 1] - 1);
        bool lane_ok[kDpPlaneCols];
        const float *col[kDpPlaneCols];
#pragma unroll
        for (int j = 0; j < kDpPlaneCols; ++j) {
          lane_ok[j] = col_ok[j] && nm <= d_of[j];
          col[j] = f_lds + (lane_ok[j] ? d_of[j] - nm : 0);
        }
        const float *rm = my_rows + q * width - k;  // rm[i]
        // 64 end layers at a time: which of them are admissible at all (the same for every
        // lane), then only those, in ascending order
        for (int i0 = i_first; i0 <= i_last; i0 += 64) {
          const int i_mine = i0 + lane;
          const float r_mine = i_mine <= i_last ? rm[i_mine] : INFINITY;
          unsigned long long todo = __ballot(i_mine <= i_last && r_mine <= t_max);
          while (todo != 0) {
            const int bit = __ffsll(todo) - 1;
            todo &= todo - 1;
            const int i = i0 + bit;
            const float rmin = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(r_mine), bit));
            float prev[kDpPlaneCols];
#pragma unroll
            for (int j = 0; j < kDpPlaneCols; ++j)
              prev[j] = lane_ok[j] ? col[j][(i + 1) * W] : INFINITY;
            const int at = (q << 8) | i;
#pragma unroll
            for (int j = 0; j < kDpPlaneCols; ++j) {
              const float target = kBottleneck ? fmaxf(rmin, prev[j]) : rmin + prev[j];
              const bool better = target < best[j];
              best[j] = better ? target : best[j];
              best_at[j] = better ? at : best_at[j];
            }
          }
        }
      }
      __builtin_amdgcn_wave_barrier();
      DpBest w[kDpPlaneCols];
#pragma unroll
      for (int j = 0; j < kDpPlaneCols; ++j) {
        if (!col_ok[j]) continue;
        const int d = d_of[j];
        if (best_at[j] >= 0) {
          w[j].best = best[j];
          w[j].arg_q = best_at[j] >> 8;
          w[j].arg_i = best_at[j] & 255;
          w[j].best_rmin = my_rows[w[j].arg_q * width + (w[j].arg_i - k)];
        }
        dp_finish_winner<kBottleneck>(w[j], shape, tabs, off, t_max, p, k, d, f_lds, m_prev);
        const int e = k * W + d;
        f_cur[e] = w[j].best;
        m_cur[e] = w[j].best_m;
        if (w[j].best < INFINITY) {
          atomicMin(&range_cur[2 * d], k);
          atomicMax(&range_cur[2 * d + 1], k);
        }
        if (k == 0) {
          range_next[2 * d] = L + 1;
          range_next[2 * d + 1] = -1;
        }
        if (argmin != nullptr && w[j].arg_i >= 0) {
          int32_t *a = argmin + (((int64_t)t * (shape.max_stages + 1) + s) * plane + e) * 4;
          a[0] = w[j].arg_i;
          a[1] = shape.mesh_n[w[j].arg_q];
          a[2] = shape.mesh_m[w[j].arg_q];
          a[3] = w[j].arg_j;
        }
        // first s wins ties (inter_tuning.py:335-340); (k = 0, d = D) is wavefront 0's first
        // task in every step, the same lane's
        if (k == 0 && d == D && w[j].best < answer_sum) {
          answer_sum = w[j].best;
          answer_s = s;
          answer_max = w[j].best_m;
        }
      }
    }
    __syncthreads();  // every scan of F(s - 1) is done, F(s) is in the scratch plane
    for (int e = threadIdx.x; e < plane; e += blockDim.x) {
      const int k = e / W, d = e - k * W;
      f_lds[e] = (k <= L - s && d >= 1) ? f_cur[e] : INFINITY;
    }
    __syncthreads();
  }
  if (wave == 0 && lane == (D - 1) % 64) {
    best_s_out[t] = answer_s;
    best_sum_out[t] = answer_sum;
    stage_max_out[t] = answer_max;
  }
}

// ------------------------------------------------------------------------------------------
// The recurrence without per-state winners.  A caller of a scan batch wants three numbers per
// instance (stage count, sum, stage maximum), so only the winners on ONE path matter; the kernels
// above find the winner of every state, carry it through a plane of maxima and walk its ckpt row
// in the tables (a gather of up to 64 cache lines per load: about half of their time).  Here a
// state is only the minimum (add + min per candidate, any order), every plane F(s) is kept in the
// workgroup's history, and the answer's path is read back from it at the end: per stage the first
// (mesh, end layer) in the reference's order that attains the value, then the first ckpt count.
// One workgroup takes instance after instance, so the history is per workgroup and not per
// instance.  A wavefront owns a start layer with all device counts; F(s - 1) lies in LDS without
// what no scan can read (row 0, row L, column D), which lets two workgroups of 80 layers x 256
// devices share a compute unit (bound: LDS reads and the add + min behind them, 13 instructions per
// admissible candidate of 256 states).  Column 0 is +inf: F(s - 1) of zero devices is reachable for
// s = 1 only, which has a step of its own, and lanes with d < n m read it.
// Threshold batches of one search, dp_plane / dp_fused -> here: 80 x 256 (four batches, 1100
// instances) 13.2 -> 5.2 ms, 48 x 128 (600) 2.9 -> 0.7 ms, 40 x 64 1.06 -> 0.40 ms, 32 x 32 0.32 ->
// 0.20 ms; bottleneck batches of 40-48 instances 2.2 -> 1.65, 0.67 -> 0.26, 0.33 -> 0.16 and 0.16 ->
// 0.11 ms.
//   An instance ends when no larger stage count can improve its answer (`rates` given, no cost of its
// g negative): a pipeline of more than s stages ends with s stages that are some state (k, d) of
// F(s), and those in front of it put k >= 1 layers on D - d devices.  With rate = the smallest cost x
// devices / layers of a stage they sum to no less than rate k / (D - d), and the largest of them is
// no less than that either.  float32 additions of costs that are not negative lose at most 2^-24 of the
// sum each, the bound is taken 1.2e-7 short for every layer.  Stage counts of all instances of a search,
// without -> with: 40 x 64 10700 -> 3000, 48 x 128 15300 -> 6300.  And columns of F(s) are the multiples of
// the greatest common divisor of the meshes that hold an admissible stage (80 x 256: 64 or fewer columns
// for most instances, a quarter of the LDS reads).  Threshold batches of a search 80 x 256 5.6 -> 2.2 ms, 48 x
// 128 0.85 -> 0.44, 40 x 64 0.42 -> 0.30; what is left are instances whose answer has many stages (16 or 32
// steps in turn, of 300 VALU instructions per start layer), and their launches end with the longest.
// ------------------------------------------------------------------------------------------
constexpr int kDpHistoryThreads = 1024;
constexpr int kDpHistoryBatch = 10;  // meshes whose row minima a lane has in flight
constexpr int kDpUnreached = 1 << 20;
// LDS of a workgroup: F(s - 1), the smallest reached device count per row (two steps), the stage
// values of the answer's path, three flags, three bounds, the answer
inline size_t dp_history_lds(int L, int D, int max_stages) {
  const size_t f = std::max((size_t)(L - 1) * D, (size_t)(kDpHistoryThreads / 64) * 2 * (L + 1));
  return (f + 2 * (size_t)L + (size_t)max_stages + 7) * sizeof(float);
}

// A float's bits as an integer in the order of the values, either zero as +0; and back.
__device__ __forceinline__ int32_t ordered_bits(float v) {
  const int32_t bits = __float_as_int(v + 0.0f);
  return bits ^ (bits >> 31 & 0x7fffffff);
}
__device__ __forceinline__ float from_ordered_bits(int32_t bits) {
  return __int_as_float(bits ^ (bits >> 31 & 0x7fffffff));
}

// Over the re-laid row minima of every g, for dp_history_kernel: the smallest stage cost x devices / layers,
// negative where some cost is, and the smallest cost on every mesh.  out[g][1 + Q] as ordered_bits, those of
// +inf before the launch; workgroup = (share of the stage counts, mesh, g).
constexpr int kRateShares = 4;
__global__ __launch_bounds__(256) void stage_rate_kernel(const MistDpShape shape, const float *__restrict__ stage_min,
                                                         int64_t g_stride, int32_t *__restrict__ out) {
  __shared__ float lds[2][4];
  const int L = shape.num_layers, tri = dp_triangle(L), q = blockIdx.y;
  const float *__restrict__ in = stage_min + blockIdx.z * g_stride + (int64_t)q * tri;
  const float rows = 2.0f * (float)L + 1.0f;
  float per_layer = INFINITY, least = INFINITY;
  for (int x = threadIdx.x; x < tri; x += 256) {
    int k = (int)((rows - __builtin_amdgcn_sqrtf(fmaxf(rows * rows - 8.0f * (float)x, 0.0f))) * 0.5f);
    k = min(max(k, 0), L - 1);
    while (dp_triangle_row(L, k) > x) --k;
    while (k < L - 1 && dp_triangle_row(L, k + 1) <= x) ++k;
    float cost = INFINITY;
#pragma unroll 4
    for (int p = blockIdx.x; p < shape.max_stages; p += kRateShares) cost = fminf(cost, in[(int64_t)p * shape.num_mesh * tri + x]);
    least = fminf(least, cost);
    per_layer = fminf(per_layer, cost / (float)(x - dp_triangle_row(L, k) + 1));
  }
  for (int step = 1; step < 64; step <<= 1) {
    per_layer = fminf(per_layer, __shfl_xor(per_layer, step));
    least = fminf(least, __shfl_xor(least, step));
  }
  if ((threadIdx.x & 63) == 0) {
    lds[0][threadIdx.x >> 6] = per_layer;
    lds[1][threadIdx.x >> 6] = least;
  }
  __syncthreads();
  if (threadIdx.x < 2) {
    float low = fminf(fminf(lds[threadIdx.x][0], lds[threadIdx.x][1]), fminf(lds[threadIdx.x][2], lds[threadIdx.x][3]));
    if (threadIdx.x == 0) {
      low *= (float)(shape.mesh_n[q] * shape.mesh_m[q]);
      // (the quotient of the smallest negative costs is a zero)
      const float least_of_all = fminf(fminf(lds[1][0], lds[1][1]), fminf(lds[1][2], lds[1][3]));
      if (least_of_all < 0.0f) low = fminf(low, least_of_all);
    }
    if (low < INFINITY)
      atomicMin(out + (int64_t)blockIdx.z * (1 + shape.num_mesh) + (threadIdx.x == 0 ? 0 : 1 + q), ordered_bits(low));
  }
}
__device__ __forceinline__ int greatest_common_divisor(int a, int b) {
  while (b != 0) {
    const int rest = a % b;
    a = b;
    b = rest;
  }
  return a;
}

// Cost of the stage k..i on mesh q, p pre-saved micro-batches, whose state has the value `best`
// behind a successor of value `prev`: the first ckpt candidate that attains it (one wavefront).
__device__ __forceinline__ float dp_stage_value(const MistDpShape &shape, const MistDpCosts &tabs,
                                                const int64_t (&off)[4], float t_max, int p, int k,
                                                int q, int i, float prev, float best, int *arg_j) {
  const int lane = threadIdx.x & 63;
  const DpRowRef ref = dp_row_ref(shape, off, p, k, q, i);
  const float *__restrict__ costs = dp_table(tabs, ref.v, false) + ref.at;
  const int j_begin = shape.ckpt_rule == MIST_DP_CKPT_ALL ? i - k + 1 : 0;
  const int j_end = dp_j_last(shape, k, i);
  for (int j0 = j_begin; j0 <= j_end; j0 += 64) {
    const float cost = j0 + lane <= j_end ? costs[j0 + lane] : INFINITY;
    const unsigned long long hit = __ballot(cost <= t_max && cost + prev == best);
    if (hit != 0) {
      const int bit = __ffsll(hit) - 1;
      *arg_j = j0 + bit;
      return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(cost), bit));
    }
  }
  return 0.0f;
}

// Third output of an instance from the stage values of its path (stage count s at s - 1).
// Threshold: the largest; bottleneck: the sum, added from the last stage on as the threshold DP
// adds it.
template <bool kBottleneck>
__device__ __forceinline__ float dp_fold_path(const float *path_value, int n_stages) {
  float value = 0.0f;
  for (int s = 0; s < n_stages; ++s)
    value = kBottleneck ? path_value[s] + value : fmaxf(value, path_value[s]);
  return value;
}

// A stage of an instance's partition, as backtrack_kernel writes it.
__device__ __forceinline__ void dp_write_stage(int32_t *at, int end, int n, int m, int ckpt) {
  at[0] = end;
  at[1] = n;
  at[2] = m;
  at[3] = ckpt;
}

template <bool kBottleneck, int kCols>
__global__ __launch_bounds__(kDpHistoryThreads, 8) void dp_history_kernel(
    const MistDpShape shape, const MistDpCosts tabs, const float *__restrict__ tmax_list,
    const int32_t *__restrict__ g_list, int n_instances, const int32_t *__restrict__ rates, const double *estimate,
    float *__restrict__ histories, int32_t *__restrict__ best_s_out, float *__restrict__ best_sum_out,
    float *__restrict__ stage_max_out, int32_t *__restrict__ path_out) {
  extern __shared__ float dp_lds[];
  const int L = shape.num_layers, D = shape.num_devices, Q = shape.num_mesh;
  const int S = shape.max_stages, plane = L * D, tri = dp_triangle(L);
  const int n_waves = kDpHistoryThreads / 64;
  const int n_f = max((L - 1) * D, n_waves * 2 * (L + 1));
  float *f = dp_lds;  // F(s - 1) of row r >= 1, column c < W: f[(r - 1) * W + c]
  int32_t *first_col = reinterpret_cast<int32_t *>(dp_lds + n_f);  // [2][L]
  float *path_value = dp_lds + n_f + 2 * L;                        // [S]
  int32_t *reached = first_col + 2 * L + S;                        // [3]
  int32_t *bound = reached + 3;  // [3]: float bits of the smallest bound of a state
  float *answer = path_value + S + 6;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // F(s) of start layer k, column c (from 1): history[(s - 1) * plane + k * W + c - 1]
  float *history = histories + (int64_t)blockIdx.x * S * plane;
  for (int t = blockIdx.x; t < n_instances; t += gridDim.x) {
    const int64_t g = g_list[t];
    for (int x = threadIdx.x; path_out != nullptr && x < 4 * S; x += kDpHistoryThreads)
      path_out[(int64_t)t * S * 4 + x] = -1;
    if (g < 0) {  // an empty slot of the batch
      if (threadIdx.x == 0) {
        best_s_out[t] = -1;
        best_sum_out[t] = INFINITY;
        stage_max_out[t] = 0.0f;
      }
      continue;
    }
    const float *__restrict__ relaid = tabs.stage_min + g * tabs.stage_min_g_stride;
    // the bottleneck DP has no threshold of its own: an upper bound of its answer serves as one.  (Not where the
    // tables end a little above the answers: it then takes longer than it saves: 70B on
    // 32x8 547 -> 412 us, 13B on 8x8 139 -> 53, 7B on 4x8 96 -> 56.)
    float t_max = kDpNoThreshold;
    if (!kBottleneck) {
      t_max = tmax_list[t];
    } else {
      if (threadIdx.x == 0) *bound = estimate != nullptr && *estimate < (double)INFINITY;
      __syncthreads();
      if (*bound == 0) t_max = fminf(kDpNoThreshold, dp_uniform_mesh_bound(shape, relaid, f, n_f, reached));
    }
    __syncthreads();  // (the bound was read by every wavefront)
    if (threadIdx.x < 3) {
      reached[threadIdx.x] = 0;
      bound[threadIdx.x] = __float_as_int(INFINITY);
      *answer = INFINITY;
    }
    const float rate = rates != nullptr ? from_ordered_bits(rates[g * (1 + Q)]) : -1.0f;
    const bool bounded = rate >= 0.0f && rate < INFINITY;
    const float short_by = 1.0f - 1.2e-7f * (float)(L + 8);
    // stages take whole multiples of `unit` devices: a state's column is d / unit - 1, of W
    int unit = rates != nullptr ? D : 1;
    for (int q = 0; rates != nullptr && q < Q; ++q)
      if (from_ordered_bits(rates[g * (1 + Q) + 1 + q]) <= t_max)
        unit = greatest_common_divisor(unit, shape.mesh_n[q] * shape.mesh_m[q]);
    const int W = D / unit;
    // lane = mesh: columns a stage on it takes; more than there are where none of its stages is admissible
    const int its_devices = lane < Q ? shape.mesh_n[min(lane, Q - 1)] * shape.mesh_m[min(lane, Q - 1)] : 0;
    const int mesh_columns = its_devices % unit == 0 ? its_devices / unit : W + 1;
    __syncthreads();
    float answer_sum = INFINITY;  // of the lane that owns (k = 0, d = D): wavefront 0's first task
    int answer_s = -1;
    for (int s = 1; s <= S; ++s) {
      const float *__restrict__ block = relaid + (int64_t)(s - 1) * Q * tri;
      float *__restrict__ out = history + (int64_t)(s - 1) * plane;
      const int32_t *col_prev = first_col + (s & 1) * L;
      int32_t *col_cur = first_col + ((s & 1) ^ 1) * L;
      // the last stage count has one state anybody reads
      const int n_tasks = s == S ? 1 : L - s + 1;
      if (threadIdx.x == 0) {
        reached[(s + 1) % 3] = 0;
        bound[(s + 1) % 3] = __float_as_int(INFINITY);
      }
      float low = INFINITY;
      auto task = [&](auto columns, int k) {  // one start layer with all its columns, 64 at a time
        constexpr int kC = decltype(columns)::value;
        const float *__restrict__ row = block + dp_triangle_row(L, k) - k;  // row[q * tri + i]
        float best[kC];
#pragma unroll
        for (int j = 0; j < kC; ++j) best[j] = INFINITY;
        if (s == 1) {
          // the stage up to the last layer, lane = mesh
          const float mine = row[min(lane, Q - 1) * tri + L - 1];
          for (unsigned long long todo = __ballot(lane < Q && mine <= t_max); todo != 0; todo &= todo - 1) {
            const int q = __ffsll(todo) - 1;
            const float rmin = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(mine), q));
            const int nm = __builtin_amdgcn_readlane(mesh_columns, q);
#pragma unroll
            for (int j = 0; j < kC; ++j)
              if (1 + lane + 64 * j == nm) best[j] = fminf(best[j], kBottleneck ? fmaxf(rmin, 0.0f) : rmin + 0.0f);
          }
        } else {
          for (int i0 = k; i0 <= L - s; i0 += 64) {  // end layers behind which s - 1 stages fit
            const int i_mine = i0 + lane;
            const bool in_row = i_mine <= L - s;
            const int col = in_row ? col_prev[i_mine + 1] : kDpUnreached;
            for (int q0 = 0; q0 < Q; q0 += kDpHistoryBatch) {
              float r[kDpHistoryBatch];
#pragma unroll
              for (int u = 0; u < kDpHistoryBatch; ++u)
                r[u] = in_row && q0 + u < Q ? row[(q0 + u) * tri + i_mine] : INFINITY;
#pragma unroll
              for (int u = 0; u < kDpHistoryBatch; ++u) {
                if (q0 + u >= Q) break;
                // admissible, and its successor reached on what the mesh leaves: the same for
                // every lane
                const int nm = __builtin_amdgcn_readlane(mesh_columns, q0 + u);
                unsigned long long todo = __ballot(r[u] <= t_max && col + nm <= W);
                if (todo == 0) continue;
                const float *from[kC];
#pragma unroll
                for (int j = 0; j < kC; ++j) {
                  const int c = 1 + lane + 64 * j;
                  from[j] = f + (c <= W && c > nm ? c - nm : 0);
                }
                while (todo != 0) {
                  const int bit = __ffsll(todo) - 1;
                  todo &= todo - 1;
                  const float rmin = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(r[u]), bit));
                  const int at = (i0 + bit) * W;  // row i + 1
#pragma unroll
                  for (int j = 0; j < kC; ++j) {
                    const float prev = from[j][at];
                    best[j] = fminf(best[j], kBottleneck ? fmaxf(rmin, prev) : rmin + prev);
                  }
                }
              }
            }
          }
        }
        int col = kDpUnreached;
#pragma unroll
        for (int j = kC - 1; j >= 0; --j) {
          const int c = 1 + lane + 64 * j;
          if (c <= W) out[k * W + c - 1] = best[j];
          const unsigned long long finite = __ballot(c <= W && best[j] < INFINITY);
          if (finite != 0) col = 64 * j + __ffsll(finite);
          if (k > 0 && c < W) {  // with what the layers in front cost on the devices left, at least
            const float front = (float)k * rate * __builtin_amdgcn_rcpf((float)((W - c) * unit));
            low = fminf(low, kBottleneck ? fmaxf(best[j], front) : best[j] + front);
          }
          // first s wins ties (inter_tuning.py:335-340)
          if (k == 0 && c == W && best[j] < answer_sum) {
            answer_sum = best[j];
            answer_s = s;
            *answer = best[j];
          }
        }
        if (lane == 0) {
          col_cur[k] = col;
          if (col != kDpUnreached) reached[s % 3] = 1;
        }
      };
      for (int k_up = wave, round = 0; k_up < n_tasks; k_up += n_waves, ++round) {
        // snake order: the cost of a task falls with k
        int k = (round & 1) ? round * n_waves + n_waves - 1 - wave : k_up;
        if ((round + 1) * n_waves > n_tasks) k = k_up;  // the last, partial round
        if (kCols > 1 && W <= 64) task(std::integral_constant<int, 1>(), k);
        else if (kCols > 2 && W <= 128) task(std::integral_constant<int, 2>(), k);
        else task(std::integral_constant<int, kCols>(), k);
      }
      if (bounded) {
        for (int step = 1; step < 64; step <<= 1) low = fminf(low, __shfl_xor(low, step));
        if (lane == 0) atomicMin(&bound[s % 3], __float_as_int(low));
      }
      __syncthreads();  // every scan of F(s - 1) is done, F(s) is in the history
      if (s == S || reached[s % 3] == 0) break;  // (no state: none behind it either)
      if (bounded && __int_as_float(bound[s % 3]) * short_by >= *answer) break;
      for (int k = 1 + wave; k <= L - s; k += n_waves) {
        if (col_cur[k] == kDpUnreached) continue;
        for (int c = lane; c < W; c += 64) f[(k - 1) * W + c] = c == 0 ? INFINITY : out[k * W + c - 1];
      }
      __syncthreads();
    }
    __syncthreads();  // every wavefront has left the loop: `reached` is free for what the path hands over
    // the answer's path: per stage the first (mesh, end layer) that attains the value, all meshes' reads of
    // 64 end layers in flight ...
    int32_t *path = reinterpret_cast<int32_t *>(f);  // [stage count - 1][4]: start layer, end layer, mesh, value behind
    if (wave == 0) {
      const int owner = (W - 1) & 63;
      answer_s = __builtin_amdgcn_readlane(answer_s, owner);
      answer_sum = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(answer_sum), owner));
      float best = answer_sum;
      int k = 0, columns = W, missing = 0;
      for (int s = answer_s; s >= 1; --s) {
        const float *__restrict__ block = relaid + (int64_t)(s - 1) * Q * tri + dp_triangle_row(L, k) - k;
        int arg_q = Q, arg_i = -1;
        float arg_rmin = 0.0f, arg_prev = 0.0f;
        for (int i0 = s == 1 ? L - 1 : k; i0 <= L - s; i0 += 64) {
          const int i = i0 + lane;
          for (int q0 = 0; q0 < arg_q; q0 += kDpHistoryBatch) {
            float rmin[kDpHistoryBatch], prev[kDpHistoryBatch];
#pragma unroll
            for (int u = 0; u < kDpHistoryBatch; ++u) {
              const int left = q0 + u < Q ? columns - __builtin_amdgcn_readlane(mesh_columns, q0 + u) : -1;
              const bool on = i <= L - s && (s == 1 ? left == 0 : left >= 1);
              rmin[u] = on ? block[(q0 + u) * tri + i] : INFINITY;
              prev[u] = !on ? INFINITY : s == 1 ? 0.0f : history[(int64_t)(s - 2) * plane + (i + 1) * W + left - 1];
            }
#pragma unroll
            for (int u = 0; u < kDpHistoryBatch; ++u) {
              if (q0 + u >= arg_q) continue;
              const float target = kBottleneck ? fmaxf(rmin[u], prev[u]) : rmin[u] + prev[u];
              const unsigned long long hit = __ballot(rmin[u] <= t_max && target == best);
              if (hit == 0) continue;
              const int bit = __ffsll(hit) - 1;
              arg_q = q0 + u;
              arg_i = i0 + bit;
              arg_rmin = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(rmin[u]), bit));
              arg_prev = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(prev[u]), bit));
            }
          }
        }
        if (arg_q >= Q) {  // (a reached state has a candidate that attains its value)
          missing = s;
          break;
        }
        if (lane == 0) {
          path[4 * (s - 1)] = k;
          path[4 * (s - 1) + 1] = arg_i;
          path[4 * (s - 1) + 2] = arg_q;
          path[4 * (s - 1) + 3] = __float_as_int(arg_prev);
          path_value[s - 1] = kBottleneck ? arg_rmin : best;
        }
        columns -= __builtin_amdgcn_readlane(mesh_columns, arg_q);
        k = arg_i + 1;
        best = arg_prev;
      }
      if (lane == 0) {
        reached[0] = answer_s;
        reached[1] = missing;
      }
    }
    __syncthreads();
    // ... then the first ckpt count of every stage, a wavefront each
    const int its_s = reached[0];
    const int64_t off[4] = {g * tabs.g_stride[0], g * tabs.g_stride[1], g * tabs.g_stride[2], g * tabs.g_stride[3]};
    for (int s = reached[1] + 1 + wave; s <= its_s; s += n_waves) {
      const int k = path[4 * (s - 1)], i = path[4 * (s - 1) + 1], q = path[4 * (s - 1) + 2];
      int arg_j = -1;
      if (!kBottleneck) {
        const float value = dp_stage_value(shape, tabs, off, t_max, s - 1, k, q, i, __int_as_float(path[4 * (s - 1) + 3]),
                                           path_value[s - 1], &arg_j);
        if (lane == 0) path_value[s - 1] = value;
      }
      if (lane == 0 && path_out != nullptr)
        dp_write_stage(path_out + ((int64_t)t * S + its_s - s) * 4, i, shape.mesh_n[q], shape.mesh_m[q], arg_j);
    }
    __syncthreads();
    if (threadIdx.x == 0) {
      best_s_out[t] = answer_s;
      best_sum_out[t] = answer_sum;
      stage_max_out[t] = dp_fold_path<kBottleneck>(path_value, answer_s);
    }
    __syncthreads();  // the next instance writes the history and LDS
  }
}

// ------------------------------------------------------------------------------------------
// The recurrence of one mesh for all stages (free_devices): a state is a start layer, F(s) has
// L + 1 values, and all of them stay in LDS.  With a launch per stage count a search of 6 stage
// counts (1, 2, .. 32) in four batches made 250 launches of 3 to 8 us with as long a gap behind
// each.  Here a workgroup runs an instance through all stage counts: per count the row minima
// (consecutive end layers of a stage length are neighbours in the tables), read while the count
// before is worked on, go to LDS, then eight lanes take a start layer.  Bound: LDS latency and two
// barriers, 0.7 us per stage count at 37 layers.  (Read where they are needed, each place from its
// row and variant, and a wavefront a start layer, five in turn with six exchanges each: 2.5 us; the
// four launches of 13B on 4x8 100, 219, 89 and 76 us; then 34, 153, 30 and 27 with the tables' addresses
// in scratch, now 25, 70, 24 and 23.)  Six families of that plan: 250 launches, 3.3 ms from the first to
// the last -> 18, 0.75.
// The families of a search wait for nothing of each other: up to kDpFreeFamilies go through one
// launch, workgroup = (instance, family), the ones given last (more stage counts as a rule) first:
// 24 launches, 0.89 ms of 13B on 4x8 -> 4, 0.50.
// ------------------------------------------------------------------------------------------
constexpr int kDpFreeThreads = 512;
constexpr int kDpFreeLoads = 4, kDpFreeMostLoads = 16;  // values a thread reads ahead: up to 45 layers, up to 90
constexpr int kDpFreeFamilies = 8;
struct DpFreeFamily {
  MistDpCosts costs;
  int32_t max_stages, p_dim, ckpt_rule, mesh_n, mesh_m;
  int32_t *best_s, *path;
  float *best_sum, *stage_max;
};
struct DpFreeFamilies {
  DpFreeFamily family[kDpFreeFamilies];
};
inline size_t dp_free_lds(int L, int S) {
  return ((size_t)L * L + (size_t)(S + 1) * (L + 1) + S) * sizeof(float);
}

// Smallest value of eight neighbouring lanes, in each of them.
__device__ __forceinline__ float eight_lane_min(float v) {
#define MIST_MIN_DPP(CTRL) v = fminf(v, __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), CTRL, 0xf, 0xf, true)))
  MIST_MIN_DPP(0xB1);   // quad_perm [1,0,3,2]
  MIST_MIN_DPP(0x4E);   // quad_perm [2,3,0,1]
  MIST_MIN_DPP(0x141);  // row_half_mirror
#undef MIST_MIN_DPP
  return v;
}

template <bool kBottleneck, int kLoads>
__global__ __launch_bounds__(kDpFreeThreads) void dp_free_kernel(
    const DpFreeFamilies families, int num_layers, const float *__restrict__ tmax_list,
    const int32_t *__restrict__ g_list) {
  extern __shared__ float dp_lds[];
  const DpFreeFamily &its = families.family[gridDim.y - 1 - blockIdx.y];
  const MistDpCosts tabs = its.costs;
  int32_t *__restrict__ best_s_out = its.best_s, *__restrict__ path_out = its.path;
  float *__restrict__ best_sum_out = its.best_sum, *__restrict__ stage_max_out = its.stage_max;
  MistDpShape shape;  // (of one mesh)
  shape.num_layers = num_layers;
  shape.num_devices = 0;
  shape.num_mesh = 1;
  shape.p_dim = its.p_dim;
  shape.max_stages = its.max_stages;
  shape.ckpt_rule = its.ckpt_rule;
  shape.free_devices = 1;
  shape.mesh_n[0] = its.mesh_n;
  shape.mesh_m[0] = its.mesh_m;
  const int L = shape.num_layers, S = shape.max_stages;
  float *rows = dp_lds;                             // [L][L] (stage layers - 1, end layer)
  float *history = rows + L * L;                    // [S + 1][L + 1]
  float *path_value = history + (S + 1) * (L + 1);  // [S]
  const int t = blockIdx.x;
  const int64_t g = g_list[t];
  for (int x = threadIdx.x; path_out != nullptr && x < 4 * S; x += kDpFreeThreads)
    path_out[(int64_t)t * S * 4 + x] = -1;
  if (g < 0) {  // an empty slot of the batch
    if (threadIdx.x == 0) {
      best_s_out[t] = -1;
      best_sum_out[t] = INFINITY;
      stage_max_out[t] = 0.0f;
    }
    return;
  }
  const int64_t off[4] = {g * tabs.g_stride[0], g * tabs.g_stride[1], g * tabs.g_stride[2],
                          g * tabs.g_stride[3]};
  const float t_max = kBottleneck ? kDpNoThreshold : tmax_list[t];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  for (int k = threadIdx.x; k <= L; k += kDpFreeThreads) history[k] = k == L ? 0.0f : INFINITY;
  // row minima of the stages (k, i) behind which s - 1 layers are left (s = 1: none); the first kLoads values of a
  // thread are read a stage count ahead, from places that move by one plane of the tables with it
  const bool all_ckpt = shape.ckpt_rule == MIST_DP_CKPT_ALL;
  const DpRows rows_of_g = dp_rows(shape, tabs, g);
  const float *__restrict__ inner = rows_of_g.inner, *__restrict__ front = rows_of_g.pre;
  const int held = rows_of_g.planes == nullptr ? S : rows_of_g.planes[0];
  int end_of[kLoads], place[kLoads];
#pragma unroll
  for (int u = 0; u < kLoads; ++u) {
    const int x = threadIdx.x + u * kDpFreeThreads, i = x % L, k = i - x / L;
    end_of[u] = x < L * L && k >= 0 ? i : L;  // (no end layer: never read)
    place[u] = k < 0 ? 0 : (((i - k) * (L + 1) + (all_ckpt ? i - k + 1 : dp_j_last(shape, k, i))) << 1) | (k == 0 ? 1 : 0);
  }
  auto row_min = [&](int s, int x) {
    const int i = x % L, k = i - x / L;
    const bool wanted = x < L * L && k >= 0 && i <= L - s && (s > 1 || i == L - 1);
    return wanted ? dp_row_min(rows_of_g, s - 1, k, 0, i) : INFINITY;
  };
  auto put = [&](int x, float value) {
    if (x < L * L) rows[x] = value <= t_max ? value : INFINITY;
  };
  float value[kLoads];
#pragma unroll
  for (int u = 0; u < kLoads; ++u) value[u] = row_min(1, threadIdx.x + u * kDpFreeThreads);
  for (int s = 1; s <= S; ++s) {
    const float *f_prev = history + (s - 1) * (L + 1);
    float *f_cur = history + s * (L + 1);
#pragma unroll
    for (int u = 0; u < kLoads; ++u) put(threadIdx.x + u * kDpFreeThreads, value[u]);
    for (int x = threadIdx.x + kLoads * kDpFreeThreads; x < L * L; x += kDpFreeThreads) put(x, row_min(s, x));
    __syncthreads();
    if (s < S) {
      const int64_t plane = (int64_t)s * L * (L + 1);
#pragma unroll
      for (int u = 0; u < kLoads; ++u) {
        const float *__restrict__ from = ((place[u] & 1) != 0 ? front : inner) + plane;
        value[u] = end_of[u] < L - s && s < held ? from[place[u] >> 1] : INFINITY;
      }
    }
    // eight lanes a start layer
    for (int k = threadIdx.x / 8; k <= L; k += kDpFreeThreads / 8) {
      float best = INFINITY;
      for (int i = k + (threadIdx.x & 7); i <= L - s; i += 8) {
        const float rmin = rows[(i - k) * L + i], prev = f_prev[i + 1];
        // (an inadmissible row is +inf here, and so is its target)
        best = fminf(best, kBottleneck ? fmaxf(rmin, prev) : rmin + prev);
      }
      best = eight_lane_min(best);
      if ((threadIdx.x & 7) == 0) f_cur[k] = best;
    }
    __syncthreads();
  }
  if (wave != 0) return;
  // first s wins ties (inter_tuning_uniform_device.py:335-340)
  float answer_sum = INFINITY;
  int answer_s = -1;
  for (int s = 1; s <= S; ++s) {
    const float sum = history[s * (L + 1)];
    if (sum < answer_sum) {
      answer_sum = sum;
      answer_s = s;
    }
  }
  int k = 0;
  for (int s = answer_s; s >= 1; --s) {
    const float *f_prev = history + (s - 1) * (L + 1);
    const float best = history[s * (L + 1) + k];
    int arg_i = -1;
    float arg_rmin = 0.0f;
    for (int i0 = k; i0 <= L - s && arg_i < 0; i0 += 64) {
      const int i = i0 + lane;
      float rmin = INFINITY, target = INFINITY;
      if (i <= L - s && f_prev[i + 1] < INFINITY) {
        rmin = dp_row_min(rows_of_g, s - 1, k, 0, i);
        target = kBottleneck ? fmaxf(rmin, f_prev[i + 1]) : rmin + f_prev[i + 1];
      }
      const unsigned long long hit = __ballot(rmin <= t_max && target == best);
      if (hit != 0) {
        const int bit = __ffsll(hit) - 1;
        arg_i = i0 + bit;
        arg_rmin = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(rmin), bit));
      }
    }
    if (arg_i < 0) break;  // (a reached state has a candidate that attains its value)
    int arg_j = -1;
    const float value = kBottleneck ? arg_rmin
                                    : dp_stage_value(shape, tabs, off, t_max, s - 1, k, 0, arg_i,
                                                     f_prev[arg_i + 1], best, &arg_j);
    if (lane == 0) {
      path_value[s - 1] = value;
      if (path_out != nullptr)
        dp_write_stage(path_out + ((int64_t)t * S + answer_s - s) * 4, arg_i, shape.mesh_n[0],
                       shape.mesh_m[0], arg_j);
    }
    k = arg_i + 1;
  }
  if (lane == 0) {
    best_s_out[t] = answer_s;
    best_sum_out[t] = answer_sum;
    stage_max_out[t] = dp_fold_path<kBottleneck>(path_value, answer_s);
  }
}

// Follows the back-pointers of each instance from (best_s, layer 0, all devices) and writes its
// stages in pipeline order (inter_tuning.py:341-355); one thread per instance.  Only entries the
// DP wrote are read: a state with a finite value has a winner, and so has every successor on
// its path.
__global__ __launch_bounds__(64) void backtrack_kernel(const MistDpShape shape,
                                                       const int32_t *__restrict__ argmin,
                                                       const int32_t *__restrict__ best_s, int n,
                                                       int32_t *__restrict__ path) {
  const int t = blockIdx.x * 64 + threadIdx.x;
  if (t >= n) return;
  const int L = shape.num_layers, W = shape.num_devices + 1;
  const int64_t plane = (int64_t)(L + 1) * W;
  int32_t *out = path + (int64_t)t * shape.max_stages * 4;
  for (int i = 0; i < shape.max_stages * 4; ++i) out[i] = -1;
  int s = best_s[t], k = 0, d = shape.num_devices, stage = 0;
  while (s > 0 && k < L && stage < shape.max_stages) {
    const int32_t *a = argmin + (((int64_t)t * (shape.max_stages + 1) + s) * plane + k * W + d) * 4;
    const int end = a[0], mesh_n = a[1], mesh_m = a[2];
    // an entry the DP did not write (caller's fill or stale memory) ends the walk: the host sees
    // a path that does not cover the layers
    if (end < k || end >= L || mesh_n < 1 || mesh_m < 1) break;
    if (shape.free_devices == 0 && mesh_n * mesh_m > d) break;
    dp_write_stage(out + stage * 4, end, mesh_n, mesh_m, a[3]);
    ++stage;
    --s;
    k = end + 1;
    if (shape.free_devices == 0) d -= mesh_n * mesh_m;
  }
}

// Row minima in the order the recurrence reads them: out[g][p][q][triangle(k, i)] =
// dp_row_min(p, k, q, i).  A workgroup scanning stage count p + 1 of g finds all it needs in one
// contiguous block, and the end layers i of one (q, k) lie next to each other.
// Workgroup = (p, mesh, g).  The row minima of inner stages with l layers lie side by side for the start
// layers, descending: read in that order (kMinimaLoads of a lane in flight), turned in LDS, written in the
// other one.  Planes that hold nothing are written alone.  Bound: the 4 bytes an entry.  (A thread per entry,
// each its own cache line, and as many threads for the planes that hold nothing: 70B on 32x8 409 us, 291 without
// reading those, now 96; 7B on 4x8 18 -> 11.)
constexpr int kMinimaLoads = 8;
constexpr int kMinimaLayers = 180;  // the turned triangle fits 64 KB
__device__ __forceinline__ void store_entries(float *__restrict__ to, int n, float value) {
  for (int x = threadIdx.x * 4; x < n; x += 1024) {
    if (x + 4 <= n) {
      *reinterpret_cast<AnyFloat4 *>(to + x) = AnyFloat4{value, value, value, value};
    } else {
      for (int u = x; u < n; ++u) to[u] = value;
    }
  }
}
// (start layer, length) of an entry of the triangle
__device__ __forceinline__ int dp_triangle_start(int L, int x) {
  const float rows = 2.0f * (float)L + 1.0f;
  int k = (int)((rows - __builtin_amdgcn_sqrtf(fmaxf(rows * rows - 8.0f * (float)x, 0.0f))) * 0.5f);
  k = min(max(k, 0), L - 1);
  while (dp_triangle_row(L, k) > x) --k;
  while (k < L - 1 && dp_triangle_row(L, k + 1) <= x) ++k;
  return k;
}
__global__ __launch_bounds__(256) void stage_minima_kernel(const MistDpShape shape,
                                                           const MistDpCosts tabs,
                                                           float *__restrict__ out, bool in_lds) {
  extern __shared__ float dp_lds[];
  const int L = shape.num_layers, tri = dp_triangle(L);
  const int p = blockIdx.x / shape.num_mesh, q = blockIdx.x % shape.num_mesh;
  const int64_t g = blockIdx.y;
  float *__restrict__ mine = out + ((g * shape.max_stages + p) * shape.num_mesh + q) * tri;
  const DpRows rows_of_g = dp_rows(shape, tabs, g);
  if (rows_of_g.planes != nullptr && p >= rows_of_g.planes[q]) {
    store_entries(mine, tri, INFINITY);
    return;
  }
  // rows of l layers, entry k: at l - 1 rows of L - l' + 1 entries each
  if (in_lds) {
    const bool all = shape.ckpt_rule == MIST_DP_CKPT_ALL;
    const float *__restrict__ table = rows_of_g.inner + ((int64_t)q * shape.p_dim + p) * L * (L + 1);
    for (int x0 = threadIdx.x; x0 < tri; x0 += kMinimaLoads * 256) {
      float value[kMinimaLoads];
#pragma unroll
      for (int u = 0; u < kMinimaLoads; ++u) {
        const int x = x0 + u * 256;
        value[u] = INFINITY;
        if (x >= tri) continue;
        const int l = dp_triangle_start(L, x) + 1, k = x - dp_triangle_row(L, l - 1), i = k + l - 1;
        if (k == 0 || i == L - 1) continue;
        value[u] = table[(int64_t)(l - 1) * (L + 1) + (all ? l : dp_j_last(shape, k, i))];
      }
#pragma unroll
      for (int u = 0; u < kMinimaLoads; ++u)
        if (x0 + u * 256 < tri) dp_lds[x0 + u * 256] = value[u];
    }
    __syncthreads();
  }
  // a stage count of p + 1 leaves start layers k <= L - 1 - p
  for (int x = threadIdx.x; x < tri; x += 256) {
    const int k = dp_triangle_start(L, x), di = x - dp_triangle_row(L, k);
    float value = INFINITY;
    if (k <= L - 1 - p)
      value = in_lds && k > 0 && k + di < L - 1 ? dp_lds[dp_triangle_row(L, di) + k]
                                                : dp_row_min(rows_of_g, p, k, q, k + di);
    mine[x] = value;
  }
}

// Dynamic LDS the one-launch kernel may use on the current device: what the device reports per
// workgroup, once the kernel has been allowed more than the default 64 KB (0 if that failed).
size_t lds_limit_of(const void *kernel) {
  int device = 0, most = 0;
  if (hipGetDevice(&device) != hipSuccess ||
      hipDeviceGetAttribute(&most, hipDeviceAttributeMaxSharedMemoryPerBlock, device) != hipSuccess)
    return 0;
  if (most > 64 * 1024 &&
      hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, most) != hipSuccess) {
    (void)hipGetLastError();
    most = 64 * 1024;
  }
  return (size_t)most;
}
template <bool kBottleneck>
size_t fused_lds_limit_of() {
  return lds_limit_of(reinterpret_cast<const void *>(&dp_fused_kernel<kBottleneck>));
}
// Allows the window walk the LDS of its largest windows (more than the default 64 KB), once per device.
int allow_window_lds() {
  static std::mutex lock;
  static std::set<int> allowed;
  int device = 0;
  MIST_HIP_CHECK(hipGetDevice(&device));
  std::lock_guard<std::mutex> guard(lock);
  if (allowed.count(device) != 0) return 0;
  MIST_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void *>(&window_walk_kernel),
                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)window_lds(kWindowMost)));
  allowed.insert(device);
  return 0;
}
size_t plane_lds_limit(int mode) {
  // per device: the attribute belongs to the device's copy of the kernel
  static std::mutex lock;
  static std::map<std::pair<int, int>, size_t> known;
  int device = 0;
  if (hipGetDevice(&device) != hipSuccess) return 0;
  std::lock_guard<std::mutex> guard(lock);
  const auto key = std::make_pair(device, mode);
  auto it = known.find(key);
  if (it == known.end())
    it = known.emplace(key, lds_limit_of(mode == MIST_DP_BOTTLENECK
                                             ? reinterpret_cast<const void *>(&dp_plane_kernel<true>)
                                             : reinterpret_cast<const void *>(&dp_plane_kernel<false>))).first;
  return it->second;
}
size_t fused_lds_limit(int mode) {
  // per device: the attribute belongs to the device's copy of the kernel
  static std::mutex lock;
  static std::map<std::pair<int, int>, size_t> known;
  int device = 0;
  if (hipGetDevice(&device) != hipSuccess) return 0;
  std::lock_guard<std::mutex> guard(lock);
  const auto key = std::make_pair(device, mode);
  auto it = known.find(key);
  if (it == known.end())
    it = known.emplace(key, mode == MIST_DP_BOTTLENECK ? fused_lds_limit_of<true>()
                                                       : fused_lds_limit_of<false>()).first;
  return it->second;
}

// Workgroups, floats of history and LDS of dp_history_kernel for a batch; n_wg 0: not this shape.
// Two workgroups per compute unit; a history that would take more than a GiB for one workgroup
// per compute unit is left to the schedules that keep two planes.
struct HistoryPlan {
  int n_wg = 0;
  int64_t floats = 0;
  size_t lds = 0;
};
constexpr int64_t kDpHistoryMaxFloats = (int64_t)256 << 20;
constexpr int kDpComputeUnits = 256;
HistoryPlan history_plan(const MistDpShape &shape, int n_tmax) {
  HistoryPlan plan;
  if (shape.free_devices != 0 || shape.num_devices > 256 || shape.max_stages < 1) return plan;
  plan.lds = dp_history_lds(shape.num_layers, shape.num_devices, shape.max_stages);
  if (plan.lds > kDpLdsPerCu) return plan;
  const int64_t each = (int64_t)shape.max_stages * shape.num_layers * shape.num_devices;
  const int64_t n_wg = std::min<int64_t>(std::min(n_tmax, 2 * kDpComputeUnits), kDpHistoryMaxFloats / each);
  if (n_wg < std::min(n_tmax, kDpComputeUnits)) return plan;
  plan.n_wg = (int)n_wg;
  plan.floats = n_wg * each;
  return plan;
}
template <bool kBottleneck>
const void *history_kernel(int cols) {
  return cols == 1   ? reinterpret_cast<const void *>(&dp_history_kernel<kBottleneck, 1>)
         : cols == 2 ? reinterpret_cast<const void *>(&dp_history_kernel<kBottleneck, 2>)
         : cols == 3 ? reinterpret_cast<const void *>(&dp_history_kernel<kBottleneck, 3>)
                     : reinterpret_cast<const void *>(&dp_history_kernel<kBottleneck, 4>);
}
size_t history_lds_limit(int mode, int cols) {
  // per device: the attribute belongs to the device's copy of the kernel
  static std::mutex lock;
  static std::map<std::tuple<int, int, int>, size_t> known;
  int device = 0;
  if (hipGetDevice(&device) != hipSuccess) return 0;
  std::lock_guard<std::mutex> guard(lock);
  const auto key = std::make_tuple(device, mode, cols);
  auto it = known.find(key);
  if (it == known.end())
    it = known.emplace(key, lds_limit_of(mode == MIST_DP_BOTTLENECK ? history_kernel<true>(cols)
                                                                    : history_kernel<false>(cols))).first;
  return it->second;
}

// Scratch of mist_dp_run_static: callers that must not allocate (HIP graph capture, serving
// loops) get the state planes from this array instead of a workspace argument.  Every GPU the
// library runs on holds its own copy at its own address until the process ends.
constexpr int64_t kStaticScratchFloats = (int64_t)4 << 20;  // 16 MiB
static __device__ __align__(256) float scratch[kStaticScratchFloats];
constexpr int kMaxKnownDevices = 64;

// Device address of `scratch` on the current device.  In host code the array's name is only a
// handle for hipGetSymbolAddress, never a pointer a kernel can use; the address is looked up
// once per device (with that device current) and kept.
int static_scratch_of_current_device(float **out) {
  static std::mutex lock;
  static float *known[kMaxKnownDevices] = {};
  int device = 0;
  MIST_HIP_CHECK(hipGetDevice(&device));
  if (device < 0 || device >= kMaxKnownDevices)
    return fail(MIST_E_INVALID, "device ordinal %d outside [0, %d)", device, kMaxKnownDevices);
  std::lock_guard<std::mutex> guard(lock);
  if (known[device] == nullptr) {
    void *ptr = nullptr;
    MIST_HIP_CHECK(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
    if (ptr == nullptr) return fail(MIST_E_HIP, "hipGetSymbolAddress returned a null address");
    known[device] = static_cast<float *>(ptr);
  }
  *out = known[device];
  return 0;
}

int check_shape(const MistDpShape *shape) {
  if (!shape) return fail(MIST_E_INVALID, "null DP shape");
  if (shape->free_devices != 0 && (shape->num_devices != 0 || shape->num_mesh != 1))
    return fail(MIST_E_INVALID, "free_devices needs num_devices = 0 and one mesh (got D=%d Q=%d)",
                shape->num_devices, shape->num_mesh);
  if (shape->ckpt_rule < MIST_DP_CKPT_TAIL || shape->ckpt_rule > MIST_DP_CKPT_ALL)
    return fail(MIST_E_INVALID, "unknown ckpt_rule %d", shape->ckpt_rule);
  if (shape->num_layers <= 0 || shape->p_dim <= 0 ||
      (shape->free_devices ? shape->num_devices != 0 : shape->num_devices <= 0))
    return fail(MIST_E_INVALID, "bad DP extents L=%d D=%d P+1=%d", shape->num_layers,
                shape->num_devices, shape->p_dim);
  if (shape->num_mesh <= 0 || shape->num_mesh > MIST_MAX_MESH)
    return fail(MIST_E_INVALID, "num_mesh %d outside [1, %d]", shape->num_mesh, MIST_MAX_MESH);
  if (shape->max_stages < 0 || shape->max_stages > shape->p_dim)
    return fail(MIST_E_INVALID, "max_stages %d exceeds the p axis (%d) of the cost tables",
                shape->max_stages, shape->p_dim);
  if (shape->max_stages > shape->num_layers)
    return fail(MIST_E_INVALID, "max_stages %d exceeds num_layers %d", shape->max_stages,
                shape->num_layers);
  for (int q = 0; q < shape->num_mesh; ++q)
    if (shape->mesh_n[q] <= 0 || shape->mesh_m[q] <= 0)
      return fail(MIST_E_INVALID, "mesh %d is (%d, %d)", q, shape->mesh_n[q], shape->mesh_m[q]);
  return 0;
}

int check_run_arguments(const MistDpShape *shape, const MistDpCosts *costs, const float *d_tmax,
                        const int32_t *d_g_index, int n_tmax, int mode, const int32_t *d_best_s,
                        const float *d_best_sum, const float *d_stage_max) {
  if (int rc = check_shape(shape)) return rc;
  if (!costs || !costs->costs || !costs->costs_pre || !costs->costs_post || !costs->costs_nopp ||
      !costs->pmin || !costs->pmin_pre || !costs->pmin_post || !costs->pmin_nopp)
    return fail(MIST_E_INVALID, "null cost table");
  if (!d_tmax || !d_g_index || !d_best_s || !d_best_sum || !d_stage_max)
    return fail(MIST_E_INVALID, "null threshold / output pointer");
  if (n_tmax <= 0 || n_tmax > 65535)
    return fail(MIST_E_INVALID, "n_tmax must be in [1, 65535], got %d", n_tmax);
  if (mode != MIST_DP_THRESHOLD && mode != MIST_DP_BOTTLENECK)
    return fail(MIST_E_INVALID, "unknown DP mode %d", mode);
  return 0;
}

// Workgroups of a request of the candidate selection: few, long-running ones, each of which appends to the
// output list once per kSelectBuffer values at most.
unsigned select_blocks(int64_t per_row) { return (unsigned)std::min<int64_t>((per_row + 16383) / 16384, 64); }

// Small batches are latency-bound: spread every state over a team of lanes.
bool dp_wide_teams(int n_tmax, int plane) { return (int64_t)n_tmax * plane <= (1 << 19); }

// One launch per stage count; the state planes and reachable ranges of all instances live in
// d_scratch (mist_dp_scratch_floats() floats, no particular contents expected on entry: the
// first kernel writes everything a later one reads).
int run_step_schedule(const MistDpShape *shape, const MistDpCosts *costs, const float *d_tmax,
                      const int32_t *d_g_index, int n_tmax, int mode, int32_t *d_best_s,
                      float *d_best_sum, float *d_stage_max, int32_t *d_argmin, float *d_scratch,
                      void *stream) {
  const int plane = (shape->num_layers + 1) * (shape->num_devices + 1);
  const bool wide = dp_wide_teams(n_tmax, plane);
  const int64_t n_init = (int64_t)n_tmax * plane;
  int32_t *d_ranges = reinterpret_cast<int32_t *>(d_scratch + (int64_t)4 * n_tmax * plane);
  hipLaunchKernelGGL(dp_init_kernel, dim3((unsigned)((n_init + 255) / 256)), dim3(256), 0,
                     (hipStream_t)stream, *shape, n_tmax, d_scratch, d_ranges, d_best_s,
                     d_best_sum, d_stage_max);
  MIST_HIP_CHECK(hipGetLastError());
  const int states_per_block = kDpThreads / (wide ? kDpWideTeam : 1);
  const dim3 grid((plane + states_per_block - 1) / states_per_block, n_tmax);
  for (int s = 1; s <= shape->max_stages; ++s) {
#define MIST_DP_STEP(BOTTLENECK, TEAM)                                                         \
  hipLaunchKernelGGL((dp_step_kernel<BOTTLENECK, TEAM>), grid, dim3(kDpThreads), 0,            \
                     (hipStream_t)stream, *shape, *costs, d_tmax, d_g_index, s, d_scratch,     \
                     d_ranges, d_best_s, d_best_sum, d_stage_max, d_argmin)
    if (mode == MIST_DP_BOTTLENECK) {
      if (wide) MIST_DP_STEP(true, kDpWideTeam); else MIST_DP_STEP(true, 1);
    } else {
      if (wide) MIST_DP_STEP(false, kDpWideTeam); else MIST_DP_STEP(false, 1);
    }
#undef MIST_DP_STEP
    MIST_HIP_CHECK(hipGetLastError());
  }
  return 0;
}

}  // namespace

extern "C" {

int mist_sizeof_dp_shape(void) { return (int)sizeof(MistDpShape); }

int mist_dp_cost_tables(const MistProblem *problem, const MistOutTables *tables,
                        const int32_t *d_grad_accum, int slot, float *const d_out[4],
                        float *const d_out_pmin[4], void *stream) {
  if (!problem || !tables || !d_grad_accum || !d_out || !d_out_pmin)
    return fail(MIST_E_INVALID, "null pointer argument");
  const int64_t L = problem->num_layers, P1 = problem->p_dim, S = problem->sample_size;
  const int64_t Gn = problem->num_grad_accum, Q = problem->num_mesh;
  if (L <= 0 || P1 <= 0 || S <= 0 || Gn <= 0 || Q <= 0)
    return fail(MIST_E_INVALID, "bad problem extents");
  if (slot < 0 || slot >= S) return fail(MIST_E_INVALID, "slot %d outside [0, %d)", slot, (int)S);
  const int64_t rows_per_g[4] = {Q * P1 * L, Q * P1 * L, Q * L, Q};
  const bool wide = S == 1 && L + 1 <= 256;  // four neighbouring cells a lane, rows of a wavefront's cells at most
  const int64_t rows_per_set = wide ? (kCostCells / (L + 1)) & ~3ll : 256 / std::min<int64_t>(L + 1, 256);
  int64_t sets = 0;
  for (int v = 0; v < 4; ++v) sets += Gn * rows_per_g[v] / rows_per_set;
  CostTableJob job = {};
  job.runs = (int)std::max<int64_t>(1, std::min<int64_t>(kCostRuns, sets / kCostResident));
  const int64_t rows_per_block = rows_per_set * job.runs;
  int64_t blocks = 0;
  for (int v = 0; v < 4; ++v) {
    if (!tables->stable[v] || !tables->delta[v] || !d_out[v] || !d_out_pmin[v])
      return fail(MIST_E_INVALID, "table %d is null", v);
    job.stable[v] = tables->stable[v];
    job.delta[v] = tables->delta[v];
    job.index[v] = tables->index[v];
    job.out[v] = d_out[v];
    job.pmin[v] = d_out_pmin[v];
    job.n_rows[v] = Gn * rows_per_g[v];
    job.rows_per_g[v] = rows_per_g[v];
    job.first_block[v] = (unsigned)blocks;
    blocks += (job.n_rows[v] + rows_per_block - 1) / rows_per_block;
  }
  if (blocks >= (int64_t)1 << 31) return fail(MIST_E_INVALID, "cost tables too large for one launch");
  job.first_block[4] = (unsigned)blocks;
  if (wide)
    hipLaunchKernelGGL(cost_rows_kernel, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream, job, d_grad_accum,
                       (int)(L + 1));
  else
    hipLaunchKernelGGL(cost_table_kernel, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream, job,
                       d_grad_accum, (int)(L + 1), (int)S, slot);
  MIST_HIP_CHECK(hipGetLastError());
  return 0;
}

int mist_dp_cost_planes(const MistProblem *problem, const MistOutTables *tables, const int32_t *d_grad_accum,
                        const int32_t *d_planes, float *const d_out[4], float *const d_out_pmin[4], void *stream) {
  if (!problem || !tables || !d_grad_accum || !d_planes || !d_out || !d_out_pmin)
    return fail(MIST_E_INVALID, "null pointer argument");
  const int64_t L = problem->num_layers, P1 = problem->p_dim, Gn = problem->num_grad_accum, Q = problem->num_mesh;
  if (L <= 0 || P1 <= 0 || Gn <= 0 || Q <= 0) return fail(MIST_E_INVALID, "bad problem extents");
  if (problem->sample_size != 1 || L + 1 > 256)
    return fail(MIST_E_INVALID, "cost planes of one sample and rows of up to 256 cells, got %d samples, %d layers",
                problem->sample_size, (int)L);
  if (Gn > 65535 || Q > 65535 || P1 * L >= (int64_t)1 << 24) return fail(MIST_E_INVALID, "cost tables too large for one launch");
  CostPlanesJob job = {};
  for (int v = 0; v < 4; ++v) {
    if (!tables->stable[v] || !tables->delta[v] || !tables->index[v] || !d_out[v] || !d_out_pmin[v])
      return fail(MIST_E_INVALID, "table %d is null", v);
    job.stable[v] = tables->stable[v];
    job.delta[v] = tables->delta[v];
    job.index[v] = tables->index[v];
    job.out[v] = d_out[v];
    job.pmin[v] = d_out_pmin[v];
  }
  job.planes = d_planes;
  job.grad_accum = d_grad_accum;
  job.L = (int)L;
  job.P1 = (int)P1;
  const int64_t rows_here = (kCostCells / (L + 1)) & ~3ll;
  const int64_t sets = 2 * ((P1 * L + rows_here - 1) / rows_here) + (L + rows_here - 1) / rows_here + 1;
  const int64_t blocks = std::max<int64_t>(1, std::min(sets, kCostPlaneBlocks / (Gn * Q)));
  hipLaunchKernelGGL(cost_planes_kernel, dim3((unsigned)blocks, (unsigned)Q, (unsigned)Gn), dim3(256), 0,
                     (hipStream_t)stream, job);
  MIST_HIP_CHECK(hipGetLastError());
  return 0;
}

int mist_dp_backtrack(const MistDpShape *shape, const int32_t *d_argmin, const int32_t *d_best_s,
                      int n_tmax, int32_t *d_path, void *stream) {
  if (int rc = check_shape(shape)) return rc;
  if (!d_argmin || !d_best_s || !d_path) return fail(MIST_E_INVALID, "null pointer argument");
  if (n_tmax <= 0 || n_tmax > 65535)
    return fail(MIST_E_INVALID, "n_tmax must be in [1, 65535], got %d", n_tmax);
  hipLaunchKernelGGL(backtrack_kernel, dim3((unsigned)((n_tmax + 63) / 64)), dim3(64), 0,
                     (hipStream_t)stream, *shape, d_argmin, d_best_s, n_tmax, d_path);
  MIST_HIP_CHECK(hipGetLastError());
  return 0;
}

int64_t mist_dp_stage_minima_floats(const MistDpShape *shape) {
  if (check_shape(shape) != 0) return -1;
  return (int64_t)shape->max_stages * shape->num_mesh * dp_triangle(shape->num_layers);
}

int mist_dp_stage_minima(const MistDpShape *shape, const MistDpCosts *costs, int num_grad_accum,
                         float *d_out, void *stream) {
  if (int rc = check_shape(shape)) return rc;
  if (!costs || !costs->costs || !costs->costs_pre || !costs->costs_post || !costs->costs_nopp ||
      !costs->pmin || !costs->pmin_pre || !costs->pmin_post || !costs->pmin_nopp)
    return fail(MIST_E_INVALID, "null cost table");
  if (!d_out) return fail(MIST_E_INVALID, "null output pointer");
  if (num_grad_accum < 1 || num_grad_accum > 65535)
    return fail(MIST_E_INVALID, "num_grad_accum must be in [1, 65535], got %d", num_grad_accum);
  if (shape->max_stages == 0) return 0;
  const bool in_lds = shape->num_layers <= kMinimaLayers;
  hipLaunchKernelGGL(stage_minima_kernel, dim3((unsigned)(shape->max_stages * shape->num_mesh), (unsigned)num_grad_accum),
                     dim3(256), in_lds ? sizeof(float) * dp_triangle(shape->num_layers) : 0, (hipStream_t)stream, *shape,
                     *costs, d_out, in_lds);
  MIST_HIP_CHECK(hipGetLastError());
  return 0;
}

int mist_dp_filter_tmax(const float *sorted_unique, int n, double gap, float *out) {
  if (n < 0 || (n > 0 && (!sorted_unique || !out))) return fail(MIST_E_INVALID, "bad t_max list");
  int kept = 0;
  float last = 0.0f;
  for (int i = 0; i < n; ++i) {
    const float t = sorted_unique[i];
    if (gap_below(t, last, gap)) continue;
    out[kept++] = t;
    last = t;
  }
  return kept;
}

int mist_dp_window_begin(const float *ascending, int n, float lo, int open_below,
                         float start_value, double gap, float *out) {
  if (n < 0 || (n > 0 && (!ascending || !out))) return fail(MIST_E_INVALID, "bad candidate list");
  if (n == 0) return 0;
  const int first = window_walk_start(ascending, n, lo, open_below != 0, start_value, gap);
  if (first < 0) return MIST_DP_NO_START;
  return mist_dp_filter_tmax(ascending + first, n - first, gap, out);  // the walk from there
}

int mist_dp_window_begin_many(const float *ascending, const int64_t *offsets, int n_windows,
                              const float *lo, const uint8_t *open_below,
                              const float *start_value, double gap, float *out,
                              int32_t *out_count) {
  if (n_windows < 0) return fail(MIST_E_INVALID, "n_windows %d < 0", n_windows);
  if (n_windows == 0) return 0;
  if (!offsets || !lo || !open_below || !start_value || !out_count)
    return fail(MIST_E_INVALID, "null pointer argument");
  for (int w = 0; w < n_windows; ++w) {
    const int64_t first = offsets[w], count = offsets[w + 1] - first;
    if (first < 0 || count < 0 || count > INT32_MAX)
      return fail(MIST_E_INVALID, "offsets of window %d are not ascending", w);
    const int kept =
        mist_dp_window_begin(count ? ascending + first : nullptr, (int)count, lo[w], open_below[w],
                             start_value[w], gap, count ? out + first : nullptr);
    if (kept < 0 && kept != MIST_DP_NO_START) return kept;
    out_count[w] = kept;
  }
  return 0;
}

int mist_dp_select_candidates(const MistDpCosts *costs, int n_requests, const int32_t *d_rows,
                              const float *d_lo, const float *d_hi, float *d_out_values,
                              int32_t *d_out_request, int capacity, int32_t *d_counts,
                              void *stream) {
  if (!costs || !costs->costs || !costs->costs_pre || !costs->costs_post)
    return fail(MIST_E_INVALID, "null cost tables");
  if (costs->planes && (costs->planes_g_stride < 1 || costs->planes_g_stride > MIST_MAX_MESH))
    return fail(MIST_E_INVALID, "planes of %d meshes", (int)costs->planes_g_stride);
  if (n_requests <= 0 || n_requests > 65535)
    return fail(MIST_E_INVALID, "n_requests %d outside [1, 65535]", n_requests);
  if (!d_rows || !d_lo || !d_hi || !d_out_values || !d_out_request || !d_counts || capacity <= 0)
    return fail(MIST_E_INVALID, "null pointer / empty output list");
  const int64_t per_row = costs->g_stride[0] + costs->g_stride[1] + costs->g_stride[2];
  const unsigned blocks = select_blocks(per_row);
  hipLaunchKernelGGL(select_candidates_kernel, dim3(blocks, n_requests), dim3(256), 0,
                     (hipStream_t)stream, *costs, d_rows, d_lo, d_hi, d_out_values, d_out_request,
                     capacity, d_counts, false);
  MIST_HIP_CHECK(hipGetLastError());
  return 0;
}

int mist_dp_first_batch_index(int k, int n_avail, int first_chunk, int first_lead) {
  if (k < 0 || first_chunk < 1 || first_lead < 1 || k >= std::min(first_chunk, n_avail)) return -1;
  return dp_first_batch_index(k, n_avail, first_chunk, first_lead);
}

int mist_dp_windows_first_batch(const MistDpCosts *costs, int n_requests, const int32_t *d_rows,
                                const float *d_lo, const float *d_hi, const float *d_start,
                                double gap, int window_capacity, int first_chunk, int first_lead,
                                float *d_values, int32_t *d_counts, float *d_kept,
                                int kept_capacity, int32_t *d_meta, float *d_inst_tmax,
                                int32_t *d_inst_row, void *stream) {
  return mist::dp_windows_first_batch(costs, n_requests, d_rows, d_lo, d_hi, d_start, gap, window_capacity, first_chunk,
                                      first_lead, d_values, d_counts, d_kept, kept_capacity, d_meta, d_inst_tmax,
                                      d_inst_row, false, (hipStream_t)stream);
}

int64_t mist_dp_scratch_floats(const MistDpShape *shape, int n_tmax) {
  if (check_shape(shape) != 0 || n_tmax <= 0) return -1;
  // four state planes per instance, then three buffers of (first, last) reachable row per
  // instance and device column
  return (int64_t)4 * n_tmax * (shape->num_layers + 1) * (shape->num_devices + 1) +
         (int64_t)6 * n_tmax * (shape->num_devices + 1);
}

int64_t mist_dp_scratch_floats_sized(const MistDpShape *shape, int n_tmax) {
  const int64_t least = mist_dp_scratch_floats(shape, n_tmax);
  return least < 0 ? least : std::max(least, history_plan(*shape, n_tmax).floats);
}

int mist_dp_run(const MistDpShape *shape, const MistDpCosts *costs, const float *d_tmax,
                const int32_t *d_g_index, int n_tmax, int mode, int32_t *d_best_s,
                float *d_best_sum, float *d_stage_max, int32_t *d_argmin, float *d_scratch,
                void *stream) {
  return mist_dp_run_sized(shape, costs, d_tmax, d_g_index, n_tmax, mode, d_best_s, d_best_sum,
                           d_stage_max, d_argmin, nullptr, d_scratch,
                           mist_dp_scratch_floats(shape, n_tmax), stream);
}

}  // extern "C"

int mist::dp_windows_first_batch(const MistDpCosts *costs, int n_requests, const int32_t *d_rows,
                                const float *d_lo, const float *d_hi, const float *d_start,
                                double gap, int window_capacity, int first_chunk, int first_lead,
                                float *d_values, int32_t *d_counts, float *d_kept,
                                int kept_capacity, int32_t *d_meta, float *d_inst_tmax,
                                int32_t *d_inst_row, bool cleared, hipStream_t st) {
  if (!costs || !costs->costs || !costs->costs_pre || !costs->costs_post)
    return fail(MIST_E_INVALID, "null cost tables");
  if (costs->planes && (costs->planes_g_stride < 1 || costs->planes_g_stride > MIST_MAX_MESH))
    return fail(MIST_E_INVALID, "planes of %d meshes", (int)costs->planes_g_stride);
  if (n_requests <= 0 || n_requests > 65535)
    return fail(MIST_E_INVALID, "n_requests %d outside [1, 65535]", n_requests);
  if (!d_rows || !d_lo || !d_hi || !d_start || !d_values || !d_counts || !d_kept || !d_meta ||
      !d_inst_tmax || !d_inst_row)
    return fail(MIST_E_INVALID, "null pointer argument");
  if (window_capacity < 128 || window_capacity > kWindowMost || (window_capacity & (window_capacity - 1)))
    return fail(MIST_E_INVALID, "window_capacity %d is no power of two in [128, %d]", window_capacity, kWindowMost);
  if (first_chunk < 1 || kept_capacity < 1 || (int64_t)n_requests * first_chunk > 65535)
    return fail(MIST_E_INVALID, "first_chunk %d x %d requests outside [1, 65535] / empty kept list",
                first_chunk, n_requests);
  if (first_lead < 1) return fail(MIST_E_INVALID, "first_lead %d < 1", first_lead);
  const int n_counts = 2 + 2 * n_requests, n_inst = n_requests * first_chunk;
  if (!cleared) {
    hipLaunchKernelGGL(window_clear_kernel, dim3((unsigned)((std::max(n_counts, n_inst) + 255) / 256)), dim3(256), 0, st,
                       d_counts, n_counts, d_inst_row, n_inst);
    MIST_HIP_CHECK(hipGetLastError());
  }
  const int64_t per_row = costs->g_stride[0] + costs->g_stride[1] + costs->g_stride[2];
  const unsigned blocks = select_blocks(per_row);
  hipLaunchKernelGGL(select_candidates_kernel, dim3(blocks, n_requests), dim3(256), 0, st, *costs,
                     d_rows, d_lo, d_hi, d_values, (int32_t *)nullptr, window_capacity, d_counts,
                     true);
  MIST_HIP_CHECK(hipGetLastError());
  const size_t lds = window_lds(window_capacity);
  if (int rc = allow_window_lds()) return rc;
  hipLaunchKernelGGL(window_walk_kernel, dim3(n_requests), dim3(kWindowThreads), lds, st, d_values,
                     window_capacity, d_counts, d_rows, d_lo, d_start, gap, first_chunk, first_lead,
                     d_kept, kept_capacity, d_meta, d_inst_tmax, d_inst_row);
  MIST_HIP_CHECK(hipGetLastError());
  return 0;
}

int mist::dp_stage_rates(const MistDpShape &shape, const MistDpCosts &costs, int n_g, int32_t *d_rates, hipStream_t stream) {
  if (costs.stage_min == nullptr || n_g < 1 || n_g > 65535) return fail(MIST_E_INVALID, "no row minima or %d tables", n_g);
  hipLaunchKernelGGL(stage_rate_kernel, dim3(kRateShares, shape.num_mesh, n_g), dim3(256), 0, stream, shape,
                     costs.stage_min, costs.stage_min_g_stride, d_rates);
  MIST_HIP_CHECK(hipGetLastError());
  return 0;
}

// Whether the whole recurrence of one mesh fits a workgroup.
static bool dp_free_runs(const MistDpShape &shape) {
  return shape.free_devices != 0 && dp_free_lds(shape.num_layers, shape.max_stages) <= 64 * 1024;
}
static int launch_dp_free(const mist::DpFreeRun *runs, int n, const float *d_tmax, const int32_t *d_g_index, int n_tmax,
                          int mode, hipStream_t stream) {
  for (int first = 0; first < n; first += kDpFreeFamilies) {
    const int here = std::min(n - first, kDpFreeFamilies), L = runs[first].shape->num_layers;
    DpFreeFamilies families = {};
    size_t lds = 0;
    for (int f = 0; f < here; ++f) {
      const mist::DpFreeRun &run = runs[first + f];
      const MistDpShape &shape = *run.shape;
      families.family[f] = {*run.costs, shape.max_stages, shape.p_dim, shape.ckpt_rule, shape.mesh_n[0], shape.mesh_m[0],
                            run.d_best_s, run.d_path, run.d_best_sum, run.d_stage_max};
      lds = std::max(lds, dp_free_lds(L, shape.max_stages));
    }
    const bool few = L * L <= kDpFreeLoads * kDpFreeThreads;
    const auto kernel = mode == MIST_DP_BOTTLENECK
                            ? (few ? dp_free_kernel<true, kDpFreeLoads> : dp_free_kernel<true, kDpFreeMostLoads>)
                            : (few ? dp_free_kernel<false, kDpFreeLoads> : dp_free_kernel<false, kDpFreeMostLoads>);
    hipLaunchKernelGGL(kernel, dim3(n_tmax, here), dim3(kDpFreeThreads), lds, stream, families, L, d_tmax, d_g_index);
    MIST_HIP_CHECK(hipGetLastError());
  }
  return 0;
}

int mist::dp_run_free(const DpFreeRun *runs, int n, const float *d_tmax, const int32_t *d_g_index, int n_tmax, int mode,
                      hipStream_t stream) {
  const char *forced = getenv("MIST_DP_FORCE_SCHEDULE");
  if (forced && *forced) return 1;
  for (int f = 0; f < n; ++f)
    if (!dp_free_runs(*runs[f].shape) || runs[f].shape->num_layers != runs[0].shape->num_layers) return 1;
  for (int f = 0; f < n; ++f)
    if (int rc = check_run_arguments(runs[f].shape, runs[f].costs, d_tmax, d_g_index, n_tmax, mode, runs[f].d_best_s,
                                     runs[f].d_best_sum, runs[f].d_stage_max))
      return rc;
  return launch_dp_free(runs, n, d_tmax, d_g_index, n_tmax, mode, stream);
}

static bool history_possible(const MistDpShape &shape, const MistDpCosts &costs, int mode, int64_t scratch_floats,
                             const HistoryPlan &plan) {
  return plan.n_wg > 0 && costs.stage_min != nullptr && plan.floats <= scratch_floats &&
         plan.lds <= history_lds_limit(mode, (shape.num_devices + 63) / 64);
}
bool mist::dp_keeps_paths(const MistDpShape &shape, const MistDpCosts &costs, int n_tmax, int mode, int64_t scratch_floats) {
  const char *forced = getenv("MIST_DP_FORCE_SCHEDULE");
  if (forced && *forced) return false;
  return dp_free_runs(shape) || history_possible(shape, costs, mode, scratch_floats, history_plan(shape, n_tmax));
}

int mist::dp_run(const MistDpShape *shape, const MistDpCosts *costs, const int32_t *d_rates, const double *estimate, const float *d_tmax,
                 const int32_t *d_g_index, int n_tmax, int mode, int32_t *d_best_s, float *d_best_sum,
                 float *d_stage_max, int32_t *d_argmin, int32_t *d_path, float *d_scratch, int64_t scratch_floats,
                 void *stream) {
  if (int rc = check_run_arguments(shape, costs, d_tmax, d_g_index, n_tmax, mode, d_best_s,
                                   d_best_sum, d_stage_max))
    return rc;
  if (!d_scratch) return fail(MIST_E_INVALID, "null scratch pointer");
  if (d_path && !d_argmin && !dp_keeps_paths(*shape, *costs, n_tmax, mode, scratch_floats))
    return fail(MIST_E_INVALID, "d_path needs d_argmin");
  const bool whole_argmin = d_argmin != nullptr && d_path == nullptr;
  const int plane = (shape->num_layers + 1) * (shape->num_devices + 1);
  const bool wide = dp_wide_teams(n_tmax, plane);
  // Larger ones: one workgroup per instance with its planes in LDS when they fit and the caller
  // prepared the re-laid row minima.
  const size_t fused_lds =
      ((size_t)4 * plane + (size_t)6 * (shape->num_devices + 1) +
       (size_t)shape->num_mesh * dp_triangle(shape->num_layers) +
       (size_t)2 * shape->num_mesh * shape->num_layers) *
      sizeof(float);
  // (threshold batches from about 64 instances on: a workgroup's run through all stage counts
  // takes as long as the 1 + max_stages launches of a few dozen instances)
  bool fused_pays = mode == MIST_DP_THRESHOLD ? n_tmax >= kDpFusedMinInstances : !wide;
  // (small planes: a workgroup's run through all stage counts is shorter than the launches it
  // replaces whatever the batch size - GPT-7B's 33 x 33 plane: bottleneck batch of 40 instances
  // and the back-pointer run of one, 0.07 ms per search; 41 x 65 is already the other way round)
  fused_pays = fused_pays || plane <= kDpFusedSmallPlane;
  // For tests: MIST_DP_FORCE_SCHEDULE = step | fused | plane takes the choice of schedule away
  // from the batch size and the LDS need, so that each schedule can be run on any shape it
  // supports (a shape it does not support is an error, not a silent fallback).
  const char *forced = getenv("MIST_DP_FORCE_SCHEDULE");
  const bool force_step = forced && !strcmp(forced, "step");
  const bool force_fused = forced && !strcmp(forced, "fused");
  const bool force_plane = forced && !strcmp(forced, "plane");
  const bool force_history = forced && !strcmp(forced, "history");
  if (forced && *forced && !force_step && !force_fused && !force_plane && !force_history)
    return fail(MIST_E_INVALID, "MIST_DP_FORCE_SCHEDULE=%s: expected step, fused, plane or history", forced);
  // Without back-pointers and with room for the history that schedule runs: it was the fastest at
  // every shape and batch size measured (33 x 33 to 81 x 257 states, 28 to 2304 instances).
  if (!(force_step || force_fused || force_plane)) {
    if (!whole_argmin && dp_free_runs(*shape)) {
      const mist::DpFreeRun run = {shape, costs, d_best_s, d_best_sum, d_stage_max, d_path};
      return launch_dp_free(&run, 1, d_tmax, d_g_index, n_tmax, mode, (hipStream_t)stream);
    }
    const HistoryPlan plan = history_plan(*shape, n_tmax);
    const int cols = (shape->num_devices + 63) / 64;
    const bool possible = !whole_argmin && history_possible(*shape, *costs, mode, scratch_floats, plan);
    if (force_history && !possible)
      return fail(MIST_E_INVALID, "forced history schedule: needs stage_min, consumed devices, D <= 256, no "
                  "back-pointers, %lld scratch floats and %zu B of LDS", (long long)plan.floats, plan.lds);
    if (possible) {
      const MistDpShape shape_arg = *shape;
      const MistDpCosts costs_arg = *costs;
      int n_arg = n_tmax;
      void *args[] = {(void *)&shape_arg, (void *)&costs_arg, &d_tmax, &d_g_index, &n_arg, &d_rates,
                      &estimate, &d_scratch, &d_best_s, &d_best_sum, &d_stage_max, &d_path};
      MIST_HIP_CHECK(hipLaunchKernel(mode == MIST_DP_BOTTLENECK ? history_kernel<true>(cols)
                                                                : history_kernel<false>(cols),
                                     dim3(plan.n_wg), dim3(kDpHistoryThreads), args, plan.lds,
                                     (hipStream_t)stream));
      MIST_HIP_CHECK(hipGetLastError());
      return 0;
    }
  }
  if (d_path) {
    if (int rc = dp_run(shape, costs, d_rates, estimate, d_tmax, d_g_index, n_tmax, mode, d_best_s, d_best_sum,
                        d_stage_max, d_argmin, nullptr, d_scratch, scratch_floats, stream))
      return rc;
    return mist_dp_backtrack(shape, d_argmin, d_best_s, n_tmax, d_path, stream);
  }
  if (force_fused) {
    if (costs->stage_min == nullptr || fused_lds > fused_lds_limit(mode))
      return fail(MIST_E_INVALID, "forced fused schedule: needs stage_min and %zu B of LDS", fused_lds);
    fused_pays = true;
  }
  if (force_step || force_plane) fused_pays = false;
  if (fused_pays && costs->stage_min != nullptr && fused_lds <= fused_lds_limit(mode)) {
    // one workgroup per CU when the planes take more than half of the LDS: then a larger one
    const int most = 2 * fused_lds > kDpLdsPerCu ? kDpFusedThreads : kDpFusedThreads / 2;
    const int threads = std::min(most, (plane + 63) / 64 * 64);
    if (mode == MIST_DP_BOTTLENECK)
      hipLaunchKernelGGL(dp_fused_kernel<true>, dim3(n_tmax), dim3(threads), fused_lds,
                         (hipStream_t)stream, *shape, *costs, d_tmax, d_g_index, d_best_s,
                         d_best_sum, d_stage_max, d_argmin);
    else
      hipLaunchKernelGGL(dp_fused_kernel<false>, dim3(n_tmax), dim3(threads), fused_lds,
                         (hipStream_t)stream, *shape, *costs, d_tmax, d_g_index, d_best_s,
                         d_best_sum, d_stage_max, d_argmin);
    MIST_HIP_CHECK(hipGetLastError());
    return 0;
  }
  // Planes beyond the LDS of a compute unit (80 layers x 256 devices): one workgroup per instance
  // with F(s - 1) alone in LDS, one launch.
  const size_t plane_lds =
      ((size_t)plane + 6 * (size_t)(shape->num_devices + 1) + 2 * (size_t)shape->num_mesh +
       (size_t)(kDpPlaneThreads / 64) * shape->num_mesh * shape->num_layers) * sizeof(float);
  const bool plane_shape_ok = shape->num_devices <= 64 * kDpPlaneCols &&
                              shape->num_mesh * shape->num_layers <= 64 * kDpPlaneLoads &&
                              shape->num_layers <= 256;  // (mesh << 8 | end layer) of a winner
  const bool plane_possible = costs->stage_min != nullptr && shape->free_devices == 0 &&
                              plane_shape_ok && plane_lds <= plane_lds_limit(mode);
  if (force_plane && !plane_possible)
    return fail(MIST_E_INVALID, "forced plane schedule: needs stage_min, consumed devices, D <= %d, "
                "Q * L <= %d and %zu B of LDS", 64 * kDpPlaneCols, 64 * kDpPlaneLoads, plane_lds);
  if (plane_possible && !force_step &&
      (force_plane || (n_tmax >= kDpPlaneMinInstances && fused_lds > fused_lds_limit(mode)))) {
    if (mode == MIST_DP_BOTTLENECK)
      hipLaunchKernelGGL(dp_plane_kernel<true>, dim3(n_tmax), dim3(kDpPlaneThreads), plane_lds,
                         (hipStream_t)stream, *shape, *costs, d_tmax, d_g_index, d_scratch,
                         d_best_s, d_best_sum, d_stage_max, d_argmin);
    else
      hipLaunchKernelGGL(dp_plane_kernel<false>, dim3(n_tmax), dim3(kDpPlaneThreads), plane_lds,
                         (hipStream_t)stream, *shape, *costs, d_tmax, d_g_index, d_scratch,
                         d_best_s, d_best_sum, d_stage_max, d_argmin);
    MIST_HIP_CHECK(hipGetLastError());
    return 0;
  }
  return run_step_schedule(shape, costs, d_tmax, d_g_index, n_tmax, mode, d_best_s, d_best_sum,
                           d_stage_max, d_argmin, d_scratch, stream);
}

extern "C" {

int mist_dp_run_sized(const MistDpShape *shape, const MistDpCosts *costs, const float *d_tmax,
                      const int32_t *d_g_index, int n_tmax, int mode, int32_t *d_best_s,
                      float *d_best_sum, float *d_stage_max, int32_t *d_argmin, int32_t *d_path,
                      float *d_scratch, int64_t scratch_floats, void *stream) {
  if (d_path && !d_argmin) return fail(MIST_E_INVALID, "d_path needs d_argmin");
  return mist::dp_run(shape, costs, nullptr, nullptr, d_tmax, d_g_index, n_tmax, mode, d_best_s, d_best_sum, d_stage_max,
                      d_argmin, d_path, d_scratch, scratch_floats, stream);
}

int64_t mist_dp_static_scratch_floats(void) { return kStaticScratchFloats; }

int mist_dp_run_static(const MistDpShape *shape, const MistDpCosts *costs, const float *d_tmax,
                       const int32_t *d_g_index, int n_tmax, int mode, int32_t *d_best_s,
                       float *d_best_sum, float *d_stage_max, int32_t *d_argmin, void *stream) {
  if (int rc = check_run_arguments(shape, costs, d_tmax, d_g_index, n_tmax, mode, d_best_s,
                                   d_best_sum, d_stage_max))
    return rc;
  const int64_t need = mist_dp_scratch_floats(shape, n_tmax);
  if (need < 0 || need > kStaticScratchFloats)
    return fail(MIST_E_INVALID,
                "mist_dp_run_static: %d instances of (L=%d, D=%d) need %lld scratch floats, the "
                "built-in scratch holds %lld; use mist_dp_run with a caller-owned scratch",
                n_tmax, shape->num_layers, shape->num_devices, (long long)need,
                (long long)kStaticScratchFloats);
  float *d_scratch = nullptr;
  if (int rc = static_scratch_of_current_device(&d_scratch)) return rc;
  return run_step_schedule(shape, costs, d_tmax, d_g_index, n_tmax, mode, d_best_s, d_best_sum,
                           d_stage_max, d_argmin, d_scratch, stream);
}

}  // extern "C"
