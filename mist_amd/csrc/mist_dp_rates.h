// Between the DP and the search driver: mist_dp_run_sized with what ends an instance early, and several
// families of one mesh at a time.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

#include "mist_dp.h"

namespace mist {
// d_rates[n_g][1 + num_mesh], kRateNone before the call: over costs.stage_min of every g the smallest stage
// cost x devices / layers (negative where a cost is), and the smallest cost on every mesh, as the floats'
// bits with the lower 31 of a negative one inverted: in the order of the values, for an integer minimum.
constexpr int32_t kRateNone = 0x7f800000;  // +inf
int dp_stage_rates(const MistDpShape &shape, const MistDpCosts &costs, int n_g, int32_t *d_rates, hipStream_t stream);

// mist_dp_run_sized; `d_rates` (may be null) holds what dp_stage_rates left for every g the instances name.
// `estimate` (device address, may be null): where it is finite when the kernels run, the tables hold next to nothing
// above what pipelines cost, and the bottleneck DP looks for no bound of its answer first.  d_path without d_argmin:
// where dp_keeps_paths.
int dp_run(const MistDpShape *shape, const MistDpCosts *costs, const int32_t *d_rates, const double *estimate, const float *d_tmax,
           const int32_t *d_g_index, int n_tmax, int mode, int32_t *d_best_s, float *d_best_sum, float *d_stage_max,
           int32_t *d_argmin, int32_t *d_path, float *d_scratch, int64_t scratch_floats, void *stream);

// Whether a run without back-pointers knows the partition of every instance.
bool dp_keeps_paths(const MistDpShape &shape, const MistDpCosts &costs, int n_tmax, int mode, int64_t scratch_floats);

// mist_dp_windows_first_batch; `cleared`: d_counts (2 + 2 n_requests) hold zeros and d_inst_row -1.
int dp_windows_first_batch(const MistDpCosts *costs, int n_requests, const int32_t *d_rows, const float *d_lo,
                           const float *d_hi, const float *d_start, double gap, int window_capacity, int first_chunk,
                           int first_lead, float *d_values, int32_t *d_counts, float *d_kept, int kept_capacity,
                           int32_t *d_meta, float *d_inst_tmax, int32_t *d_inst_row, bool cleared, hipStream_t stream);

struct DpFreeRun {
  const MistDpShape *shape;
  const MistDpCosts *costs;
  int32_t *d_best_s;
  float *d_best_sum, *d_stage_max;
  int32_t *d_path;  // may be null
};
// dp_run of the same instances for every family, all on one mesh, without a launch per family; > 0 and nothing
// is done where a family needs another schedule.
int dp_run_free(const DpFreeRun *runs, int n, const float *d_tmax, const int32_t *d_g_index, int n_tmax, int mode,
                hipStream_t stream);
}  // namespace mist
