// Between the reduction and the search driver: how far below the smallest feasible threshold the search reads stage
// costs as threshold candidates.  A window begins window_margin below it and is fetched again from kMarginGrowth
// times as far while it has no certain start; what MistProblem.incumbent_close leaves out lies below
// kExactMargins of them, and a search that goes further than kExactWidenings times calls its result undecided.
#pragma once
#include <hip/hip_runtime.h>

#include <cmath>

namespace mist {
constexpr double kMarginGrowth = 4.0;
constexpr int kExactWidenings = 2;
constexpr double margins_of(int widenings) { return widenings == 0 ? 1.0 : kMarginGrowth * margins_of(widenings - 1); }
constexpr double kExactMargins = margins_of(kExactWidenings);

__host__ __device__ inline double window_margin(double threshold) { return 1e-4 + 1e-5 * fabs(threshold); }
}  // namespace mist
