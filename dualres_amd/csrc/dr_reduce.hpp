// Reduction operators whose handling of NaN matters.
#pragma once

#include <hip/hip_runtime.h>

namespace drh {

// the larger of a and b, NaN if either is
__host__ __device__ inline double max_nan(double a, double b) { return a != a || b <= a ? a : b; }

}  // namespace drh
