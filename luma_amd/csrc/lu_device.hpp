// lu_device.hpp -- device LU of the marker systems (lu_device.hip).
#pragma once

#include <hip/hip_runtime.h>

namespace lumagpu {

// Below this many markers the host's banded or dense solve is done before the device's chain of
// pivots (3.5 us each) and the copies; above kLuDeviceMax a panel's rows outgrow a block's
// registers, and the host solves.
constexpr int kLuDeviceMin = 192, kLuDeviceMax = 4096;

// The factors of lu_solve's column-major view, in place (a[j * n + i], unit lower triangle below the
// diagonal), piv[j] = the row swapped with row j, *info = 0 or 1 + the column of a zero pivot;
// device pointers, asynchronous on s.
hipError_t lu_factor_device(int n, double *a, int *piv, int *info, hipStream_t s);
// x = the solution of the transposed system (lu_solve's substitutions) from factors on the host
void lu_substitute(int n, const double *a, const int *piv, double *x);

}  // namespace lumagpu
