// lu_device.hpp -- device LU of the marker systems (lu_device.hip).
#pragma once

#include <hip/hip_runtime.h>

namespace lumagpu {

// Below this many markers the host's whole chain is done before the device's pivots (3.5 us each) and the
// copies; above kLuDeviceMax a panel's rows outgrow a block's
// registers, and the host solves.
constexpr int kLuDeviceMin = 192, kLuDeviceMax = 4096;
// Nonzeros per marker up to which the host solves the matrix that the device made: chains and rings of
// markers a cell apart have about 7, and their factors stay sparse, where the device's work grows with n^3;
// surfaces of such markers about 30.  A gradient over 4 steps, dense on the device -> on the host: chain of
// 200 / 800 / 1600 markers 1.8 -> 1.0, 6.6 -> 2.7, 32 -> 8 ms, ring of 1600 33 -> 13; all on the host
// 1.9, 7.3, 26, 32; a sphere of 1600 is 35 ms on the device, 176 on the host.
constexpr int kLuSparse = 12;

// The factors of lu_solve's column-major view, in place (a[j * n + i], unit lower triangle below the
// diagonal), piv[j] = the row swapped with row j, *info = 0 or 1 + the column of a zero pivot;
// device pointers, asynchronous on s.
hipError_t lu_factor_device(int n, double *a, int *piv, int *info, hipStream_t s);
// x = the solution of the transposed system (lu_solve's substitutions) from factors on the host
void lu_substitute(int n, const double *a, const int *piv, double *x);

}  // namespace lumagpu
