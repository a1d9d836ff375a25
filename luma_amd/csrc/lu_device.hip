// lu_device.hip -- LU factorisation with row pivoting of the marker systems (A eps = 1) on the device, for the
// position gradient of large bodies (adjoint.hip).
//
// The systems are dense in storage and a few hundred to a few thousand markers large.  lu_solve on the
// host takes its rank-1 updates one column after another; here the same operations run column
// panel by column panel: one block factors a panel held in registers (a thread holds whole rows
// of it), then one block per remaining column swaps its rows, solves the panel's triangle and
// updates the rest.  Every element takes its updates in the order of the column they come from,
// as in dgetf2, and the first largest pivot is taken, so the factors are the host's (up to the
// sign of zeros, which the host's loops skip).  A chain of n pivots bounds it, 3.5 us each
// (two barriers, the pivot's reduction and its row's way through LDS): 804 markers 3.3 ms.
#include <hip/hip_runtime.h>

#include <string>

#include "aa_kernels.hpp"
#include "internal.hpp"
#include "lu_device.hpp"

namespace lumagpu {
namespace {

// Columns j0 .. j0 + NB - 1 of the column-major n x n matrix, rows from j0 on; piv[j] the row swapped
// with j, *info = j + 1 at the first zero pivot.  One block of 1024 threads, RPT rows each.
template <int RPT, int NB>
__global__ __launch_bounds__(1024) void k_lu_panel(int n, int j0, double *a, int *piv, int *info) {
    __shared__ double pb[NB], jb[NB], redv[16];
    __shared__ int redi[16];
    if (*info) return;   // an earlier panel met a zero pivot
    const int t = threadIdx.x, w = min(NB, n - j0);
    double row[RPT][NB];
    int ri[RPT];
#pragma unroll
    for (int r = 0; r < RPT; ++r) {
        ri[r] = j0 + t + 1024 * r;
#pragma unroll
        for (int c = 0; c < NB; ++c) row[r][c] = (ri[r] < n && c < w) ? a[(size_t)(j0 + c) * n + ri[r]] : 0.0;
    }
    bool ok = true;
    static_for<NB>([&](auto jc) {
        constexpr int jj = decltype(jc)::value;
        if (!ok || jj >= w) return;   // the same in every thread
        const int j = j0 + jj;
        double bv = -1.0;
        int bi = n;
#pragma unroll
        for (int r = 0; r < RPT; ++r) {
            const double v = ::fabs(row[r][jj]);
            if (ri[r] >= j && ri[r] < n && v > bv) {
                bv = v;
                bi = ri[r];
            }
        }
        for (int off = 32; off > 0; off >>= 1) {
            const double ov = __shfl_xor(bv, off, 64);
            const int oi = __shfl_xor(bi, off, 64);
            if (ov > bv || (ov == bv && oi < bi)) {
                bv = ov;
                bi = oi;
            }
        }
        if ((t & 63) == 0) {
            redv[t >> 6] = bv;
            redi[t >> 6] = bi;
        }
        __syncthreads();
        bv = redv[0];
        int p = redi[0];
        for (int k = 1; k < 16; ++k)
            if (redv[k] > bv || (redv[k] == bv && redi[k] < p)) {
                bv = redv[k];
                p = redi[k];
            }
        if (p >= n) p = j;   // no comparable entry (NaN): as the host, which keeps the diagonal
#pragma unroll
        for (int r = 0; r < RPT; ++r) {
            if (ri[r] == p)
#pragma unroll
                for (int c = 0; c < NB; ++c) pb[c] = row[r][c];
            if (ri[r] == j)
#pragma unroll
                for (int c = 0; c < NB; ++c) jb[c] = row[r][c];
        }
        __syncthreads();
        if (pb[jj] == 0.0) {
            ok = false;
            if (t == 0) *info = j + 1;
            return;
        }
        if (t == 0) piv[j] = p;
        const double rcp = 1.0 / pb[jj];
#pragma unroll
        for (int r = 0; r < RPT; ++r) {
            if (ri[r] == j) {
#pragma unroll
                for (int c = 0; c < NB; ++c) row[r][c] = pb[c];
            } else if (ri[r] > j && ri[r] < n) {
                if (ri[r] == p) {
#pragma unroll
                    for (int c = 0; c < NB; ++c) row[r][c] = jb[c];
                }
                const double l = row[r][jj] * rcp;
                row[r][jj] = l;
#pragma unroll
                for (int c = jj + 1; c < NB; ++c) row[r][c] -= l * pb[c];
            }
        }
    });
#pragma unroll
    for (int r = 0; r < RPT; ++r)
#pragma unroll
        for (int c = 0; c < NB; ++c)
            if (ri[r] < n && c < w) a[(size_t)(j0 + c) * n + ri[r]] = row[r][c];
}

// One block per column outside the panel: its row swaps and, right of the panel, its updates.
template <int NB>
__global__ __launch_bounds__(256) void k_lu_update(int n, int j0, double *a, const int *piv, const int *info) {
    extern __shared__ double col[];   // [n]
    __shared__ double u[NB];
    const int k = blockIdx.x, t = threadIdx.x, w = min(NB, n - j0);
    if (*info || (k >= j0 && k < j0 + w)) return;
    double *ck = a + (size_t)k * n;
    for (int i = t; i < n; i += 256) col[i] = ck[i];
    __syncthreads();
    if (t == 0)
        for (int jj = 0; jj < w; ++jj) {
            const int p = piv[j0 + jj];
            const double x = col[j0 + jj];
            col[j0 + jj] = col[p];
            col[p] = x;
        }
    __syncthreads();
    if (k >= j0 + w) {
        if (t < 64) {   // the triangle of the panel's own rows, a lane per row
            const bool in = t < w;
            double v = in ? col[j0 + t] : 0.0;
            for (int jj = 0; jj < w; ++jj) {
                const double uj = __shfl(v, jj, 64);
                if (in && t > jj) v -= a[(size_t)(j0 + jj) * n + j0 + t] * uj;
            }
            if (in) {
                u[t] = v;
                col[j0 + t] = v;
            }
        }
        __syncthreads();
        for (int i = j0 + w + t; i < n; i += 256) {
            double v = col[i];
            for (int jj = 0; jj < w; ++jj) v -= a[(size_t)(j0 + jj) * n + i] * u[jj];
            col[i] = v;
        }
        __syncthreads();
    }
    for (int i = t; i < n; i += 256) ck[i] = col[i];
}

template <int RPT, int NB>
hipError_t factor(int n, double *a, int *piv, int *info, hipStream_t s) {
    for (int j0 = 0; j0 < n; j0 += NB) {
        k_lu_panel<RPT, NB><<<1, 1024, 0, s>>>(n, j0, a, piv, info);
        k_lu_update<NB><<<n, 256, n * sizeof(double), s>>>(n, j0, a, piv, info);
        if (hipError_t e = hipGetLastError(); e != hipSuccess) return e;
    }
    return hipSuccess;
}

__global__ void k_clear_int(int *p) { *p = 0; }

}  // namespace

hipError_t lu_factor_device(int n, double *a, int *piv, int *info, hipStream_t s) {
    if (n < 1 || n > kLuDeviceMax) return hipErrorInvalidValue;
    k_clear_int<<<1, 1, 0, s>>>(info);
    if (n <= 1024) return factor<1, 16>(n, a, piv, info, s);
    if (n <= 2048) return factor<2, 16>(n, a, piv, info, s);
    return factor<4, 8>(n, a, piv, info, s);
}

void lu_substitute(int n, const double *a, const int *piv, double *x) {
    for (int j = 0; j < n; ++j) {
        const double *c = a + (size_t)j * n;
        double t = x[j];
        for (int i = 0; i < j; ++i) t -= c[i] * x[i];
        x[j] = t / c[j];
    }
    for (int j = n - 1; j >= 0; --j) {
        const double *c = a + (size_t)j * n;
        double t = x[j];
        for (int i = j + 1; i < n; ++i) t -= c[i] * x[i];
        x[j] = t;
    }
    for (int j = n - 1; j >= 0; --j)
        if (piv[j] != j) {
            const double t = x[j];
            x[j] = x[piv[j]];
            x[piv[j]] = t;
        }
}

}  // namespace lumagpu
