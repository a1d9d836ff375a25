// adjoint_kernels.hpp -- discrete adjoint of one fused stream / IB / collide step.
//
// Forward step t (post-collision f of step t-1  ->  post-collision f' of step t):
//   g_v(x)  = stream of f (periodic pull, halfway bounce-back, ExtrapolateRight source,
//             forced-equilibrium velocity source), _LBM_stream_opt :206-297;
//   IB      : rho_s, j_s at support sites from g; (rho u)_m = sum_s j_s d_ms, rho_m = sum_s
//             rho_s d_ms; F_m = 2((rho u)_m - rho_m U_m); F_s = -sum_m d_ms F_m eps_m ds_m vd_m
//             (ObjectManager_ops_ibm.cpp:498-689);
//   collide : rho = sum g, u = (sum c g + B F/2)/rho, f'_v = g_v + omega (feq_v - g_v) + Guo_v
//             (:765-990; B adds F_z to the x momentum under the :833 quirk).
// Objective: J = (1/T) sum_t dir . sum_m F_m eps_m ds_m vd_m (the body force LUMA writes to
// Body_<id>_LD, ObjectManager_ops_io.cpp:98-121, averaged over the T steps).
//
// The adjoint runs the step backwards: reverse streaming of the later step (adj_lam: every
// population adjoint is gathered from the site that pulled it) and the collision's transposed
// Jacobian per site in one kernel (k_adj_collide; regularised faces in k_adj_faces, edges and
// corners in k_adj_edges), then spread and interpolation swapped (the spread's adjoint gathers the
// site force adjoint to the markers, k_adj_ibm_marker; the interpolation's adjoint spreads the
// marker adjoint to the sites through the same per-site gather lists, k_adj_ibm_site).  Only
// gbar = dJ/dg goes through memory, in two arrays that trade places; lam = dJ/df is written once,
// after the first step (k_adj_stream).  Adjoint arrays are plain [v][cell] (no AA layout), their
// planes padded like the populations'.
#pragma once

#include "aa_kernels.hpp"
#include "ibm_kernels.hpp"

namespace lumagpu {

template <class T>
struct AdjArgs {
    const T *gin;    // [Q][ps] adjoint of the populations the later step streamed
    T *gbar;         // [Q][ps] adjoint of the streamed populations
    size_t ps;       // plane stride of both
    double ramp_feq; // StepArgs::ramp_feq of the later step (its velocity sources)
    int ramp_on;
    double *fbar;    // [3][ncell] adjoint of the body-force field (flagged sites)
    // per-block partial sums: omega [0, nblk_all), the later step's inlet scale [nblk_all, 2 nblk_all);
    // nblk blocks over the grid, then those of the site list
    double *part;
    int nblk, nblk_all;
    int outlet;      // the grid has ExtrapolateRight sites
};

__device__ __forceinline__ int block_linear() {
    return blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z);
}

// deterministic block sum (blocks of 64 to 1024 threads, a multiple of 64): a fixed tree over
// each wave's lanes, then the waves' sums in wave order; every thread gets the sum
__device__ __forceinline__ double block_sum(double v) {
    __shared__ double sh[16];
    for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
    __syncthreads();
    double s = 0.0;
    for (int w = 0; w < (int)(blockDim.x >> 6); ++w) s += sh[w];
    __syncthreads();
    return s;
}

// A regularised velocity face site (not an edge or corner) of a grid stepped with
// regularised boundaries; with the edge and corner sites and the pressure faces, every
// regularised boundary site (each streams like a fluid site and is pulled like one).
__device__ __forceinline__ bool regularised_face_site(const StepArgs &a, unsigned fl) {
    return a.regularised && (fl & kTypeMask) == kVelocity && ((fl >> kNormalShift) & 7) != kNormalEdge;
}
__device__ __forceinline__ bool regularised_boundary_site(const StepArgs &a, unsigned fl) {
    const int ty = fl & kTypeMask;
    return a.regularised && (ty == kVelocity || ty == kPressure);
}

// Reverse streaming at a fluid or regularised boundary site: lam_w(x) gathers the adjoint of
// every streamed population that read f_w(x) -- the pull by x + c_w (a fluid or regularised
// boundary site), the bounce-back at x itself when x + c_w is solid, and the pull through an
// ExtrapolateRight source two cells to the right.  pl: a plain site (every neighbour fluid) is
// pulled by its neighbours alone, no neighbour flag is read.  fx: the flag byte two cells to the
// right (of the site itself at the grid's last two columns).
template <int Q, class T>
__device__ __forceinline__ void adj_lam(const StepArgs &a, const AdjArgs<T> &b, int x, int y, int z, size_t cell,
                                        const Nbr &nb, bool pl, unsigned fx, T *acc) {
    using L = Lattice<Q>;
    const int nx = a.nx, ny = a.ny;
    if (pl) {
        static_for<Q>([&](auto wc) {
            constexpr int w = decltype(wc)::value;
            acc[w] = b.gin[(size_t)w * b.ps + nb.at(L::c(w, 0), L::c(w, 1), L::c(w, 2), nx, ny)];
        });
    } else {
#pragma unroll
        for (int w = 0; w < Q; ++w) {
            const size_t yn = nb.at(L::c(w, 0), L::c(w, 1), L::c(w, 2), nx, ny);
            const unsigned fn = a.flags[yn];
            const int tn = fn & kTypeMask;
            const bool pulled = tn == kFluid || regularised_boundary_site(a, fn);
            // one load at a selected address: a load in each branch took the kernel from 138 to 256 registers
            const T t = b.gin[tn == kSolid ? (size_t)L::opp(w) * b.ps + cell : (size_t)w * b.ps + yn];
            acc[w] = (pulled || tn == kSolid) ? t : T(0);
        }
    }
    if (x + 2 < nx && (fx & kTypeMask) == kExtrapRight) {
        Nbr ns;
        ns.init(x + 2, y, z, nx, ny, a.nz);
#pragma unroll
        for (int w = 0; w < Q; ++w) {
            const size_t yp = ns.at(L::c(w, 0), L::c(w, 1), L::c(w, 2), nx, ny);
            if ((a.flags[yp] & kTypeMask) == kFluid) acc[w] += b.gin[(size_t)w * b.ps + yp];
        }
    }
}
// the same at a listed boundary site
template <int Q, class T>
__device__ __forceinline__ void adj_lam_site(const StepArgs &a, const AdjArgs<T> &b, int x, int y, int z, size_t cell,
                                             const Nbr &nb, double *lam) {
    T acc[Q];
    adj_lam<Q, T>(a, b, x, y, z, cell, nb, false, a.flags[x + 2 < a.nx ? cell + 2 : cell], acc);
#pragma unroll
    for (int v = 0; v < Q; ++v) lam[v] = double(acc[v]);
}

// The later step's derivative with respect to a scale s of the inlet profile (u_in -> s u_in) at a
// site that pulls from forced-equilibrium velocity sources: gbar_v d feq_v(rho_in, s u_in) / ds at
// s = 1.  A rolled loop over v (uniform, so its velocities come from scalar loads): few sites need it,
// and unrolled its FP64 terms would hold registers that the whole kernel pays for.
template <int Q, class T>
__device__ __forceinline__ double adj_inlet(const StepArgs &a, const AdjArgs<T> &b, int x, int y, int z, size_t cell) {
    using L = Lattice<Q>;
    const int nx = a.nx, ny = a.ny;
    double in_site = 0.0;
#pragma unroll 1
    for (int v = 0; v < Q; ++v) {
        const int c0 = L::c(v, 0), c1 = L::c(v, 1), c2 = L::c(v, 2);
        int sx = x - c0, sy = y - c1, sz = z - c2;
        sx = sx < 0 ? nx - 1 : (sx >= nx ? 0 : sx);
        sy = sy < 0 ? ny - 1 : (sy >= ny ? 0 : sy);
        sz = sz < 0 ? a.nz - 1 : (sz >= a.nz ? 0 : sz);
        if ((a.flags[cell_of(sx, sy, sz, nx, ny)] & kTypeMask) != kVelocity) continue;
        // the source's velocity as the step's gather_in takes it (with a velocity ramp, the ramped
        // profile of the pulling site's row)
        const int js = b.ramp_on ? y : sy;
        const double rf = b.ramp_feq;
        const double us[3] = {a.uin[js] * rf, a.uin[ny + js] * rf, (L::D == 3) ? a.uin[2 * ny + js] * rf : 0.0};
        const double cu = c0 * us[0] + c1 * us[1] + c2 * us[2];
        // d feq_v / du . u_in = w rho_in (3 c.u + 9 (c.u)^2 - 3 u.u)
        const double usq = us[0] * us[0] + us[1] * us[1] + us[2] * us[2];
        const double d = L::w(v) * a.rho_in * (3.0 * cu + 9.0 * cu * cu - 3.0 * usq);
        in_site += double(b.gin[(size_t)v * b.ps + cell]) * d;
    }
    return in_site;
}

// One forward-mode (Dual) pass of the transposed Jacobian of a regularised velocity face site's
// update (regularised_face, :313-510, then BGK, :765-790) at its streamed populations g
// (absolute): lam . d f' / d p for seed s, p = population s for s < Q, omega for s = Q and the
// inlet profile scale (u_in -> p u_in at p = 1) for s = Q + 1.  The site carries no body force
// (the adjoint refuses IB supports on velocity sites).
template <int Q>
__device__ double adj_regularised_face(const StepArgs &a, unsigned fl, int y, const double *g, const double *lam,
                                       int s) {
    using L = Lattice<Q>;
    const int ncode = (fl >> kNormalShift) & 7;
    const double r = a.ramp_reg;
    const double vin0[3] = {a.uin[y] * r, a.uin[a.ny + y] * r, (L::D == 3) ? a.uin[2 * a.ny + y] * r : 0.0};
    Dual ga[Q];
#pragma unroll
    for (int v = 0; v < Q; ++v) ga[v] = Dual(g[v], v == s ? 1.0 : 0.0);
    Dual vin[3];
    for (int d = 0; d < 3; ++d) vin[d] = Dual(vin0[d], s == Q + 1 ? vin0[d] : 0.0);
    Dual rr, uu[3];
    regularised_face<Q, Dual>(ga, ncode, vin, Dual(a.rho_in), Dual(a.cs2), Dual(a.den2), rr, uu);
    const CollideExact<Q, Dual> col{rr, {uu[0], uu[1], uu[2]}, Dual(a.omega, s == Q ? 1.0 : 0.0),
                                    Dual(a.cs2), Dual(a.den2), nullptr};
    double acc = 0.0;
#pragma unroll
    for (int w = 0; w < Q; ++w) acc += lam[w] * col(w, ga[w]).d;
    return acc;
}

// Which sites a launch of k_adj_collide takes.  Small grids: all, in one launch.  Large ones as the
// forward step: the plain sites by bitmap, without a flag, and a list of the others; rows whose
// first and last sites are not plain otherwise send most waves through both paths one after the
// other.  The column that feeds an outlet (x = nx - 3) is listed too: its populations are pulled
// twice.
enum AdjMode : int { kAdjAll = 0, kAdjPlain = 1, kAdjList = 2 };

// One fluid site: reverse streaming of the later step (adj_lam) and the transposed collision Jacobian:
// gbar = (d f'/d g)^T lam, fbar = (d f'/d F)^T lam at a forced site; returns the omega derivative
// sum_v lam_v d f'_v / d omega.
template <int Q, class P, bool ODD, int MODE>
__device__ __forceinline__ double adj_site(const StepArgs &a, const AdjArgs<typename P::T> &b, int x, int y, int z,
                                           size_t cell, bool pl, unsigned fx, unsigned fl, double &in_site) {
    using L = Lattice<Q>;
    using T = typename P::T;
    Nbr nb;
    nb.init(x, y, z, a.nx, a.ny, a.nz);
    T lam[Q];
    adj_lam<Q, T>(a, b, x, y, z, cell, nb, pl, fx, lam);
    if constexpr (MODE != kAdjPlain)
        if (!a.regularised && !pl) in_site = adj_inlet<Q, T>(a, b, x, y, z, cell);
    T fin[Q];
    if (pl) gather_plain<Q, P, ODD>(a, cell, nb, fin);
    else if constexpr (MODE != kAdjPlain) gather_in<Q, P, ODD>(a, x, y, z, cell, nb, kFluid, fin);
    T g[Q];
#pragma unroll
    for (int v = 0; v < Q; ++v) g[v] = P::kShift ? fin[v] + T(L::w(v) * a.rho0) : fin[v];
    const bool forced = (fl & kForcedBit) != 0;
    T F[3] = {T(0), T(0), T(0)};
    if (forced) {
        F[0] = T(a.force[cell]);
        F[1] = T(a.force[a.ncell + cell]);
        if constexpr (L::D == 3) F[2] = T(a.force[2 * a.ncell + cell]);
    }
    T rho = T(0), j[3] = {T(0), T(0), T(0)};
#pragma unroll
    for (int v = 0; v < Q; ++v) {
        rho += g[v];
        j[0] += T(L::c(v, 0)) * g[v];
        j[1] += T(L::c(v, 1)) * g[v];
        j[2] += T(L::c(v, 2)) * g[v];
    }
    j[0] += T(0.5) * F[0];
    j[1] += T(0.5) * F[1];
    if constexpr (L::D == 3) {
        if (a.fz_compat) j[0] += T(0.5) * F[2];
        else j[2] += T(0.5) * F[2];
    }
    const T u[3] = {j[0] / rho, j[1] / rho, j[2] / rho};
    const T usq = u[0] * u[0] + u[1] * u[1] + u[2] * u[2];
    const T uF = u[0] * F[0] + u[1] * F[1] + u[2] * F[2];
    const T om = T(a.omega), guo = T(1) - T(0.5) * om;
    T S0 = T(0), Ua[3] = {T(0), T(0), T(0)}, Ga[3] = {T(0), T(0), T(0)}, Fb[3] = {T(0), T(0), T(0)};
    T omb = T(0);
#pragma unroll
    for (int v = 0; v < Q; ++v) {
        const T cx = T(L::c(v, 0)), cy = T(L::c(v, 1)), cz = T(L::c(v, 2)), w = T(L::w(v));
        const T cu = cx * u[0] + cy * u[1] + cz * u[2];
        const T cF = cx * F[0] + cy * F[1] + cz * F[2];
        const T e = T(1) + T(3) * cu + T(4.5) * cu * cu - T(1.5) * usq;
        const T lw = lam[v] * w;
        S0 += lw * e;
        Ua[0] += lw * (T(3) * cx + T(9) * cu * cx - T(3) * u[0]);
        Ua[1] += lw * (T(3) * cy + T(9) * cu * cy - T(3) * u[1]);
        Ua[2] += lw * (T(3) * cz + T(9) * cu * cz - T(3) * u[2]);
        T dom = w * rho * e - g[v];
        if (forced) {
            Ga[0] += lw * (T(-3) * F[0] + T(9) * cx * cF);
            Ga[1] += lw * (T(-3) * F[1] + T(9) * cy * cF);
            Ga[2] += lw * (T(-3) * F[2] + T(9) * cz * cF);
            Fb[0] += lw * (T(3) * (cx - u[0]) + T(9) * cu * cx);
            Fb[1] += lw * (T(3) * (cy - u[1]) + T(9) * cu * cy);
            Fb[2] += lw * (T(3) * (cz - u[2]) + T(9) * cu * cz);
            dom -= T(0.5) * w * (T(3) * (cF - uF) + T(9) * cu * cF);
        }
        omb += lam[v] * dom;
    }
    T ub[3], jb[3];
    for (int d = 0; d < 3; ++d) {
        ub[d] = om * rho * Ua[d] + guo * Ga[d];
        jb[d] = ub[d] / rho;
    }
    if constexpr (L::D == 2) jb[2] = T(0);
    const T rb = om * S0 - (ub[0] * u[0] + ub[1] * u[1] + ub[2] * u[2]) / rho;
#pragma unroll
    for (int v = 0; v < Q; ++v)
        b.gbar[(size_t)v * b.ps + cell] = (T(1) - om) * lam[v] + rb + T(L::c(v, 0)) * jb[0] +
                                            T(L::c(v, 1)) * jb[1] + T(L::c(v, 2)) * jb[2];
    if (forced) {
        double Fbar[3] = {double(guo * Fb[0] + T(0.5) * jb[0]), double(guo * Fb[1] + T(0.5) * jb[1]),
                          double(guo * Fb[2])};
        if constexpr (L::D == 3) Fbar[2] += double(T(0.5) * (a.fz_compat ? jb[0] : jb[2]));
        for (int d = 0; d < L::D; ++d) b.fbar[(size_t)d * a.ncell + cell] = Fbar[d];
    }
    return double(omb);
}

// Every fluid site (see AdjMode), one pass: f and gin read, gbar written, 3 Q values per cell; with
// the streaming in a kernel of its own it was 5 Q, lam written and read again.  192 x 80 x 80 FP32
// per reversed step: 133 + 59 us in two kernels over all sites, 52 + 45 us (plain sites, list) here.  Regularised
// velocity faces run in k_adj_faces: their forward-mode passes take several times this path's
// registers, and one kernel holding both ran at one wave per SIMD with spills.
// FP64 D3Q19: at most 256 VGPRs, two waves per SIMD (it needs 286 for one: 1.83 ms against
// 1.21 ms with 28 B of spills on 6.3 M cells)
template <int Q, class P, bool ODD, int MODE>
__global__ __launch_bounds__(256, (sizeof(typename P::T) == 8 && Q == 19) ? 2 : 1) void k_adj_collide(
    StepArgs a, AdjArgs<typename P::T> b, const int *cells, int n) {
    double om_site = 0.0, in_site = 0.0;
    if constexpr (MODE == kAdjList) {
        const int i = blockIdx.x * blockDim.x + threadIdx.x;
        if (i < n) {
            const size_t cell = (size_t)cells[i];
            int x, y, z;
            cell_coords(a, (uint32_t)cell, x, y, z);
            const bool pl = (a.plain[cell >> 5] >> (cell & 31)) & 1u;
            const unsigned fx = a.flags[x + 2 < a.nx ? cell + 2 : cell];
            om_site = adj_site<Q, P, ODD, MODE>(a, b, x, y, z, cell, pl, fx, a.flags[cell], in_site);
        }
    } else {
        const int x = blockIdx.x * blockDim.x + threadIdx.x;
        const int y = blockIdx.y, z = blockIdx.z;
        if (x < a.nx) {
            const size_t cell = cell_of(x, y, z, a.nx, a.ny);
            // the flag bytes and the plain-site bit in one round trip (plain sites are fluid sites
            // whose pulls read no neighbour flag)
            const bool pl = (a.plain[cell >> 5] >> (cell & 31)) & 1u;   // never null in the adjoint
            const unsigned fl = a.flags[cell];
            if constexpr (MODE == kAdjPlain) {
                // the flag byte of the cell itself is no outlet's
                if (pl && !(b.outlet && x == a.nx - 3))
                    om_site = adj_site<Q, P, ODD, MODE>(a, b, x, y, z, cell, true, kFluid, fl, in_site);
            } else {
                const unsigned fx = a.flags[x + 2 < a.nx ? cell + 2 : cell];
                if (pl || (fl & kTypeMask) == kFluid)   // a plain site is a fluid site
                    om_site = adj_site<Q, P, ODD, MODE>(a, b, x, y, z, cell, pl, fx, fl, in_site);
            }
        }
    }
    const double s = block_sum(om_site), si = MODE == kAdjPlain ? 0.0 : block_sum(in_site);
    if (threadIdx.x == 0) {
        const int blk = block_linear() + (MODE == kAdjList ? b.nblk : 0);
        b.part[blk] = s;
        b.part[b.nblk_all + blk] = si;
    }
}

// Regularised velocity face sites (cells[i]): gbar from adj_regularised_face at the site's
// streamed populations; the omega and inlet-scale derivatives per site in fpart[i] and
// fpart[n + i].  One thread per (site, seed), the sites of one seed side by side: a face is a
// few dozen to a few thousand sites, and the Q + 2 passes of a site one after another made one
// wave's chain the kernel's whole time (58 sites of a 220 x 60 FP64 channel: 113 -> 14 us).
template <int Q, class P, bool ODD>
__global__ __launch_bounds__(64) void k_adj_faces(StepArgs a, AdjArgs<typename P::T> b, const int *cells, int n,
                                                  double *fpart) {
    using L = Lattice<Q>;
    using T = typename P::T;
    const int i = blockIdx.x * blockDim.x + threadIdx.x, s = blockIdx.y;
    if (i >= n) return;
    const size_t cell = (size_t)cells[i];
    const int nx = a.nx, ny = a.ny;
    const int x = (int)(cell % nx), y = (int)((cell / nx) % ny), z = (int)(cell / ((size_t)nx * ny));
    Nbr nb;
    nb.init(x, y, z, nx, ny, a.nz);
    T fin[Q];
    gather_in<Q, P, ODD>(a, x, y, z, cell, nb, kVelocity, fin);
    double g[Q], lam[Q];
    adj_lam_site<Q, T>(a, b, x, y, z, cell, nb, lam);
#pragma unroll
    for (int v = 0; v < Q; ++v) g[v] = double(fin[v]) + (P::kShift ? L::w(v) * a.rho0 : 0.0);
    const double d = adj_regularised_face<Q>(a, a.flags[cell], y, g, lam, s);
    if (s < Q) b.gbar[(size_t)s * b.ps + cell] = T(d);
    else fpart[(s - Q) * n + i] = d;
}

// Sites that extrapolate from their two inward neighbours (k_edge_sites), one thread per (site,
// seed) as in k_adj_faces: edge and corner velocity sites (regularised_edge with the density
// 2 rho(x+n) - rho(x+2n) from the neighbours' sweep-1 values) and pressure faces
// (regularised_pressure with the tangential velocity 2 u(x+n) - u(x+2n)), then BGK.  The site's own gbar comes from forward-mode passes
// over its populations; the extrapolated quantities' adjoints (dbar[i], or tbar[3 i + d] for
// the velocity components) reach the neighbours' streamed populations through
// d rho / d g_v = 1 and d u_d / d g_v = (c_vd - u_d) / rho (k_adj_edge_nbrs); omega and
// inlet-scale derivatives per site in epart[i] and epart[n + i].
template <int Q, class P, bool ODD>
__global__ __launch_bounds__(64) void k_adj_edges(StepArgs a, EdgeArgs e, AdjArgs<typename P::T> b,
                                                  double *dbar, double *tbar, double *epart) {
    using L = Lattice<Q>;
    using T = typename P::T;
    const int i = blockIdx.x * blockDim.x + threadIdx.x, s = blockIdx.y;
    if (i >= e.n) return;
    const size_t cell = (size_t)e.cell[i];
    const int nx = a.nx, ny = a.ny;
    const int x = (int)(cell % nx), y = (int)((cell / nx) % ny), z = (int)(cell / ((size_t)nx * ny));
    const int pk = e.nrm[i];
    const int n[3] = {(pk & 3) - 1, ((pk >> 2) & 3) - 1, ((pk >> 4) & 3) - 1};
    Nbr nb;
    nb.init(x, y, z, nx, ny, a.nz);
    T fin[Q];
    gather_in<Q, P, ODD>(a, x, y, z, cell, nb, kVelocity, fin);
    double g[Q], lam[Q];
    adj_lam_site<Q, T>(a, b, x, y, z, cell, nb, lam);
#pragma unroll
    for (int v = 0; v < Q; ++v) g[v] = double(fin[v]) + (P::kShift ? L::w(v) * a.rho0 : 0.0);
    const double *er1 = e.erho + 8 * (size_t)i, *er2 = er1 + 4;
    const bool pressure = (a.flags[cell] & kTypeMask) == kPressure;
    const int ncode = (a.flags[cell] >> kNormalShift) & 7;
    const double dens0 = 2.0 * er1[0] - er2[0];
    const double vt0[3] = {2.0 * er1[1] - er2[1], 2.0 * er1[2] - er2[2], (L::D == 3) ? 2.0 * er1[3] - er2[3] : 0.0};
    const double r = a.ramp_reg;
    const double vin0[3] = {a.uin[y] * r, a.uin[ny + y] * r, (L::D == 3) ? a.uin[2 * ny + y] * r : 0.0};
    // seeds: populations 0..Q-1, then omega, then the extrapolated density and the inlet scale
    // (velocity edges, s = Q + 3 idle) or the three extrapolated velocity components (pressure
    // faces)
    Dual fa[Q];
#pragma unroll
    for (int v = 0; v < Q; ++v) fa[v] = Dual(g[v], v == s ? 1.0 : 0.0);
    Dual rr, uu[3], fout[Q];
    if (pressure) {
        Dual vt[3];
        for (int d = 0; d < 3; ++d) vt[d] = Dual(vt0[d], s == Q + 1 + d ? 1.0 : 0.0);
        regularised_pressure<Q, Dual>(fa, ncode, vt, Dual(a.rho_p), Dual(a.cs2), Dual(a.den2), rr, uu);
    } else {
        Dual vin[3];
        for (int d = 0; d < 3; ++d) vin[d] = Dual(vin0[d], s == Q + 2 ? vin0[d] : 0.0);
        regularised_edge<Q, Dual>(fa, n, vin, Dual(dens0, s == Q + 1 ? 1.0 : 0.0), Dual(a.cs2), Dual(a.den2), rr, uu);
    }
    collide_exact<Q, Dual>(fa, rr, uu, static_cast<const Dual *>(nullptr), Dual(a.omega, s == Q ? 1.0 : 0.0),
                           Dual(a.cs2), Dual(a.den2), fout);
    double acc = 0.0;
#pragma unroll
    for (int w = 0; w < Q; ++w) acc += lam[w] * fout[w].d;
    // every output of the site has one seed that writes it; the other kind's are zero
    if (s < Q) b.gbar[(size_t)s * b.ps + cell] = T(acc);
    else if (s == Q) epart[i] = acc;
    else if (pressure) tbar[3 * (size_t)i + (s - Q - 1)] = acc;
    else if (s == Q + 1) dbar[i] = acc;
    else if (s == Q + 2) epart[e.n + i] = acc;
    if (pressure && s == Q) dbar[i] = epart[e.n + i] = 0.0;
    if (!pressure && s == Q)
        for (int d = 0; d < 3; ++d) tbar[3 * (size_t)i + d] = 0.0;
}

// The extrapolation's reach into the neighbours: gbar_v(x) += sum over the sites that
// extrapolate from x of coef * (dbar + sum_d tbar_d (c_vd - u_d(x)) / rho(x)) (coef 2 for the
// neighbour x + n, -1 for x + 2n; rho, u the neighbour's sweep-1 values in erho); one thread per
// neighbour cell, its entries in a fixed order (no atomics).
template <int Q, class T>
__global__ void k_adj_edge_nbrs(int nn, const int *ncell, const int *ptr, const int *ent, const double *dbar,
                                const double *tbar, const double *erho, size_t ps, T *gbar) {
    using L = Lattice<Q>;
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= nn) return;
    double s[Q];
    for (int v = 0; v < Q; ++v) s[v] = 0.0;
    for (int j = ptr[k]; j < ptr[k + 1]; ++j) {
        const int code = ent[j];   // 2 * site + (0: x + n, 1: x + 2n)
        const int i = code >> 1;
        const double coef = (code & 1) ? -1.0 : 2.0;
        const double *er = erho + 4 * (size_t)code;   // this neighbour's rho, u
        for (int v = 0; v < Q; ++v) {
            double t = dbar[i];
            for (int d = 0; d < L::D; ++d) t += tbar[3 * (size_t)i + d] * (L::c(v, d) - er[1 + d]) / er[0];
            s[v] += coef * t;
        }
    }
    const size_t cell = (size_t)ncell[k];
    for (int v = 0; v < Q; ++v) gbar[(size_t)v * ps + cell] += T(s[v]);
}

// Reverse streaming alone, after the first step has been reversed: lam = dJ/df of the initial
// populations (null: only that step's inlet derivative, part[nblk_all + block]).
template <int Q, class P>
__global__ __launch_bounds__(256) void k_adj_stream(StepArgs a, AdjArgs<typename P::T> b, typename P::T *out) {
    using T = typename P::T;
    const int x = blockIdx.x * blockDim.x + threadIdx.x;
    const int y = blockIdx.y, z = blockIdx.z;
    double in_site = 0.0;
    if (x < a.nx) {
        const size_t cell = cell_of(x, y, z, a.nx, a.ny);
        const bool pl = (a.plain[cell >> 5] >> (cell & 31)) & 1u;   // never null in the adjoint
        const unsigned fx = a.flags[x + 2 < a.nx ? cell + 2 : cell];
        const unsigned fl = a.flags[cell];
        T acc[Q];
        if (pl || (fl & kTypeMask) == kFluid || regularised_boundary_site(a, fl)) {
            Nbr nb;
            nb.init(x, y, z, a.nx, a.ny, a.nz);
            if (out) adj_lam<Q, T>(a, b, x, y, z, cell, nb, pl, fx, acc);
            if (!a.regularised && !pl) in_site = adj_inlet<Q, T>(a, b, x, y, z, cell);
        } else {
#pragma unroll
            for (int w = 0; w < Q; ++w) acc[w] = T(0);
        }
        if (out)
#pragma unroll
            for (int w = 0; w < Q; ++w) out[(size_t)w * b.ps + cell] = acc[w];
    }
    const double s = block_sum(in_site);
    if (threadIdx.x == 0) {
        b.part[block_linear()] = 0.0;
        b.part[b.nblk_all + block_linear()] = s;
    }
}

// IB adjoint, marker side: the spread's adjoint gathers the site force adjoint to the
// markers; the marker's force adjoint then feeds the interpolation's adjoint (mbar) and the
// derivatives with respect to the marker's epsilon, ds and position (through its delta
// weights), accumulated over the steps.
struct AdjIbm {
    const double *fbar;      // [3][ncell]
    const double *sddelta;   // [nm][S][3] d delta_ms / d x_m
    double *mbar;            // [nm][4]: adjoint of (rho u)_m, rho_m
    double *xbar, *epsbar, *dsbar;
    double dir[3];
    double invT;
};

// sum over a 64-lane wave, fixed tree, lane 0's result in every lane (so every lane goes on
// with the same value)
__device__ __forceinline__ double wave_sum_bcast(double v) {
    for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
    return __shfl(v, 0, 64);
}

// One 64-lane wave per marker (blocks of 256: four markers): the lanes take the marker's
// supports, and the two sums over them are wave reductions.
static __global__ __launch_bounds__(256) void k_adj_ibm_marker(IbmArgs ib, AdjIbm aj) {
    const int m = blockIdx.x * 4 + (int)(threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (m >= ib.nm) return;   // the whole wave
    const int D = ib.D;
    const double eps = ib.eps[m], ds = ib.ds[m];
    const double vd = (D == 3) ? ds : 1.0;
    const double wgt = eps * ds * vd;
    double Fs[3] = {0.0, 0.0, 0.0};
    for (int k = lane; k < ib.ns[m]; k += 64) {
        const size_t cell = (size_t)ib.scell[m * ib.S + k];
        const double dl = ib.sdelta[m * ib.S + k];
        for (int d = 0; d < D; ++d) Fs[d] += dl * aj.fbar[(size_t)d * ib.ncell + cell];
    }
    for (int d = 0; d < 3; ++d) Fs[d] = wave_sum_bcast(Fs[d]);
    double Fb[3], mom[3], FdotFs = 0.0, Fdir = 0.0, rb = 0.0;
    for (int d = 0; d < 3; ++d) {
        const double Fm = (d < D) ? ib.force[3 * m + d] : 0.0;
        Fb[d] = (d < D) ? (-wgt * Fs[d] + aj.dir[d] * wgt * aj.invT) : 0.0;
        mom[d] = 2.0 * Fb[d];
        rb += -2.0 * Fb[d] * ((d < D) ? ib.vel[3 * m + d] : 0.0);
        FdotFs += Fm * Fs[d];
        Fdir += Fm * aj.dir[d];
    }
    if (lane == 0) {
        for (int d = 0; d < 3; ++d) aj.mbar[4 * m + d] = mom[d];
        aj.mbar[4 * m + 3] = rb;
        aj.epsbar[m] += -ds * vd * FdotFs + Fdir * ds * vd * aj.invT;
        aj.dsbar[m] += ((D == 3) ? 2.0 * eps * ds : eps) * (-FdotFs + Fdir * aj.invT);
    }
    double xb[3] = {0.0, 0.0, 0.0};
    for (int k = lane; k < ib.ns[m]; k += 64) {
        const size_t cell = (size_t)ib.scell[m * ib.S + k];
        const double r = ib.rho[cell];
        double term = rb * r;
        for (int d = 0; d < D; ++d) {
            term += mom[d] * r * ib.u[(size_t)d * ib.ncell + cell];
            term -= wgt * ib.force[3 * m + d] * aj.fbar[(size_t)d * ib.ncell + cell];
        }
        for (int d = 0; d < D; ++d) xb[d] += aj.sddelta[((size_t)m * ib.S + k) * 3 + d] * term;
    }
    for (int d = 0; d < 3; ++d) xb[d] = wave_sum_bcast(xb[d]);
    if (lane == 0)
        for (int d = 0; d < D; ++d) aj.xbar[3 * m + d] += xb[d];
}

// IB adjoint, site side: the interpolation's adjoint spread through the per-site gather lists
// (no atomics): gbar_v(s) += rho_bar_s + c_v . j_bar_s at every fluid support site.
template <int Q, class T>
__global__ void k_adj_ibm_site(IbmArgs ib, const double *mbar, const uint8_t *flags, size_t ps, T *gbar) {
    using L = Lattice<Q>;
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= ib.nsites) return;
    const size_t cell = (size_t)ib.sites[s];
    if ((flags[cell] & kTypeMask) != kFluid) return;
    // every load of a step before its sums and stores: a chunk's entries, their weights and markers,
    // and the site's Q adjoints (which a store between them would put behind it)
    T old[Q];
#pragma unroll
    for (int v = 0; v < Q; ++v) old[v] = gbar[(size_t)v * ps + cell];
    constexpr int CH = 6;
    double jb[3] = {0.0, 0.0, 0.0}, rb = 0.0;
    const int e0 = ib.sptr[s], e1 = ib.sptr[s + 1];
    for (int eb = e0; eb < e1; eb += CH) {
        int code[CH];
        double dl[CH], mb[CH][4];
#pragma unroll
        for (int k = 0; k < CH; ++k) code[k] = ib.sent[eb + k < e1 ? eb + k : eb];
#pragma unroll
        for (int k = 0; k < CH; ++k) {
            dl[k] = ib.sdelta[code[k]];
            const double *m = mbar + 4 * (code[k] / ib.S);
#pragma unroll
            for (int d = 0; d < 4; ++d) mb[k][d] = m[d];
        }
#pragma unroll
        for (int k = 0; k < CH; ++k)
            if (eb + k < e1) {
#pragma unroll
                for (int d = 0; d < 3; ++d) jb[d] += dl[k] * mb[k][d];
                rb += dl[k] * mb[k][3];
            }
    }
#pragma unroll
    for (int v = 0; v < Q; ++v)
        gbar[(size_t)v * ps + cell] = old[v] + T(rb + L::c(v, 0) * jb[0] + L::c(v, 1) * jb[1] + L::c(v, 2) * jb[2]);
}

// ---- positions through epsilon and ds -------------------------------------------------------
// One system's markers (a body's, or with the universal system every marker's), index 0 .. n-1.
struct EpsSystem {
    int n, S, D;
    double dh;
    const double *pos, *dil, *area;   // [3n], [n], [n]
    const double *sxyz;               // [n][S][3] support positions
    const int *ns;                    // [n]
    const double *sdelta, *sddelta;   // [n][S] delta weights, [n][S][3] their gradients in the position
    const double *eps, *ds;           // [n]
};

// delta_kernel (ObjectManager_ops_ibm.cpp:255-272) and its derivative, as the host evaluates them
__device__ __forceinline__ double dev_delta(double radius, double dil) {
    const double m = ::fabs(radius) / dil;
    if (m > 1.5) return 0.0;
    if (m > 0.5) return (5.0 - (3.0 * m) - ::sqrt(-3.0 * ((1.0 - m) * (1.0 - m)) + 1.0)) / 6.0;
    return (1.0 + ::sqrt(1.0 - 3.0 * (m * m))) / 3.0;
}
__device__ __forceinline__ double dev_delta_deriv(double radius, double dil) {
    const double m = ::fabs(radius) / dil, sgn = radius < 0.0 ? -1.0 : 1.0;
    if (m > 1.5) return 0.0;
    double d;
    if (m > 0.5) {
        const double q = 1.0 - m;
        d = (-3.0 - 3.0 * q / ::sqrt(1.0 - 3.0 * q * q)) / 6.0;
    } else {
        d = -m / ::sqrt(1.0 - 3.0 * m * m);
    }
    return sgn * d / dil;
}
// far_apart: no support of one carries a delta weight of the other
__device__ __forceinline__ bool eps_far(const EpsSystem &e, int I, int J) {
    const double lim = (1.5 * e.dil[I] + 1.5 * e.dil[J] + 0.01) * e.dh;
    for (int a = 0; a < e.D; ++a)
        if (::fabs(e.pos[3 * J + a] - e.pos[3 * I + a]) > lim) return true;
    return false;
}
__device__ __forceinline__ double eps_delta_at(const EpsSystem &e, int J, const double *s) {
    double v = 1.0;
    for (int a = 0; a < e.D; ++a) v *= dev_delta((e.pos[3 * J + a] - s[a]) / e.dh, e.dil[J]);
    return v;
}

// A_IJ = ds_J sum_k delta_I(s_k) delta(x_J; s_k) area_I into a[J * n + I], one thread per pair, and
// how far the nonzero ones lie below and above the diagonal (I - J, J - I) and how many they are into shape[3]
static __global__ __launch_bounds__(256) void k_eps_matrix(EpsSystem e, double *a, int *shape) {
    const int I = blockIdx.x * blockDim.x + threadIdx.x, J = blockIdx.y;
    double v = 0.0;
    if (I < e.n) {
        double acc = 0.0;
        if (!eps_far(e, I, J))
            for (int k = 0; k < e.ns[I]; ++k)
                acc += e.sdelta[(size_t)I * e.S + k] * eps_delta_at(e, J, e.sxyz + ((size_t)I * e.S + k) * 3) * e.area[I];
        v = acc * e.ds[J];
        a[(size_t)J * e.n + I] = v;
    }
    // atomics of a wave that holds a nonzero: its first and last lane with one, and their number
    const uint64_t m = __ballot(v != 0.0);
    if (m && (threadIdx.x & 63) == 0) {
        const int lo = I + __ffsll((unsigned long long)m) - 1, hi = I + 63 - __clzll((long long)m);
        atomicMax(shape, hi - J);
        atomicMax(shape + 1, J - lo);
        atomicAdd(shape + 2, __popcll(m));
    }
}

// With A^T mu = epsbar: dJ/dA_IJ = -mu_I eps_J, and A's entries depend on both markers' positions and
// on ds_J.  One wave per marker m, its lanes the other markers: m as the row (its own weights'
// gradients) and as the column (its delta at the other's supports, and ds_m).
static __global__ __launch_bounds__(256) void k_eps_chain(EpsSystem e, const double *mu, double *xg, double *dsbar) {
    const int m = blockIdx.x * 4 + (int)(threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (m >= e.n) return;   // the whole wave
    double x[3] = {0.0, 0.0, 0.0}, dsb = 0.0;
    for (int q = lane; q < e.n; q += 64) {
        if (eps_far(e, m, q)) continue;
        const double row = -mu[m] * e.eps[q], col = -mu[q] * e.eps[m];
        if (row != 0.0)
            for (int k = 0; k < e.ns[m]; ++k) {
                const size_t mk = (size_t)m * e.S + k;
                const double t = row * e.ds[q] * eps_delta_at(e, q, e.sxyz + 3 * mk) * e.area[m];
                for (int a = 0; a < e.D; ++a) x[a] += t * e.sddelta[3 * mk + a];
            }
        if (col != 0.0) {
            double acc = 0.0;
            for (int k = 0; k < e.ns[q]; ++k) {
                const size_t qk = (size_t)q * e.S + k;
                double ph[3] = {1.0, 1.0, 1.0}, dph[3] = {0.0, 0.0, 0.0};
                for (int a = 0; a < e.D; ++a) {
                    const double r = (e.pos[3 * m + a] - e.sxyz[3 * qk + a]) / e.dh;
                    ph[a] = dev_delta(r, e.dil[m]);
                    dph[a] = dev_delta_deriv(r, e.dil[m]) / e.dh;
                }
                const double w = e.sdelta[qk] * e.area[q];
                acc += w * (ph[0] * ph[1] * ph[2]);
                const double t = col * e.ds[m] * w;
                x[0] += t * dph[0] * ph[1] * ph[2];
                x[1] += t * ph[0] * dph[1] * ph[2];
                x[2] += t * ph[0] * ph[1] * dph[2];
            }
            dsb += col * acc;
        }
    }
    for (int a = 0; a < 3; ++a) x[a] = wave_sum_bcast(x[a]);
    dsb = wave_sum_bcast(dsb);
    if (lane == 0) {
        for (int a = 0; a < 3; ++a) xg[3 * m + a] += x[a];
        dsbar[m] += dsb;
    }
}

// (1/T) dir . sum_m F_m eps_m ds_m vd_m added to acc[0]; one 64-lane wave, fixed order
static __global__ void k_adj_objective(IbmArgs ib, double dx, double dy, double dz, double invT, double *acc) {
    const int lane = threadIdx.x;
    const double dir[3] = {dx, dy, dz};
    double s = 0.0;
#pragma unroll 4
    for (int m = lane; m < ib.nm; m += 64) {
        const double w = ib.eps[m] * ((ib.D == 3) ? ib.ds[m] : 1.0) * ib.ds[m];
        double fd = 0.0;
        for (int d = 0; d < ib.D; ++d) fd += ib.force[3 * m + d] * dir[d];
        s += fd * w;
    }
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
    if (lane == 0) acc[0] += s * invT;
}

// A forced-equilibrium velocity site never steps, so the slots it would write keep what stepping in place
// leaves in them, and along the tape they are in the state before the last step.  After an even step: its own
// slots that its neighbours pushed to in the odd step before.  After an odd step: the slots of its
// neighbours that its pushes would fill, with what their even step wrote.
template <int Q, class S>
__global__ __launch_bounds__(256) void k_adj_carry(StepArgs a, const S *from, S *to, int odd) {
    using L = Lattice<Q>;
    const size_t cell = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (cell >= a.ncell || (a.flags[cell] & kTypeMask) != kVelocity) return;
    int x, y, z;
    cell_coords(a, (uint32_t)cell, x, y, z);
    Nbr nb;
    nb.init(x, y, z, a.nx, a.ny, a.nz);
    static_for<Q>([&](auto vc) {
        constexpr int v = decltype(vc)::value;
        const int s = odd ? 1 : -1;
        const size_t n = nb.at(s * L::c(v, 0), s * L::c(v, 1), s * L::c(v, 2), a.nx, a.ny);
        const int t = a.flags[n] & kTypeMask;
        const size_t slot = (size_t)v * a.ps + (odd ? n : cell);
        if (t == kFluid || t == kExtrapRight) to[slot] = from[slot];
    });
}

// The initial populations' adjoint in LUMA's layout f[v + Q*id], id = k + j*K + i*K*M, from
// the [v][cell] array: one thread per cell, reads coalesced, each thread's Q values contiguous
template <int Q, class T>
__global__ void k_adj_to_luma(const T *lam, size_t ps, size_t nc, int N, int M, int K, double *out) {
    const size_t cell = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (cell >= nc) return;
    const size_t i = cell % N, j = (cell / N) % M, k = cell / ((size_t)N * M);
    const size_t id = k + j * K + i * (size_t)K * M;
    for (int v = 0; v < Q; ++v) out[v + Q * id] = double(lam[(size_t)v * ps + cell]);
}

// Up to three pairs of partial sums in one launch, a block each: acc[0] += w0 * sum of part[0 .. n)
// (omega, w0 this step's d omega_t / d omega, 1 without a ramp), acc[1] += sum of part[n .. 2n)
// (inlet scale).  Each thread has four independent running sums (loads in flight), then a fixed
// tree: the order is fixed.
struct AdjSums {
    const double *part[3];
    int n[3];
    double *acc[3];
};
static __global__ __launch_bounds__(1024) void k_adj_sum_partials(AdjSums sums, double w0) {
    __shared__ double sh[1024];
    const double *part = sums.part[blockIdx.x];
    double *acc = sums.acc[blockIdx.x];
    const int n = sums.n[blockIdx.x];
    for (int k = 0; k < 2; ++k) {
        const double *p = part + (size_t)k * n;
        double s0 = 0.0, s1 = 0.0, s2 = 0.0, s3 = 0.0;
        int i = threadIdx.x;
        for (; i + 3 * 1024 < n; i += 4 * 1024) {
            s0 += p[i];
            s1 += p[i + 1024];
            s2 += p[i + 2 * 1024];
            s3 += p[i + 3 * 1024];
        }
        for (; i < n; i += 1024) s0 += p[i];
        sh[threadIdx.x] = (s0 + s1) + (s2 + s3);
        __syncthreads();
        for (int st = 512; st > 0; st >>= 1) {
            if ((int)threadIdx.x < st) sh[threadIdx.x] += sh[threadIdx.x + st];
            __syncthreads();
        }
        if (threadIdx.x == 0) acc[k] += k == 0 ? w0 * sh[0] : sh[0];
        __syncthreads();
    }
}

}  // namespace lumagpu
