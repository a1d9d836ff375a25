// multi2d_kernels.hpp -- several AA steps per launch on a small D2Q9 grid.
//
// A step of a 256 x 256 grid is a few microseconds of work and as much again of launch and drain,
// with every step's populations going through the caches.  Here a block loads a window of
// 32 x 32 cells into LDS, takes H steps there and writes the (32 - 2H)^2 tile in the middle:
// step s is right on the window without its outermost s cells, so the H steps' results are right
// on the tile.  The AA pattern keeps one LDS copy: a site reads and writes the same slots and no
// other site touches them in that step, so one barrier per step is all the synchronisation.
// H is even and the launch starts and ends in the post-local layout, where a tile's state is
// its own cells' slots; the tile goes to a second array, since other blocks still read the
// cells around it.
//
// The window's sites away from the tile are computed by several blocks: (32 / (32 - 2H))^2 times
// the work, 4 for H = 8.  plan_multi2d weighs that against the launch.  Per step on the 256 x 256
// cavity, one step per launch -> here: 9.9 -> 2.9 us FP32, 11.1 -> 4.2 us FP64; 1.9 us (FP32) on
// a periodic box of that size, where no wave has the lid's condition to compute after its
// fluid sites.
//
// Every site update is masked_site's code, and populations rest in LDS in the storage type, so
// the result is that of H single steps bit for bit, slots of solid and forced-equilibrium
// cells included.
#pragma once

#include "aa_kernels.hpp"

namespace lumagpu {

constexpr int kMultiWindow = 32;

template <class P>
__global__ __launch_bounds__(kMultiWindow *kMultiWindow) void k_multi2d(StepArgs a, void *dst_v, int H, int store) {
    using L = Lattice<9>;
    using S = typename P::S;
    using T = typename P::T;
    using M = typename P::M;
    constexpr int Q = 9, W = kMultiWindow, C = W * W;
    __shared__ S sh[Q * C];
    const int t = threadIdx.x, lx = t % W, ly = t / W;
    const int tile = W - 2 * H;
    // the window wraps as often as a grid smaller than it needs
    const int tx = blockIdx.x * tile + lx - H, ty0 = blockIdx.y * tile + ly - H;
    const int x = (tx + W * a.nx) % a.nx, y = (ty0 + W * a.ny) % a.ny;
    const size_t cell = (size_t)x + (size_t)a.nx * y;
    const S *__restrict__ src = static_cast<const S *>(a.f);
    S *__restrict__ dst = static_cast<S *>(dst_v);
#pragma unroll
    for (int v = 0; v < Q; ++v) sh[v * C + t] = src[(size_t)v * a.ps + cell];
    // an unlabelled grid is all fluid
    const uint64_t w = a.link ? a.link[cell] : (uint64_t)kFluid << kLinkType;
    const unsigned fl = a.flags ? a.flags[cell] : 0u;
    const int ty = (int)(w >> kLinkType) & 15;
    const bool stepped = ty == kFluid || (ty == kVelocity && a.regularised);
    M Fv[3] = {M(0.0), M(0.0), M(0.0)};
    const M *F = nullptr;
    if (fl & kForcedBit) {
        const M *fx = mv<M>(a.force);
        Fv[0] = fx[cell];
        Fv[1] = fx[a.ncell + cell];
        F = Fv;
    }
    // forced-equilibrium sources keep their value from step to step
    const bool feq_any = ((w >> kLinkVel) & kLinkMask) != 0;
    const int edge = min(min(lx, W - 1 - lx), min(ly, W - 1 - ly));
    const bool out = edge >= H && tx < a.nx && ty0 < a.ny;   // a cell of this block's tile
    __syncthreads();

    auto step = [&](auto odd_c, bool last) {
        constexpr bool ODD = decltype(odd_c)::value;
        T fin[Q], fout[Q];
        static_for<Q>([&](auto vc) {
            constexpr int v = decltype(vc)::value;
            if constexpr (!ODD || v == Q - 1) {
                fin[v] = static_cast<T>(sh[v * C + t]);
            } else {
                const int reg = L::opp(v) * C + t - L::c(v, 0) - W * L::c(v, 1);
                fin[v] = static_cast<T>(sh[((w >> v) & 1) ? v * C + t : reg]);
            }
        });
        if (feq_any)
            static_for<Q - 1>([&](auto vc) {
                constexpr int v = decltype(vc)::value;
                if ((w >> (kLinkVel + v)) & 1) {
                    const int js = y - L::c(v, 1) < 0 ? a.ny - 1 : (y - L::c(v, 1) >= a.ny ? 0 : y - L::c(v, 1));
                    const double us[3] = {a.uin[js], a.uin[a.ny + js], 0.0};
                    fin[v] = feq_store<Q, P>(v, a.rho_in, us, a);
                }
            });
        M rho, u[3];
        if (ty == kVelocity) {
            velocity_collide<Q, P>(a, fl, y, fin, F, fout, rho, u);
        } else {
            const auto col = make_collider<Q, P>(fin, F, a, rho, u);
            collide_pairs<Q>(col, fin, fout);
        }
        if (last && store && out) store_macro<2>(a, cell, rho, u);
        static_for<Q>([&](auto vc) {
            constexpr int v = decltype(vc)::value;
            int to = L::opp(v) * C + t;
            if constexpr (ODD && v < Q - 1)
                if (!((w >> L::opp(v)) & 1)) to = v * C + t + L::c(v, 0) + W * L::c(v, 1);
            sh[to] = static_cast<S>(fout[v]);
        });
    };
    for (int s = 1; s < H; s += 2) {
        if (stepped && edge >= s) step(std::true_type{}, false);
        __syncthreads();
        if (stepped && edge >= s + 1) step(std::false_type{}, s + 1 == H);
        __syncthreads();
    }
    if (out) {
#pragma unroll
        for (int v = 0; v < Q; ++v) dst[(size_t)v * a.ps + cell] = sh[v * C + t];
    }
}

// blocks of a launch of H steps
inline long multi2d_blocks(int nx, int ny, int H) {
    const int tile = kMultiWindow - 2 * H;
    return (long)((nx + tile - 1) / tile) * ((ny + tile - 1) / tile);
}

// Steps per launch for up to n (even) steps: the H whose launch, rounds of blocks over the
// 256 CUs and window steps cost least per step.  The two constants lie between boxes and lids, whose
// sites run after the fluid of their wave: a launch of H = 8 on 256 x 256 (one block per CU) takes 14.7 us
// FP32 on a box and 23.5 with a lid (17.1 by the constants), 27.4 and 33.7 FP64 (31.5); of H = 12 on
// 48 x 48 14.6 and 28.7 us FP32 (21.9), 28 and 39 FP64 (43.5).
inline int plan_multi2d(int nx, int ny, int n, bool fp64) {
    const double launch_us = 7.5, step_us = fp64 ? 3.0 : 1.2;
    int best = 0;
    double cost = 0.0;
    for (int H = 2; H <= 12 && H <= n; H += 2) {
        const double c = (launch_us + H * step_us * ((multi2d_blocks(nx, ny, H) + 255) / 256)) / H;
        if (best == 0 || c < cost) {
            best = H;
            cost = c;
        }
    }
    return best;
}

template <class P>
hipError_t launch_multi2d_p(const StepArgs &a, void *dst, int H, int store, hipStream_t s) {
    if (H < 2 || H > 14 || (H & 1)) return hipErrorInvalidValue;
    const int tile = kMultiWindow - 2 * H;
    k_multi2d<P><<<dim3((a.nx + tile - 1) / tile, (a.ny + tile - 1) / tile), kMultiWindow * kMultiWindow, 0, s>>>(
        a, dst, H, store);
    return hipGetLastError();
}

}  // namespace lumagpu
