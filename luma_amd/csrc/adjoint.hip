// adjoint.hip -- discrete adjoint of the time step with checkpointing (the differentiation
// form): gradients of the time-averaged IB body force with respect to the relaxation
// frequency, the inlet velocity scale, the marker positions and the initial populations.
//
// Forward: T steps of the ordinary step (lumagpu_step semantics), the population array copied
// to a checkpoint every K steps and the objective accumulated on the device.  Backward: for
// each segment, newest first, the segment's K states run from its checkpoint along a tape in
// HBM, each step writing its successor there (the last segment in the forward run already); then
// every step of the segment is reversed from its stored input state (the IB forces are recomputed
// from it, the outlet side buffer is on the tape, then the adjoint kernels of
// adjoint_kernels.hpp run).  The marker-position gradient adds the dependence of epsilon (the RKPM
// system A eps = 1, ObjectManager_ops_ibm.cpp:773-920) and of ds (nearest-marker spacing,
// :927-981) on the positions.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <string>
#include <vector>

#include "adjoint_kernels.hpp"
#include "ibm_system.hpp"
#include "launch.hpp"
#include "lu_device.hpp"

namespace lumagpu {
namespace {

// A device buffer of a run, from the blocks the grid keeps between runs: allocating and freeing some
// thirty arrays of the grid's size took 12 ms of a 100-step gradient on 1.2 M cells.  Everything on them
// is ordered by the grid's stream.  Contents are what the last user left.
struct DevBuf {
    lumagpu_grid *g = nullptr;
    void *p = nullptr;
    DevBuf() = default;
    DevBuf(const DevBuf &) = delete;
    DevBuf &operator=(const DevBuf &) = delete;
    ~DevBuf() {
        if (!p) return;
        for (auto &b : g->blocks)
            if (b.p == p) b.used = 0;
    }
    int alloc(lumagpu_grid *grid, size_t bytes) {
        g = grid;
        for (auto &b : g->blocks)
            if (!b.used && b.bytes >= bytes && b.bytes - bytes <= bytes / 8 + 4096) {
                b.used = 1;
                p = b.p;
                return 0;
            }
        if (dev_malloc(&p, bytes) != hipSuccess) {
            p = nullptr;
            return fail(LUMAGPU_ENOMEM, "adjoint buffer allocation failed (" + std::to_string(bytes) + " bytes)");
        }
        g->blocks.push_back({p, bytes, 1});
        return 0;
    }
};

// The grid keeps its blocks while there is room for them beside what other grids keep (api.hip).
void trim_blocks(lumagpu_grid *g) {
    if (!scratch_room(g, 0)) {
        for (auto &b : g->blocks) (void)hipFree(b.p);
        g->blocks.clear();
    }
    scratch_note(g);
}

// nlist < 0: every site in one launch; else the plain sites and a list of the others (see AdjMode)
constexpr int kAdjListBlock = 64;
// cells from which the reversed step splits its sites: below, one launch more costs as much as the waves
// that take both paths
constexpr size_t kAdjSplitMin = size_t(1) << 17;
template <int Q, class P>
void launch_adj_collide_q(const lumagpu_grid *g, const StepArgs &a, const AdjArgs<typename P::T> &b, const int *cells,
                          int nlist) {
    const dim3 bl = cell_block(a.nx), gr((a.nx + bl.x - 1) / bl.x, a.ny, a.nz);
    with_bool(g->parity == 0, [&](auto o) {
        constexpr bool ODD = decltype(o)::value;
        if (nlist < 0) {
            k_adj_collide<Q, P, ODD, kAdjAll><<<gr, bl, 0, g->stream>>>(a, b, nullptr, 0);
            return;
        }
        k_adj_collide<Q, P, ODD, kAdjPlain><<<gr, bl, 0, g->stream>>>(a, b, nullptr, 0);
        if (nlist > 0)
            k_adj_collide<Q, P, ODD, kAdjList>
                <<<(nlist + kAdjListBlock - 1) / kAdjListBlock, kAdjListBlock, 0, g->stream>>>(a, b, cells, nlist);
    });
}
template <class P>
hipError_t launch_adj_collide(const lumagpu_grid *g, const StepArgs &a, const AdjArgs<typename P::T> &b,
                              const int *cells, int nlist) {
    if (g->Q == 9) launch_adj_collide_q<9, P>(g, a, b, cells, nlist);
    else launch_adj_collide_q<19, P>(g, a, b, cells, nlist);
    return hipGetLastError();
}

template <class P>
hipError_t launch_adj_stream(const lumagpu_grid *g, const StepArgs &a, const AdjArgs<typename P::T> &b,
                             typename P::T *out) {
    const dim3 bl = cell_block(a.nx), gr((a.nx + bl.x - 1) / bl.x, a.ny, a.nz);
    if (g->Q == 9) k_adj_stream<9, P><<<gr, bl, 0, g->stream>>>(a, b, out);
    else k_adj_stream<19, P><<<gr, bl, 0, g->stream>>>(a, b, out);
    return hipGetLastError();
}

int check_adjoint_grid(const lumagpu_grid *g) {
    if (g->d.precision != LUMAGPU_FP64 && g->d.precision != LUMAGPU_FP32S)
        return fail(LUMAGPU_EUNSUPPORTED, "the adjoint runs in the FP64 and FP32-shifted forms");
    if (g->parent || !g->kids.empty()) return fail(LUMAGPU_EUNSUPPORTED, "the adjoint runs on a single grid level");
    if (g->zslab) return fail(LUMAGPU_EUNSUPPORTED, "the adjoint does not cover z-slabs");
    if (g->gravity_on) return fail(LUMAGPU_EUNSUPPORTED, "the adjoint does not cover the gravity reset");
    for (size_t c = 0; c < g->hflags.size(); ++c) {
        const int ty = g->hflags[c] & kTypeMask;
        if (ty == kFluid || ty == kSolid || ty == kExtrapRight) continue;
        // forced-equilibrium velocity sources, regularised velocity and pressure sites
        if (ty == kVelocity || ty == kPressure) continue;
        return fail(LUMAGPU_EUNSUPPORTED,
                    "the adjoint covers fluid, solid, velocity, pressure and ExtrapolateRight sites only");
    }
    if (g->ibm) {
        for (const auto &b : g->ibm->bodies)
            if (b.flexible) return fail(LUMAGPU_EUNSUPPORTED, "the adjoint covers rigid IB bodies only");
        // the interpolation's adjoint spreads to fluid support sites
        for (const auto &b : g->ibm->bodies)
            for (const auto &m : b.m)
                for (int k = 0; k < m.ns; ++k) {
                    const size_t c = (size_t)m.sijk[k][0] +
                                     (size_t)g->d.N * ((size_t)m.sijk[k][1] + (size_t)g->d.M * m.sijk[k][2]);
                    const int t = c < g->hflags.size() ? (g->hflags[c] & kTypeMask) : kFluid;
                    if (t == kVelocity || t == kPressure)
                        return fail(LUMAGPU_EUNSUPPORTED,
                                    "the adjoint does not cover IB supports on velocity or pressure sites");
                }
    }
    return 0;
}

// The epsilon chain of one system (a body's markers, or with the universal system every marker
// of the grid in body order): xg += dJ/dx through eps (A eps = 1), and dsbar += the part of
// dJ/d ds that enters through A's columns.
int epsilon_chain(const lumagpu_grid *g, const std::vector<const Marker *> &ms, const double *epsbar, double *dsbar,
                  double *xg) {
    const int n = (int)ms.size(), D = g->D;
    const double dh = g->d.dh;
    // A_IJ = ds_J sum_k delta(x_I; s^I_k) delta(x_J; s^I_k) area_I; solve A^T mu = epsbar
    std::vector<double> A((size_t)n * n, 0.0);
    int kl = 0, ku = 0;   // band of A^T's column-major view, which the solvers factor: A's own
    for (int I = 0; I < n; ++I)
        for (int J = 0; J < n; ++J) {
            if (far_apart(*ms[I], *ms[J], D, dh)) continue;
            double acc = 0.0;
            for (int k = 0; k < ms[I]->ns; ++k)
                acc += ms[I]->delta[k] * delta_at(ms[J]->pos, ms[I]->sxyz[k], dh, ms[J]->dilation, D) * ms[I]->area;
            A[(size_t)I * n + J] = acc * ms[J]->ds;
            if (A[(size_t)I * n + J] != 0.0) {
                kl = std::max(kl, I - J);
                ku = std::max(ku, J - I);
            }
        }
    std::vector<double> At((size_t)n * n), mu(epsbar, epsbar + n);
    for (int I = 0; I < n; ++I)
        for (int J = 0; J < n; ++J) At[(size_t)J * n + I] = A[(size_t)I * n + J];
    // markers ordered along a body (a sphere's lattice by height, a filament along its length)
    // couple only near neighbours in index: the banded solver skips the exact zeros outside the
    // band and otherwise does the dense solver's operations in its order (the same solution)
    const int r = (kl + ku < n - 1) ? lu_solve_band(n, kl, ku, At, mu, "singular IB epsilon system")
                                    : lu_solve(n, At, mu);
    if (r) return r;
    for (int I = 0; I < n; ++I) {
        const Marker &mI = *ms[I];
        for (int J = 0; J < n; ++J) {
            const Marker &mJ = *ms[J];
            const double Abar = -mu[I] * mJ.eps;
            if (Abar == 0.0 || far_apart(mI, mJ, D, dh)) continue;
            dsbar[J] += Abar * A[(size_t)I * n + J] / mJ.ds;
            for (int k = 0; k < mI.ns; ++k) {
                double gI[3], gJ[3];
                delta_grad(mI.pos, mI.sxyz[k], dh, mI.dilation, D, gI);
                delta_grad(mJ.pos, mI.sxyz[k], dh, mJ.dilation, D, gJ);
                const double dJk = delta_at(mJ.pos, mI.sxyz[k], dh, mJ.dilation, D);
                for (int a = 0; a < D; ++a) {
                    xg[3 * I + a] += Abar * mJ.ds * gI[a] * dJk * mI.area;
                    xg[3 * J + a] += Abar * mJ.ds * mI.delta[k] * gJ[a] * mI.area;
                }
            }
        }
    }
    return 0;
}

// The ds chain of one body (ibm_computeDs is per body): ds_m = min(10, min_n |x_m - x_n| / dh)
void ds_chain(const lumagpu_grid *g, const Body &b, const double *dsbar, double *xg) {
    const int n = (int)b.m.size(), D = g->D;
    const double dh = g->d.dh;
    // positions side by side (a marker record spans 1.6 KB)
    std::vector<double> p(3 * (size_t)n);
    for (int m = 0; m < n; ++m)
        for (int a = 0; a < 3; ++a) p[3 * (size_t)m + a] = b.m[m].pos[a];
    for (int m = 0; m < n; ++m) {
        double best = 10.0;
        int arg = -1;
        for (int q = 0; q < n; ++q) {
            if (q == m) continue;
            double acc = 0.0;
            for (int a = 0; a < 3; ++a) acc += std::pow(p[3 * (size_t)m + a] - p[3 * (size_t)q + a], 2);
            const double dist = std::sqrt(acc) / dh;
            if (dist < best) {
                best = dist;
                arg = q;
            }
        }
        if (arg < 0 || best <= 0.0) continue;
        for (int a = 0; a < D; ++a) {
            const double gdir = (b.m[m].pos[a] - b.m[arg].pos[a]) / (best * dh * dh);
            xg[3 * m + a] += dsbar[m] * gdir;
            xg[3 * arg + a] -= dsbar[m] * gdir;
        }
    }
}

// epsilon_chain on the device for a system of kLuDeviceMin markers and more: assembly, LU and the sums
// over near pairs are O(n^2) and O(n^3) work that one host thread took 94 ms for at 804 markers
// (here 6.5 ms); the O(n^2) substitutions stay on the host, and so does the whole solve of a sparse
// matrix (kLuSparse).  first: the system's first marker in the grid's marker arrays; sdd: the gradients of
// the delta weights.  LUMAGPU_ENOMEM before anything of the caller's has been written.
int epsilon_chain_device(lumagpu_grid *g, const std::vector<const Marker *> &ms, int first, const double *sdd,
                         const double *epsbar, double *dsbar, double *xg) {
    const IbmSystem *s = g->ibm;
    const size_t n = ms.size(), S = (size_t)s->S;
    std::vector<double> h(5 * n + 3 * n * S, 0.0);
    for (size_t i = 0; i < n; ++i) {
        for (int a = 0; a < 3; ++a) h[3 * i + a] = ms[i]->pos[a];
        h[3 * n + i] = ms[i]->dilation;
        h[4 * n + i] = ms[i]->area;
        for (int k = 0; k < ms[i]->ns; ++k)
            for (int a = 0; a < 3; ++a) h[5 * n + 3 * (i * S + k) + a] = ms[i]->sxyz[k][a];
    }
    // markers; then mu, xg and dsbar; the matrix; pivots, info and its shape
    DevBuf geo, vec, mat, piv;
    if (int r = geo.alloc(g, h.size() * sizeof(double))) return r;
    if (int r = vec.alloc(g, 5 * n * sizeof(double))) return r;
    if (int r = mat.alloc(g, n * n * sizeof(double))) return r;
    if (int r = piv.alloc(g, (n + 4) * sizeof(int))) return r;
    double *gd = static_cast<double *>(geo.p), *vd = static_cast<double *>(vec.p), *a = static_cast<double *>(mat.p);
    int *pd = static_cast<int *>(piv.p);
    HIP_TRY(hipMemcpyAsync(gd, h.data(), h.size() * sizeof(double), hipMemcpyHostToDevice, g->stream));
    const EpsSystem e{(int)n,       s->S,           g->D,          g->d.dh,
                      gd,           gd + 3 * n,     gd + 4 * n,    gd + 5 * n,
                      s->d_ns + first, s->d_sdelta + (size_t)first * S, sdd + (size_t)first * S * 3, s->d_eps + first,
                      s->d_ds + first};
    HIP_TRY(hipMemsetAsync(pd + n + 1, 0, 3 * sizeof(int), g->stream));
    k_eps_matrix<<<dim3((unsigned)((n + 255) / 256), (unsigned)n), 256, 0, g->stream>>>(e, a, pd + n + 1);
    HIP_TRY(hipGetLastError());
    int shape[3];   // the band of A^T's column-major view, as in epsilon_chain, and the nonzeros
    HIP_TRY(hipMemcpyAsync(shape, pd + n + 1, sizeof shape, hipMemcpyDeviceToHost, g->stream));
    HIP_TRY(hipStreamSynchronize(g->stream));
    const bool sparse = (size_t)shape[2] <= kLuSparse * n;
    if (!sparse) HIP_TRY(lu_factor_device((int)n, a, pd, pd + n, g->stream));
    // the host's pages while the device factors
    std::vector<double> lu(n * n), v(epsbar, epsbar + n);
    std::vector<int> hp(n + 1);
    HIP_TRY(hipMemcpyAsync(hp.data(), pd, hp.size() * sizeof(int), hipMemcpyDeviceToHost, g->stream));
    if (int r = copy_to_host(g, lu.data(), a, lu.size() * sizeof(double))) return r;
    HIP_TRY(hipStreamSynchronize(g->stream));
    if (sparse) {
        const int kl = shape[0], ku = shape[1];
        if (int r = kl + ku < (int)n - 1 ? lu_solve_band((int)n, kl, ku, lu, v, "singular IB epsilon system")
                                         : lu_solve((int)n, lu, v))
            return r;
    } else {
        if (hp[n]) return fail(LUMAGPU_EPHYS, "singular IB epsilon system");
        lu_substitute((int)n, lu.data(), hp.data(), v.data());
    }
    v.resize(5 * n);
    std::copy(xg, xg + 3 * n, v.begin() + n);
    std::copy(dsbar, dsbar + n, v.begin() + 4 * n);
    HIP_TRY(hipMemcpyAsync(vd, v.data(), v.size() * sizeof(double), hipMemcpyHostToDevice, g->stream));
    k_eps_chain<<<(unsigned)((n + 3) / 4), 256, 0, g->stream>>>(e, vd, vd + n, vd + 4 * n);
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipMemcpyAsync(v.data(), vd, v.size() * sizeof(double), hipMemcpyDeviceToHost, g->stream));
    HIP_TRY(hipStreamSynchronize(g->stream));
    std::copy(v.begin() + n, v.begin() + 4 * n, xg);
    std::copy(v.begin() + 4 * n, v.end(), dsbar);
    return 0;
}

// dJ/dx of every marker through epsilon and ds, per body or through the universal system
int position_chains(lumagpu_grid *g, const double *sdd, const double *epsbar, const double *dsbar_dev,
                    double *xg) {
    const IbmSystem *s = g->ibm;
    std::vector<double> dsbar(dsbar_dev, dsbar_dev + s->nm);
    auto chain = [&](const std::vector<const Marker *> &ms, int first) {
        const double *eb = epsbar + first;
        double *db = dsbar.data() + first, *xb = xg + 3 * (size_t)first;
        const int n = (int)ms.size();
        if (n >= kLuDeviceMin && n <= kLuDeviceMax) {
            const int r = epsilon_chain_device(g, ms, first, sdd, eb, db, xb);
            if (r != LUMAGPU_ENOMEM) return r;
            (void)hipGetLastError();   // no room for its matrix: nothing has been written yet
        }
        return epsilon_chain(g, ms, eb, db, xb);
    };
    if (s->universal) {
        std::vector<const Marker *> ms;
        for (const auto &b : s->bodies)
            for (const auto &m : b.m) ms.push_back(&m);
        if (int r = chain(ms, 0)) return r;
    } else {
        for (const auto &b : s->bodies) {
            std::vector<const Marker *> ms;
            for (const auto &m : b.m) ms.push_back(&m);
            if (int r = chain(ms, b.first)) return r;
        }
    }
    for (const auto &b : s->bodies) ds_chain(g, b, dsbar.data() + b.first, xg + 3 * (size_t)b.first);
    return 0;
}

// While a segment runs along the tape or is reversed, the grid's pointers stand on the tape; they go
// back to the grid's own arrays on every way out.
struct OnTape {
    lumagpu_grid *g;
    void *own;
    int store;
    ~OnTape() {
        g->store_macro = store;
        g->f = own;
        g->f_to = nullptr;
        g->xr_tape = nullptr;
        g->xr_ready = 0;
    }
};

template <class P>
int adj_run(lumagpu_grid *g, int nsteps, int every, const double dir[3], int backward, lumagpu_adj_result *res,
            double *dpos, double *lambda0) {
    g->xr_ready = 0;   // the populations change outside the step kernels
    g->pair_synced = 0;
    using T = typename P::T;
    IbmSystem *s = g->ibm;
    const bool ib = s && s->nm > 0;
    const size_t fbytes = (size_t)g->elem * g->Q * g->ps;
    const double invT = 1.0 / nsteps;
    const int nck = (nsteps + every - 1) / every;
    const int t_start = g->t;   // step t of the run runs at grid time t_start + t (velocity ramp)
    // A labelled step can write its successor state elsewhere, so a segment runs from its checkpoint
    // along the tape without a copy per step, the last segment already in the forward run; outlet
    // sources are taped beside the states.  Every slot a step reads was written by the step before,
    // except where an outlet row's source is a site that never steps (xr_fold): such grids, and unlabelled
    // ones, step in place and copy.
    const bool along = backward && g->masked && (!g->has_outlet || g->xr_fold);
    const size_t xr_size = (size_t)g->Q * g->d.M * g->d.K;

    OnTape guard{g, g->f, g->store_macro};
    std::vector<DevBuf> ck(nck), tape(every);
    std::vector<int> ckpar(nck), tpar(every);
    for (auto &b : ck)
        if (int r = b.alloc(g, fbytes)) return r;
    DevBuf fin, accJ, xrt;
    if (!along && backward)
        if (int r = fin.alloc(g, fbytes)) return r;
    if (backward)
        for (int i = along ? 1 : 0; i < std::min(every, nsteps); ++i)
            if (int r = tape[i].alloc(g, fbytes)) return r;
    if (along && g->has_outlet)
        if (int r = xrt.alloc(g, (size_t)(std::min(every, nsteps) + 1) * xr_size * sizeof(double))) return r;
    // J; omega (fluid sites) and inlet scale (sources); omega and inlet scale (edge, corner and
    // pressure sites); omega and inlet scale (regularised faces)
    if (int r = accJ.alloc(g, 7 * sizeof(double))) return r;
    HIP_TRY(hipMemsetAsync(accJ.p, 0, 7 * sizeof(double), g->stream));

    auto objective = [&]() {
        if (!ib) return 0;
        k_adj_objective<<<1, 64, 0, g->stream>>>(ibm_args(g), dir[0], dir[1], dir[2], invT,
                                                 static_cast<double *>(accJ.p));
        HIP_TRY(hipGetLastError());
        return 0;
    };
    // state i of segment seg on the tape
    auto state = [&](int seg, int i) { return along && i == 0 ? ck[seg].p : tape[i].p; };
    // along the tape: the steps of a segment from its checkpoint, n of them, the last one into `end`
    auto run_along = [&](int seg, int n, void *end, bool forward) {
        g->parity = ckpar[seg];
        g->t = t_start + seg * every;
        g->xr_ready = 0;
        const int len = std::min(nsteps, (seg + 1) * every) - seg * every;
        for (int i = 0; i < len; ++i) {
            tpar[i] = g->parity;
            g->f = state(seg, i);
            if (g->has_outlet) g->xr_tape = static_cast<double *>(xrt.p) + i * xr_size;
            if (i >= n) {
                // the segment's last state: its outlet sources came with the step before
                if (g->has_outlet && !g->xr_ready) HIP_TRY(outlet_prepass(g));
                break;
            }
            g->f_to = i + 1 < len ? state(seg, i + 1) : end;
            if (int r = step_grid(g, 0)) return r;
            g->xr_ready = 1;
            if (forward)
                if (int r = objective()) return r;
        }
        g->f = guard.own;
        g->f_to = nullptr;
        g->xr_tape = nullptr;
        g->xr_ready = 0;
        // the end state's slots that no step wrote: those of forced-equilibrium sites
        if (forward && !g->d.regularised && len >= 2) {
            using S = typename P::S;
            const S *from = static_cast<const S *>(state(seg, len - 1));
            const unsigned nb = (unsigned)((g->ncell + 255) / 256);
            const StepArgs a = make_args(g);
            const int odd = tpar[len - 1] == 0;
            if (g->Q == 9) k_adj_carry<9, S><<<nb, 256, 0, g->stream>>>(a, from, static_cast<S *>(end), odd);
            else k_adj_carry<19, S><<<nb, 256, 0, g->stream>>>(a, from, static_cast<S *>(end), odd);
            HIP_TRY(hipGetLastError());
        }
        return 0;
    };

    // forward with checkpoints
    for (int t = 0; t < nsteps; ++t) {
        if (t % every == 0) {
            HIP_TRY(hipMemcpyAsync(ck[t / every].p, g->f, fbytes, hipMemcpyDeviceToDevice, g->stream));
            ckpar[t / every] = g->parity;
            if (along && t / every == nck - 1) {
                if (int r = run_along(nck - 1, nsteps - t, g->f, true)) return r;
                break;
            }
        }
        if (int r = step_grid(g, 0)) return r;
        if (int r = objective()) return r;
    }
    if (fin.p) HIP_TRY(hipMemcpyAsync(fin.p, g->f, fbytes, hipMemcpyDeviceToDevice, g->stream));
    const int fin_par = g->parity, fin_t = g->t;
    const double fin_omega = g->d.omega;
    double hacc[7] = {0, 0, 0, 0, 0, 0, 0};
    if (!backward) {
        HIP_TRY(hipMemcpyAsync(hacc, accJ.p, sizeof(hacc), hipMemcpyDeviceToHost, g->stream));
        HIP_TRY(hipStreamSynchronize(g->stream));
        if (res) *res = lumagpu_adj_result{hacc[0], 0.0, 0.0};
        return 0;
    }

    // backward buffers
    const size_t nc = g->ncell;
    // the macro arrays as the forward run left them: the reversed steps rewrite them at the supports
    DevBuf mrho, mu;
    const size_t mbytes = nc * g->melem;
    if (ib) {
        if (int r = mrho.alloc(g, mbytes)) return r;
        if (int r = mu.alloc(g, mbytes * g->D)) return r;
        HIP_TRY(hipMemcpyAsync(mrho.p, g->rho, mbytes, hipMemcpyDeviceToDevice, g->stream));
        HIP_TRY(hipMemcpyAsync(mu.p, g->u, mbytes * g->D, hipMemcpyDeviceToDevice, g->stream));
    }
    guard.store = g->store_macro;   // the recomputed steps' fields are nobody's
    g->store_macro = 0;
    // blocks of the collide and stream launches (cell_block rows)
    const int nblk = (int)((g->d.N + cell_block(g->d.N).x - 1) / cell_block(g->d.N).x) * g->d.M * g->d.K;
    // the adjoint of the streamed populations, this step's and the later one's (zero after the last
    // step), with the populations' plane stride: planes of a power of two times the element apart
    // fall on the same memory channels
    const size_t gbytes = (size_t)g->Q * g->ps * sizeof(T);
    DevBuf gb[2], fbar, part;
    if (int r = gb[0].alloc(g, gbytes)) return r;
    if (int r = gb[1].alloc(g, gbytes)) return r;
    if (int r = fbar.alloc(g, 3 * nc * sizeof(double))) return r;
    // large grids: the fluid sites that are not plain, and those that feed an outlet
    DevBuf list_cells;
    int nlist = -1;
    if (nc >= kAdjSplitMin && g->plain) {
        const size_t words = (nc + 31) / 32;
        std::vector<uint32_t> plain(words);
        HIP_TRY(hipMemcpyAsync(plain.data(), g->plain, words * sizeof(uint32_t), hipMemcpyDeviceToHost, g->stream));
        HIP_TRY(hipStreamSynchronize(g->stream));
        std::vector<int> lc;
        for (size_t w = 0; w < words; ++w)
            for (uint32_t m = ~plain[w]; m; m &= m - 1) {
                const size_t c = 32 * w + __builtin_ctz(m);
                if (c < nc && (g->hflags[c] & kTypeMask) == kFluid) lc.push_back((int)c);
            }
        if (g->has_outlet)
            for (size_t row = 0; row < nc; row += g->d.N) {
                const size_t c = row + g->d.N - 3;
                if ((plain[c >> 5] >> (c & 31)) & 1u) lc.push_back((int)c);
            }
        std::sort(lc.begin(), lc.end());
        nlist = (int)lc.size();
        if (nlist > 0) {
            if (int r = list_cells.alloc(g, lc.size() * sizeof(int))) return r;
            HIP_TRY(hipMemcpy(list_cells.p, lc.data(), lc.size() * sizeof(int), hipMemcpyHostToDevice));
        }
    }
    const int nblk_all = nblk + (nlist > 0 ? (nlist + kAdjListBlock - 1) / kAdjListBlock : 0);
    // omega (collision), inlet scale (streaming from forced-equilibrium sources)
    if (int r = part.alloc(g, 2 * (size_t)nblk_all * sizeof(double))) return r;
    HIP_TRY(hipMemsetAsync(gb[0].p, 0, gbytes, g->stream));
    HIP_TRY(hipMemsetAsync(fbar.p, 0, 3 * nc * sizeof(double), g->stream));
    AdjArgs<T> ab{};
    ab.gin = static_cast<const T *>(gb[0].p);
    ab.gbar = static_cast<T *>(gb[1].p);
    ab.ps = g->ps;
    ab.fbar = static_cast<double *>(fbar.p);
    ab.part = static_cast<double *>(part.p);
    ab.nblk = nblk;
    ab.nblk_all = nblk_all;
    ab.outlet = g->has_outlet;
    ab.ramp_feq = 1.0;
    DevBuf mbar, xbar, epsbar, dsbar, sdd;
    AdjIbm aj{};
    if (ib) {
        const size_t nm = (size_t)s->nm;
        if (int r = mbar.alloc(g, 4 * nm * sizeof(double))) return r;
        if (int r = xbar.alloc(g, 3 * nm * sizeof(double))) return r;
        if (int r = epsbar.alloc(g, nm * sizeof(double))) return r;
        if (int r = dsbar.alloc(g, nm * sizeof(double))) return r;
        if (int r = sdd.alloc(g, nm * s->S * 3 * sizeof(double))) return r;
        HIP_TRY(hipMemsetAsync(xbar.p, 0, 3 * nm * sizeof(double), g->stream));
        HIP_TRY(hipMemsetAsync(epsbar.p, 0, nm * sizeof(double), g->stream));
        HIP_TRY(hipMemsetAsync(dsbar.p, 0, nm * sizeof(double), g->stream));
        std::vector<double> h(nm * s->S * 3, 0.0);
        for (const auto &b : s->bodies)
            for (size_t i = 0; i < b.m.size(); ++i) {
                const Marker &m = b.m[i];
                for (int k = 0; k < m.ns; ++k)
                    delta_grad(m.pos, m.sxyz[k], g->d.dh, m.dilation, g->D,
                               &h[((size_t)(b.first + i) * s->S + k) * 3]);
            }
        HIP_TRY(hipMemcpyAsync(sdd.p, h.data(), h.size() * sizeof(double), hipMemcpyHostToDevice, g->stream));
        HIP_TRY(hipStreamSynchronize(g->stream));
        aj.fbar = static_cast<double *>(fbar.p);
        aj.sddelta = static_cast<double *>(sdd.p);
        aj.mbar = static_cast<double *>(mbar.p);
        aj.xbar = static_cast<double *>(xbar.p);
        aj.epsbar = static_cast<double *>(epsbar.p);
        aj.dsbar = static_cast<double *>(dsbar.p);
        for (int d = 0; d < 3; ++d) aj.dir[d] = dir[d];
        aj.invT = invT;
    }
    double *acc = static_cast<double *>(accJ.p);
    // edge and corner velocity sites: per-site density adjoints and parameter derivatives, and
    // the neighbour cells they extrapolate from with their entries (2 * site + 0 for x + n,
    // + 1 for x + 2n), in ascending order
    EdgeArgs ea{};
    ea.n = g->nedge;
    ea.cell = g->edge;
    ea.nrm = g->edge + g->nedge;
    ea.n1 = g->edge + 2 * g->nedge;
    ea.n2 = g->edge + 3 * g->nedge;
    ea.erho = g->erho;
    DevBuf dbar, tbar, epart, enb_cell, enb_ptr, enb_ent;
    int n_enb = 0;
    if (g->nedge > 0) {
        const int ne = g->nedge;
        std::vector<int> he(4 * (size_t)ne);
        HIP_TRY(hipMemcpyAsync(he.data(), g->edge, he.size() * sizeof(int), hipMemcpyDeviceToHost, g->stream));
        HIP_TRY(hipStreamSynchronize(g->stream));
        std::vector<std::pair<int, int>> pairs;   // (cell, code)
        for (int i = 0; i < ne; ++i) {
            pairs.emplace_back(he[2 * (size_t)ne + i], 2 * i);
            pairs.emplace_back(he[3 * (size_t)ne + i], 2 * i + 1);
        }
        std::sort(pairs.begin(), pairs.end());
        std::vector<int> cells, ptr{0}, ent;
        for (size_t k = 0; k < pairs.size(); ++k) {
            if (k == 0 || pairs[k].first != pairs[k - 1].first) {
                if (k) ptr.push_back((int)ent.size());
                cells.push_back(pairs[k].first);
            }
            ent.push_back(pairs[k].second);
        }
        ptr.push_back((int)ent.size());
        n_enb = (int)cells.size();
        if (int r = dbar.alloc(g, ne * sizeof(double))) return r;
        if (int r = tbar.alloc(g, 3 * (size_t)ne * sizeof(double))) return r;
        if (int r = epart.alloc(g, 2 * (size_t)ne * sizeof(double))) return r;
        if (int r = enb_cell.alloc(g, cells.size() * sizeof(int))) return r;
        if (int r = enb_ptr.alloc(g, ptr.size() * sizeof(int))) return r;
        if (int r = enb_ent.alloc(g, ent.size() * sizeof(int))) return r;
        HIP_TRY(hipMemcpy(enb_cell.p, cells.data(), cells.size() * sizeof(int), hipMemcpyHostToDevice));
        HIP_TRY(hipMemcpy(enb_ptr.p, ptr.data(), ptr.size() * sizeof(int), hipMemcpyHostToDevice));
        HIP_TRY(hipMemcpy(enb_ent.p, ent.data(), ent.size() * sizeof(int), hipMemcpyHostToDevice));
    }

    // the adjoint kernels read the plain-site bitmap without a null check: a grid whose flags
    // the IB set-up made (no bitmap) gets one with no plain site
    DevBuf nobits;
    if (!g->plain) {
        if (int r = nobits.alloc(g, (nc + 31) / 32 * sizeof(uint32_t))) return r;
        HIP_TRY(hipMemsetAsync(nobits.p, 0, (nc + 31) / 32 * sizeof(uint32_t), g->stream));
    }

    // regularised velocity faces (not edges or corners): their own kernel, over a list
    DevBuf face_cells, fpart;
    int nface = 0;
    if (g->d.regularised) {
        std::vector<int> fc;
        for (size_t c = 0; c < g->hflags.size(); ++c) {
            const unsigned fl = g->hflags[c];
            if ((fl & kTypeMask) == kVelocity && ((fl >> kNormalShift) & 7) != kNormalEdge) fc.push_back((int)c);
        }
        nface = (int)fc.size();
        if (nface > 0) {
            if (int r = face_cells.alloc(g, fc.size() * sizeof(int))) return r;
            if (int r = fpart.alloc(g, 2 * fc.size() * sizeof(double))) return r;
            HIP_TRY(hipMemcpy(face_cells.p, fc.data(), fc.size() * sizeof(int), hipMemcpyHostToDevice));
        }
    }

    int rc = 0;
    StepArgs a_first;   // the arguments of the step reversed last
    for (int seg = nck - 1; seg >= 0 && !rc; --seg) {
        const int t0 = seg * every, t1 = std::min(nsteps, t0 + every);
        if (along) {
            // the states of the last segment are on the tape from the forward run
            if (seg < nck - 1) rc = run_along(seg, t1 - t0 - 1, nullptr, false);
        } else {
            HIP_TRY(hipMemcpyAsync(g->f, ck[seg].p, fbytes, hipMemcpyDeviceToDevice, g->stream));
            g->parity = ckpar[seg];
            g->t = t_start + t0;
            g->xr_ready = 0;
            for (int t = t0; t < t1 && !rc; ++t) {
                HIP_TRY(hipMemcpyAsync(tape[t - t0].p, g->f, fbytes, hipMemcpyDeviceToDevice, g->stream));
                tpar[t - t0] = g->parity;
                if (t + 1 < t1) rc = step_grid(g, 0);
            }
        }
        for (int t = t1 - 1; t >= t0 && !rc; --t) {
            // the step's input state stands in for the grid's populations while it is reversed
            g->f = state(seg, t - t0);
            g->t = t_start + t;
            g->parity = tpar[t - t0];
            if (along && g->has_outlet) {
                g->xr_tape = static_cast<double *>(xrt.p) + (t - t0) * xr_size;
            } else if (g->has_outlet) {
                hipError_t e = outlet_prepass(g);
                if (e != hipSuccess) rc = fail(LUMAGPU_EHIP, std::string("adjoint outlet: ") + hipGetErrorString(e));
            }
            if (!rc && ib) rc = apply_core(g);
            // a Reynolds ramp: this step's omega, and its omega partial weighted onto the omega
            // after the ramp
            double w_om = 1.0;
            if (g->re_ramp > 0.0) {
                update_reynolds(g);
                w_om = reynolds_omega_weight(g);
            }
            StepArgs a = make_args(g);
            if (!a.plain) a.plain = static_cast<const uint32_t *>(nobits.p);
            if (!rc) {
                AdjSums sums{};
                int nsum = 0;
                auto add_sum = [&](const double *part, int n, double *to) {
                    sums.part[nsum] = part;
                    sums.n[nsum] = n;
                    sums.acc[nsum++] = to;
                };
                // the edge sites' extrapolation densities of this step
                hipError_t e = g->nedge ? launch_edges(g, a, 0) : hipSuccess;
                if (e == hipSuccess) e = launch_adj_collide<P>(g, a, ab, static_cast<const int *>(list_cells.p), nlist);
                if (e == hipSuccess && nface) {
                    const dim3 fb(64), fg((unsigned)((nface + 63) / 64), (unsigned)(g->Q + 2));
                    const int *fcp = static_cast<const int *>(face_cells.p);
                    double *fp = static_cast<double *>(fpart.p);
                    const bool odd = g->parity == 0;
                    if (g->Q == 9) {
                        if (odd) k_adj_faces<9, P, true><<<fg, fb, 0, g->stream>>>(a, ab, fcp, nface, fp);
                        else k_adj_faces<9, P, false><<<fg, fb, 0, g->stream>>>(a, ab, fcp, nface, fp);
                    } else {
                        if (odd) k_adj_faces<19, P, true><<<fg, fb, 0, g->stream>>>(a, ab, fcp, nface, fp);
                        else k_adj_faces<19, P, false><<<fg, fb, 0, g->stream>>>(a, ab, fcp, nface, fp);
                    }
                    e = hipGetLastError();
                    add_sum(fp, nface, acc + 5);
                }
                if (e == hipSuccess && g->nedge) {
                    const dim3 eb(64), eg((unsigned)((g->nedge + 63) / 64), (unsigned)(g->Q + 4));
                    double *db = static_cast<double *>(dbar.p), *tb = static_cast<double *>(tbar.p);
                    double *ep = static_cast<double *>(epart.p);
                    const int *nc_p = static_cast<const int *>(enb_cell.p), *np_p = static_cast<const int *>(enb_ptr.p);
                    const int *ne_p = static_cast<const int *>(enb_ent.p);
                    const dim3 nbb(128), nbg((unsigned)((n_enb + 127) / 128));
                    if (g->Q == 9) {
                        if (g->parity == 0) k_adj_edges<9, P, true><<<eg, eb, 0, g->stream>>>(a, ea, ab, db, tb, ep);
                        else k_adj_edges<9, P, false><<<eg, eb, 0, g->stream>>>(a, ea, ab, db, tb, ep);
                        e = hipGetLastError();
                        if (e == hipSuccess)
                            k_adj_edge_nbrs<9, T><<<nbg, nbb, 0, g->stream>>>(n_enb, nc_p, np_p, ne_p, db, tb, g->erho,
                                                                             ab.ps, ab.gbar);
                    } else {
                        if (g->parity == 0) k_adj_edges<19, P, true><<<eg, eb, 0, g->stream>>>(a, ea, ab, db, tb, ep);
                        else k_adj_edges<19, P, false><<<eg, eb, 0, g->stream>>>(a, ea, ab, db, tb, ep);
                        e = hipGetLastError();
                        if (e == hipSuccess)
                            k_adj_edge_nbrs<19, T><<<nbg, nbb, 0, g->stream>>>(n_enb, nc_p, np_p, ne_p, db, tb, g->erho,
                                                                              ab.ps, ab.gbar);
                    }
                    if (e == hipSuccess) e = hipGetLastError();
                    add_sum(ep, g->nedge, acc + 3);
                }
                if (e == hipSuccess && ib) {
                    IbmArgs ia = ibm_args(g);
                    k_adj_ibm_marker<<<(s->nm + 3) / 4, 256, 0, g->stream>>>(ia, aj);
                    e = hipGetLastError();
                    if (e == hipSuccess) {
                        if (g->Q == 9)
                            k_adj_ibm_site<9, T><<<(s->nsites + 127) / 128, 128, 0, g->stream>>>(
                                ia, aj.mbar, g->flags, ab.ps, ab.gbar);
                        else
                            k_adj_ibm_site<19, T><<<(s->nsites + 127) / 128, 128, 0, g->stream>>>(
                                ia, aj.mbar, g->flags, ab.ps, ab.gbar);
                        e = hipGetLastError();
                    }
                }
                if (e == hipSuccess) {
                    add_sum(ab.part, nblk_all, acc + 1);
                    k_adj_sum_partials<<<nsum, 1024, 0, g->stream>>>(sums, w_om);
                    e = hipGetLastError();
                }
                if (e != hipSuccess) rc = fail(LUMAGPU_EHIP, std::string("adjoint launch: ") + hipGetErrorString(e));
            }
            // what this step streamed is the later step's adjoint for the one before it
            T *next = const_cast<T *>(ab.gin);
            ab.gin = ab.gbar;
            ab.gbar = next;
            ab.ramp_feq = a.ramp_feq;
            ab.ramp_on = a.ramp_on;
            a_first = a;
            g->f = guard.own;
            g->xr_tape = nullptr;
        }
    }
    if (!rc) {
        // the first step's streaming: the initial populations' adjoint (into the free array) and its
        // share of the inlet scale, from the blocks over the grid alone
        ab.nblk_all = nblk;
        hipError_t e = launch_adj_stream<P>(g, a_first, ab, lambda0 ? ab.gbar : nullptr);
        if (e == hipSuccess) {
            AdjSums sums{};
            sums.part[0] = ab.part;
            sums.n[0] = nblk;
            sums.acc[0] = acc + 1;
            k_adj_sum_partials<<<1, 1024, 0, g->stream>>>(sums, 1.0);
            e = hipGetLastError();
        }
        if (e != hipSuccess) rc = fail(LUMAGPU_EHIP, std::string("adjoint launch: ") + hipGetErrorString(e));
    }
    // the grid returns to the end of the forward run
    if (ib) {
        HIP_TRY(hipMemcpyAsync(g->rho, mrho.p, mbytes, hipMemcpyDeviceToDevice, g->stream));
        HIP_TRY(hipMemcpyAsync(g->u, mu.p, mbytes * g->D, hipMemcpyDeviceToDevice, g->stream));
    }
    if (fin.p) HIP_TRY(hipMemcpyAsync(g->f, fin.p, fbytes, hipMemcpyDeviceToDevice, g->stream));
    g->parity = fin_par;
    g->t = fin_t;
    g->d.omega = fin_omega;
    g->xr_ready = 0;
    if (rc) return rc;
    HIP_TRY(hipMemcpyAsync(hacc, accJ.p, sizeof(hacc), hipMemcpyDeviceToHost, g->stream));
    if (lambda0) {
        // LUMA's layout on the device, then one copy
        DevBuf lout;
        if (int r = lout.alloc(g, (size_t)g->Q * nc * sizeof(double))) return r;
        const unsigned nb = (unsigned)((nc + 255) / 256);
        if (g->Q == 9)
            k_adj_to_luma<9, T><<<nb, 256, 0, g->stream>>>(ab.gbar, g->ps, nc, g->d.N, g->d.M, g->d.K,
                                                         static_cast<double *>(lout.p));
        else
            k_adj_to_luma<19, T><<<nb, 256, 0, g->stream>>>(ab.gbar, g->ps, nc, g->d.N, g->d.M,
                                                          g->d.K, static_cast<double *>(lout.p));
        HIP_TRY(hipGetLastError());
        if (int r = copy_to_host(g, lambda0, lout.p, (size_t)g->Q * nc * sizeof(double))) return r;
        HIP_TRY(hipStreamSynchronize(g->stream));
    }
    std::vector<double> hx, he, hd;
    if (ib && dpos) {
        hx.resize(3 * (size_t)s->nm);
        he.resize(s->nm);
        hd.resize(s->nm);
        HIP_TRY(hipMemcpyAsync(hx.data(), xbar.p, hx.size() * sizeof(double), hipMemcpyDeviceToHost, g->stream));
        HIP_TRY(hipMemcpyAsync(he.data(), epsbar.p, he.size() * sizeof(double), hipMemcpyDeviceToHost, g->stream));
        HIP_TRY(hipMemcpyAsync(hd.data(), dsbar.p, hd.size() * sizeof(double), hipMemcpyDeviceToHost, g->stream));
    }
    HIP_TRY(hipStreamSynchronize(g->stream));
    if (res) *res = lumagpu_adj_result{hacc[0], hacc[1] + hacc[3] + hacc[5], hacc[2] + hacc[4] + hacc[6]};
    if (ib && dpos) {
        for (size_t i = 0; i < hx.size(); ++i) dpos[i] = hx[i];
        if (int r = position_chains(g, static_cast<const double *>(sdd.p), he.data(), hd.data(), dpos)) return r;
    }
    return 0;
}

}  // namespace
}  // namespace lumagpu

using namespace lumagpu;

extern "C" int lumagpu_adj_run(lumagpu_grid *g, int nsteps, int checkpoint_every, const double *dir, int backward,
                               lumagpu_adj_result *res, double *dJ_dpos, double *lambda0) {
    if (!g) return fail(LUMAGPU_EINVAL, "null grid handle");
    if (!g->has_state) return fail(LUMAGPU_ESTATE, "adjoint before the populations were initialised");
    if (nsteps <= 0 || checkpoint_every <= 0) return fail(LUMAGPU_EINVAL, "step count and checkpoint interval must be positive");
    if (!dir) return fail(LUMAGPU_EINVAL, "null objective direction");
    if (int r = check_adjoint_grid(g)) return r;
    if (g->ibm && !g->ibm->initialised && g->ibm->nm > 0)
        return fail(LUMAGPU_ESTATE, "IB bodies added but lumagpu_ibm_initialise not called");
    if (!g->flags) {
        if (int r = ensure_flags(g)) return r;
        if (int r = upload_flags(g)) return r;
    }
    std::lock_guard<std::recursive_mutex> lock(g->f2_mu);
    const int r = g->d.precision == LUMAGPU_FP64
                      ? adj_run<P64>(g, nsteps, checkpoint_every, dir, backward, res, dJ_dpos, lambda0)
                      : adj_run<P32S>(g, nsteps, checkpoint_every, dir, backward, res, dJ_dpos, lambda0);
    // a run that ended early may have kernels queued on the blocks that the next one takes, and writes
    // from the host without regard to this stream
    if (r) (void)hipStreamSynchronize(g->stream);
    trim_blocks(g);
    return r;
}
