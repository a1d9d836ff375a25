// api.hip -- the C ABI (include/lumagpu.h): grid handles, state transfer and the step driver.
//
// A grid owns one population array in the AA in-place layout, a per-cell flag byte (only
// for labelled grids), optional FP64 macro arrays and force field, and one HIP stream at the
// default priority.  `parity` records which layout the population array is in:
//   0  post-local: A[opp v][x] = f_v(x)   (after upload, init, or an even step)
//   1  post-neighbour: A[v][x + c_v] = f_v(x), or A[opp v][x] where x + c_v is solid
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdio>
#include <algorithm>
#include <cstring>
#include <mutex>
#include <string>
#include <vector>

#include "internal.hpp"

using namespace lumagpu;

namespace lumagpu {
namespace {
thread_local std::string g_last_error;
}
int fail(int code, const std::string &msg) {
    g_last_error = msg;
    return code;
}
}  // namespace lumagpu

namespace {
hipError_t launch_step(const lumagpu_grid *g, const LaunchSpec &ls, const StepArgs &a) {
    switch (g->d.precision) {
        case LUMAGPU_FP64: return launch_step_f64(ls, a, g->stream);
        case LUMAGPU_FP32S: return launch_step_f32s(ls, a, g->stream);
        case LUMAGPU_FP64T: return launch_step_dual(ls, a, g->stream);
        case LUMAGPU_FP32T: return launch_step_dual32(ls, a, g->stream);
        default: return launch_step_f16s(ls, a, g->stream);
    }
}

hipError_t launch_aux(const lumagpu_grid *g, int op, const double *p0, const double *p1, double *out) {
    const StepArgs a = make_args(g);
    switch (g->d.precision) {
        case LUMAGPU_FP64: return launch_aux_f64(op, g->Q, a, p0, p1, out, g->parity, g->masked, g->stream);
        case LUMAGPU_FP32S: return launch_aux_f32s(op, g->Q, a, p0, p1, out, g->parity, g->masked, g->stream);
        case LUMAGPU_FP64T: return launch_aux_dual(op, g->Q, a, p0, p1, out, g->parity, g->masked, g->stream);
        case LUMAGPU_FP32T: return launch_aux_dual32(op, g->Q, a, p0, p1, out, g->parity, g->masked, g->stream);
        default: return launch_aux_f16s(op, g->Q, a, p0, p1, out, g->parity, g->masked, g->stream);
    }
}

// ---- what runs take for themselves --------------------------------------------------------------
// A run allocates a second population array where its kernels take several steps per launch, if that leaves
// at least half of the free memory free; an adjoint run keeps its blocks.  Both stay with the grid for its
// next run, but all grids of a device together keep at most a sixteenth of its memory (18 GB here: second
// arrays of 236 M FP32 D3Q19 cells), so that a program's other allocations find what they found without
// them.  When an allocation of this library fails, the arrays of grids that are not stepping at that
// moment are given back (g_f2_grids) and it is tried again.
std::mutex g_f2_grids_mu;
std::vector<lumagpu_grid *> g_f2_grids;   // the grids that keep any; their `scratch` says how much

size_t f2_bytes(const lumagpu_grid *g) { return g->ps * g->Q * g->elem; }

// what g keeps, with its f2_mu held
size_t scratch_of(const lumagpu_grid *g) {
    size_t n = g->f2_auto ? f2_bytes(g) : 0;
    for (const auto &b : g->blocks) n += b.bytes;
    return n;
}

// with g_f2_grids_mu held: g is to keep n bytes
void scratch_set(lumagpu_grid *g, size_t n) {
    g->scratch = n;
    const auto it = std::find(g_f2_grids.begin(), g_f2_grids.end(), g);
    if (n > 0 && it == g_f2_grids.end()) g_f2_grids.push_back(g);
    if (n == 0 && it != g_f2_grids.end()) g_f2_grids.erase(it);
}

// the arrays of grids that no run holds, back to the device.  f2_mu is recursive: on the thread of a run
// its own grid's lock is no obstacle, and f2_busy says that its second array is in use.
void f2_give_back() {
    std::lock_guard<std::mutex> lock(g_f2_grids_mu);
    const std::vector<lumagpu_grid *> grids = g_f2_grids;
    for (lumagpu_grid *o : grids) {
        if (!o->f2_mu.try_lock()) continue;
        if (o->stream) (void)hipStreamSynchronize(o->stream);
        if (!o->f2_busy) {
            if (o->f2_auto) {
                (void)hipFree(o->f2);
                o->f2 = nullptr;
            }
            o->f2_auto = o->pair_synced = 0;
        }
        std::vector<lumagpu_grid::Block> kept;
        for (auto &b : o->blocks) {
            if (b.used) kept.push_back(b);
            else (void)hipFree(b.p);
        }
        o->blocks = std::move(kept);
        scratch_set(o, scratch_of(o));
        o->f2_mu.unlock();
    }
}

}  // namespace
namespace lumagpu {
void scratch_note(lumagpu_grid *g) {
    std::lock_guard<std::mutex> lock(g_f2_grids_mu);
    scratch_set(g, scratch_of(g));
}

bool scratch_room(lumagpu_grid *g, size_t more) {
    size_t avail = 0, total = 0;
    if (hipMemGetInfo(&avail, &total) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    std::lock_guard<std::mutex> lock(g_f2_grids_mu);
    size_t n = scratch_of(g) + more;
    for (const lumagpu_grid *o : g_f2_grids)
        if (o != g && o->device == g->device) n += o->scratch;
    if (n > total / 16 || more > avail / 2) return false;
    scratch_set(g, scratch_of(g) + more);
    return true;
}
}  // namespace lumagpu
namespace {

// the second array is being stepped from or into: no allocation meanwhile takes it back
struct F2Use {
    lumagpu_grid *g;
    explicit F2Use(lumagpu_grid *grid) : g(grid) { ++g->f2_busy; }
    F2Use(const F2Use &) = delete;
    F2Use &operator=(const F2Use &) = delete;
    ~F2Use() { --g->f2_busy; }
};

// with g->f2_mu held: true when g->f2 is there.  A run allocates on the device current in the caller; where
// that is not the grid's, it steps as it can without.
bool f2_ensure(lumagpu_grid *g) {
    int device = -1;
    if (hipGetDevice(&device) != hipSuccess || device != g->device) {
        (void)hipGetLastError();
        return false;
    }
    if (g->f2) return true;
    if (!scratch_room(g, f2_bytes(g))) return false;
    if (hipMalloc(&g->f2, f2_bytes(g)) != hipSuccess) {
        (void)hipGetLastError();
        g->f2 = nullptr;
        scratch_note(g);
        return false;
    }
    g->f2_auto = 1;
    g->pair_synced = 0;
    return true;
}

int ensure_stage(lumagpu_grid *g, size_t bytes) {
    if (g->stage_bytes >= bytes) return 0;
    if (g->stage) {
        HIP_TRY(hipStreamSynchronize(g->stream));
        HIP_TRY(hipFree(g->stage));
        g->stage = nullptr;
        g->stage_bytes = 0;
    }
    if (dev_malloc(&g->stage, bytes) != hipSuccess) return fail(LUMAGPU_ENOMEM, "staging allocation failed");
    g->stage_bytes = bytes;
    return 0;
}

// Macro downloads up to this size go through pinned memory that the kernel writes: two copies and
// their hand-over to the DMA engine less, against one more pass of the host over the values.
// 16 steps of a 48 x 48 grid from a checkpoint to the fields on the host: 152 -> 104 us with this
// and the one-kernel checkpoint copy.
constexpr size_t kPinDownload = size_t(1) << 20;
bool ensure_pin(lumagpu_grid *g, size_t bytes) {
    if (g->pin_bytes >= bytes) return true;
    (void)hipHostFree(g->pin);
    g->pin = nullptr;
    g->pin_bytes = 0;
    if (hipHostMalloc(&g->pin, bytes, hipHostMallocDefault) != hipSuccess) {
        (void)hipGetLastError();
        g->pin = nullptr;
        return false;
    }
    g->pin_bytes = bytes;
    return true;
}

int check_grid(const lumagpu_grid *g) {
    if (!g) return fail(LUMAGPU_EINVAL, "null grid handle");
    return 0;
}

// GridUtils::isWithinDomainWall, LUMA/src/GridUtils.cpp:1369-1430: returns edge count and
// the code of the last inward normal found (1..6 = +x,-x,+y,-y,+z,-z).
// GridUtils::isWithinDomainWall (GridUtils.cpp:1369-1430): the number of walls the position
// lies in, the code of the last one (1..6 = +x,-x,+y,-y,+z,-z inward normal) and the combined
// inward vector n.
int wall_normal(const lumagpu_grid_desc &d, double px, double py, double pz, int *code, int n[3]) {
    const double *th = d.wall_thk;
    int cnt = 0;
    *code = 0;
    n[0] = n[1] = n[2] = 0;
    if (px > 0.0 && px < th[0]) { *code = 1; n[0] = 1; cnt++; }
    if (px < d.xmax && px > d.xmax - th[1]) { *code = 2; n[0] = -1; cnt++; }
    if (py > 0.0 && py < th[2]) { *code = 3; n[1] = 1; cnt++; }
    if (py < d.ymax && py > d.ymax - th[3]) { *code = 4; n[1] = -1; cnt++; }
    if (d.dims == 3) {
        if (pz > 0.0 && pz < th[4]) { *code = 5; n[2] = 1; cnt++; }
        if (pz < d.zmax && pz > d.zmax - th[5]) { *code = 6; n[2] = -1; cnt++; }
    }
    return cnt;
}

hipError_t launch_zslab(const lumagpu_grid *g, const StepArgs &a, int phase) {
    switch (g->d.precision) {
        case LUMAGPU_FP64: return launch_zslab_f64(a, phase, g->stream);
        case LUMAGPU_FP32S: return launch_zslab_f32s(a, phase, g->stream);
        case LUMAGPU_FP16S: return launch_zslab_f16s(a, phase, g->stream);
        default: return hipErrorInvalidValue;   // refused by lumagpu_set_zslab
    }
}

}  // namespace

namespace lumagpu {
hipError_t dev_malloc(void **p, size_t bytes) {
    hipError_t e = hipMalloc(p, bytes);
    if (e == hipErrorOutOfMemory) {
        (void)hipGetLastError();
        f2_give_back();
        e = hipMalloc(p, bytes);
    }
    if (e != hipSuccess) *p = nullptr;
    return e;
}

hipError_t launch_edges(const lumagpu_grid *g, const StepArgs &a, int phase) {
    EdgeArgs e{};
    e.n = g->nedge;
    e.cell = g->edge;
    e.nrm = g->edge + g->nedge;
    e.n1 = g->edge + 2 * g->nedge;
    e.n2 = g->edge + 3 * g->nedge;
    e.erho = g->erho;
    const int store = (g->store_macro && a.rho_out) ? 1 : 0;
    const bool odd = g->parity == 0;
    switch (g->d.precision) {
        case LUMAGPU_FP64: return launch_edges_f64(g->Q, a, e, odd, phase, store, g->stream);
        case LUMAGPU_FP32S: return launch_edges_f32s(g->Q, a, e, odd, phase, store, g->stream);
        case LUMAGPU_FP64T: return launch_edges_dual(g->Q, a, e, odd, phase, store, g->stream);
        case LUMAGPU_FP32T: return launch_edges_dual32(g->Q, a, e, odd, phase, store, g->stream);
        default: return launch_edges_f16s(g->Q, a, e, odd, phase, store, g->stream);
    }
}

// _LBM_updateReynolds (GridObj_ops_lbm_optimised.cpp:1313-1321) at the start of
// LBM_multi_opt (:39-42): Re = L_RE * getReynoldsRampCoefficient((t + 1) dt)
// (GridUtils.cpp:1825-1833: 1 - cos(pi t / T) up to T, 1 after), nu = nud2nulbm(1 / Re)
// (GridUnits.h:128-131), omega = 1 / (nu / cs^2 + 0.5)
void update_reynolds(lumagpu_grid *g) {
    const double t = (g->t + 1) * g->d.dt;
    double coef = 1.0;
    if (t <= g->re_ramp) coef = 1.0 - std::cos(3.14159265358979323846 * t / g->re_ramp);
    const double re = g->re * coef;
    const double nu = ((1.0 / re) * g->d.dt) / (g->d.dh * g->d.dh);
    const double cs = 1.0 / std::sqrt(3.0);
    g->d.omega = 1.0 / ((nu / (cs * cs)) + 0.5);
}

// d omega_t / d omega_end for the step update_reynolds sets up: omega_t = 1 / (nu_t / cs^2 + 0.5)
// with nu_t = c / (L_RE coef_t), and omega_end, the omega after the ramp (coef = 1), follows
// L_RE the same way, so d omega_t / d omega_end = omega_t^2 nu_t / (omega_end^2 nu_end)
double reynolds_omega_weight(const lumagpu_grid *g) {
    const double t = (g->t + 1) * g->d.dt;
    double coef = 1.0;
    if (t <= g->re_ramp) coef = 1.0 - std::cos(3.14159265358979323846 * t / g->re_ramp);
    const double cs2 = 1.0 / 3.0, c = g->d.dt / (g->d.dh * g->d.dh);
    const double nt = c / (g->re * coef), ne = c / g->re;
    const double ot = 1.0 / (nt / cs2 + 0.5), oe = 1.0 / (ne / cs2 + 0.5);
    return (ot * ot * nt) / (oe * oe * ne);
}
}  // namespace lumagpu

namespace {

// LUMA-layout rho, u <-> the grid's macro arrays (Duals with zero derivative in the tangent
// form); macro_to_luma takes the values, or with tan the derivatives
hipError_t macro_from_luma(lumagpu_grid *g, const double *rho, const double *u) {
    const dim3 b = cell_block(g->d.N), gr = cell_grid(g->d.N, g->d.M, g->d.K);
    const int N = g->d.N, M = g->d.M, K = g->d.K;
    const bool t = g->melem != sizeof(double);
    if (g->D == 2) {
        if (t) k_macro_from_luma<2, Dual><<<gr, b, 0, g->stream>>>(g->rho, g->u, g->ncell, N, M, K, rho, u);
        else k_macro_from_luma<2><<<gr, b, 0, g->stream>>>(g->rho, g->u, g->ncell, N, M, K, rho, u);
    } else {
        if (t) k_macro_from_luma<3, Dual><<<gr, b, 0, g->stream>>>(g->rho, g->u, g->ncell, N, M, K, rho, u);
        else k_macro_from_luma<3><<<gr, b, 0, g->stream>>>(g->rho, g->u, g->ncell, N, M, K, rho, u);
    }
    return hipGetLastError();
}
hipError_t macro_to_luma(lumagpu_grid *g, double *rho, double *u, bool tan) {
    const dim3 b(256), gr = macro_to_luma_grid(g->d.N, g->d.M, g->d.K);
    const int N = g->d.N, M = g->d.M, K = g->d.K;
    const bool t = g->melem != sizeof(double);
    if (g->D == 2) {
        if (t && tan) k_macro_to_luma<2, Dual, true><<<gr, b, 0, g->stream>>>(g->rho, g->u, g->ncell, N, M, K, rho, u);
        else if (t) k_macro_to_luma<2, Dual><<<gr, b, 0, g->stream>>>(g->rho, g->u, g->ncell, N, M, K, rho, u);
        else k_macro_to_luma<2><<<gr, b, 0, g->stream>>>(g->rho, g->u, g->ncell, N, M, K, rho, u);
    } else {
        if (t && tan) k_macro_to_luma<3, Dual, true><<<gr, b, 0, g->stream>>>(g->rho, g->u, g->ncell, N, M, K, rho, u);
        else if (t) k_macro_to_luma<3, Dual><<<gr, b, 0, g->stream>>>(g->rho, g->u, g->ncell, N, M, K, rho, u);
        else k_macro_to_luma<3><<<gr, b, 0, g->stream>>>(g->rho, g->u, g->ncell, N, M, K, rho, u);
    }
    return hipGetLastError();
}

hipError_t launch_extrap(const lumagpu_grid *g) {
    const StepArgs a = make_args(g);
    double *xr = const_cast<double *>(a.xr);
    switch (g->d.precision) {
        case LUMAGPU_FP64: return launch_aux_f64(kAuxExtrapRight, g->Q, a, nullptr, nullptr, xr, g->parity, 1, g->stream);
        case LUMAGPU_FP32S: return launch_aux_f32s(kAuxExtrapRight, g->Q, a, nullptr, nullptr, xr, g->parity, 1, g->stream);
        case LUMAGPU_FP64T: return launch_aux_dual(kAuxExtrapRight, g->Q, a, nullptr, nullptr, xr, g->parity, 1, g->stream);
        case LUMAGPU_FP32T: return launch_aux_dual32(kAuxExtrapRight, g->Q, a, nullptr, nullptr, xr, g->parity, 1, g->stream);
        default: return launch_aux_f16s(kAuxExtrapRight, g->Q, a, nullptr, nullptr, xr, g->parity, 1, g->stream);
    }
}

// The first half of one grid's LBM_multi_opt once its children have stepped: stream order
// against the child and parent grids, the outlet side buffer, and _LBM_resetForces on a level
// holding IB bodies (:53-57).  Sweep 1's stream, BC and macro happen in the step kernel, which
// end_step launches; what the IB step reads of sweep 1 is recomputed at its supports.
int begin_step(lumagpu_grid *g) {
    if (g->masked && !g->sites_ok)
        return fail(LUMAGPU_ESTATE, "the grid's labels or force were not set to the end: set them again");
    // the outlet side buffer reads this grid's own populations only (the children read them
    // too, but nobody writes them before this grid's step): it runs while the children step
    // the previous step wrote this step's outlet sources unless the state changed since
    if (g->has_outlet && !g->xr_ready) {
        hipError_t e = launch_extrap(g);
        if (e != hipSuccess) return fail(LUMAGPU_EHIP, std::string("outlet launch: ") + hipGetErrorString(e));
    }
    for (lumagpu_grid *c : g->kids) {
        // the child reads this grid's populations, so order the two streams (one stream, as
        // lumagpu_grid_add_child sets up, orders them already)
        if (c->stream != g->stream) {
            HIP_TRY(hipEventRecord(c->ev_done, c->stream));
            HIP_TRY(hipStreamWaitEvent(g->stream, c->ev_done, 0));
        }
        if (c->parity != 0) return fail(LUMAGPU_ESTATE, "child grid out of step with its parent");
    }
    if (g->parent && g->parent->stream != g->stream) {
        // this grid reads the parent's populations: wait for the parent's previous work
        HIP_TRY(hipEventRecord(g->parent->ev_ready, g->parent->stream));
        HIP_TRY(hipStreamWaitEvent(g->stream, g->parent->ev_ready, 0));
    }
    // _LBM_resetForces at the start of the step on a level holding IB bodies (:53-57); with
    // gravity it writes the gravity component from the previous step's rho, and every site
    // then carries a force
    const int has_bodies = ibm_marker_count(g) > 0;
    g->all_forced = (g->gravity_on && has_bodies) ? 1 : 0;
    g->sweep1_zero = (has_bodies && !g->gravity_on) ? 1 : 0;
    if (g->all_forced) {
        const StepArgs ga = make_args(g);
        const double rr = 1.0 / std::pow(2.0, (double)g->d.level);   // GridObj.cpp:54
        const unsigned nb = (unsigned)((g->ncell + 255) / 256);
        if (g->melem == sizeof(double))
            k_gravity_reset<double><<<nb, 256, 0, g->stream>>>(ga, g->force, g->gravity, rr, g->gravity_dir);
        else
            k_gravity_reset<Dual><<<nb, 256, 0, g->stream>>>(ga, g->force, g->gravity, rr, g->gravity_dir);
        HIP_TRY(hipGetLastError());
    }
    return 0;
}

// after a step's kernels: the next step's outlet sources are in the other buffer if they wrote them
void outlet_written(lumagpu_grid *g, const StepArgs &a) {
    if (g->xr_tape) return;   // the caller moves along its tape
    if (a.xr_next) {
        g->xr_sel ^= 1;
        g->xr_ready = 1;
    } else {
        g->xr_ready = 0;
    }
}

// The second half: stream, BC, macro (with the IB force), Guo forcing and BGK collision in one
// pass, the edge/corner and pressure sites around it, then the swap (AA parity) and ++t.
int end_step(lumagpu_grid *g, int subcycle, hipEvent_t e0, hipEvent_t e1) {
    LaunchSpec ls{g->Q, g->masked != 0, g->parity == 0, g->store_macro != 0, g->mlist, g->link, g->nmlist};
    ls.forced = g->all_forced || g->ibm || g->host_forced;
    StepArgs a = make_args(g);
    a.subcycle = subcycle;
    if (g->ib_fold) ibm_fold_args(g, a);
    g->ib_fold = 0;
    if (g->nedge) {
        hipError_t e = launch_edges(g, a, 0);
        if (e != hipSuccess) return fail(LUMAGPU_EHIP, std::string("edge launch: ") + hipGetErrorString(e));
    }
    const bool halo = g->zslab && g->parity == 0;
    if (halo) {
        hipError_t e = launch_zslab(g, a, 0);
        if (e != hipSuccess) return fail(LUMAGPU_EHIP, std::string("halo launch: ") + hipGetErrorString(e));
    }
    if (e0) HIP_TRY(hipEventRecord(e0, g->stream));
    hipError_t e = launch_step(g, ls, a);
    if (e != hipSuccess) return fail(LUMAGPU_EHIP, std::string("step launch: ") + hipGetErrorString(e));
    if (e1) HIP_TRY(hipEventRecord(e1, g->stream));
    outlet_written(g, a);
    if (halo) {
        e = launch_zslab(g, a, 1);
        if (e != hipSuccess) return fail(LUMAGPU_EHIP, std::string("halo launch: ") + hipGetErrorString(e));
    }
    if (g->nedge) {
        e = launch_edges(g, a, 1);
        if (e != hipSuccess) return fail(LUMAGPU_EHIP, std::string("edge launch: ") + hipGetErrorString(e));
    }
    g->parity ^= 1;
    g->t += 1;
    return 0;
}

int apply_step(lumagpu_grid *g, int subcycle, hipEvent_t e0, hipEvent_t e1) {
    if (!g->has_state) return fail(LUMAGPU_ESTATE, "step before the populations were initialised");
    if (g->half) return fail(LUMAGPU_ESTATE, "a split step is open on this grid: finish it with lumagpu_force_collide_swap");
    if (g->re_ramp > 0.0) update_reynolds(g);
    // GridObj_ops_lbm_optimised.cpp:45-49: two sub-steps of each child first, child by child
    for (lumagpu_grid *c : g->kids)
        for (int sc = 0; sc < 2; ++sc)
            if (int r = apply_step(c, sc, nullptr, nullptr)) return r;
    if (int r = begin_step(g)) return r;
    // ObjectManager::ibm_apply between sweep 1 and sweep 2 (:120-121)
    if (g->ibm)
        if (int r = ibm_apply(g, true)) return r;
    return end_step(g, subcycle, e0, e1);
}

}  // namespace

namespace {

// The two-step kernel applies to a grid that the unlabelled periodic kernel steps on its own,
// with the same omega for both steps.  It fuses the local (even) step with the following
// neighbour (odd) step, so it starts at parity 1 (the local step's input layout) and leaves the
// grid there.
bool fused_ready(const lumagpu_grid *g) {
    return g->fuse_shape >= 0 && g->f2 && !g->masked && !g->zslab && !g->parent && g->kids.empty() &&
           ibm_marker_count(g) == 0 && !(g->re_ramp > 0.0) && g->parity == 1 && g->has_state;
}

// two steps (local, then neighbour) in one launch from g->f into g->f2, then the arrays trade places
int fused_pair(lumagpu_grid *g, hipEvent_t e0, hipEvent_t e1) {
    const StepArgs a = make_args(g);
    const bool store = g->store_macro != 0;
    if (e0) HIP_TRY(hipEventRecord(e0, g->stream));
    hipError_t e;
    switch (g->d.precision) {
        case LUMAGPU_FP64: e = launch_fused2_f64(g->fuse_shape, a, g->f2, g->fuse_zc, store, g->stream); break;
        case LUMAGPU_FP32S: e = launch_fused2_f32s(g->fuse_shape, a, g->f2, g->fuse_zc, store, g->stream); break;
        case LUMAGPU_FP16S: e = launch_fused2_f16s(g->fuse_shape, a, g->f2, g->fuse_zc, store, g->stream); break;
        default: return fail(LUMAGPU_EUNSUPPORTED, "no two-step kernel for this precision");
    }
    if (e != hipSuccess) return fail(LUMAGPU_EHIP, std::string("two-step launch: ") + hipGetErrorString(e));
    if (e1) HIP_TRY(hipEventRecord(e1, g->stream));
    std::swap(g->f, g->f2);
    g->t += 2;
    return 0;
}

// Capture two two-step launches (f -> f2 -> f, four steps) into a graph and replay it reps
// times.  Returns 0 when the steps ran, 1 when the capture was not possible (nothing ran, host
// state restored), or an error code.
int run_fused_graph(lumagpu_grid *g, int reps) {
    const int t0 = g->t;
    void *const f0 = g->f, *const f20 = g->f2;
    if (hipStreamBeginCapture(g->stream, hipStreamCaptureModeThreadLocal) != hipSuccess) {
        (void)hipGetLastError();
        return 1;
    }
    int rc = 0;
    for (int k = 0; k < 2 && !rc; ++k) rc = fused_pair(g, nullptr, nullptr);
    hipGraph_t graph = nullptr;
    const hipError_t ec = hipStreamEndCapture(g->stream, &graph);
    g->t = t0;
    g->f = f0;
    g->f2 = f20;
    if (rc || ec != hipSuccess) {
        if (graph) (void)hipGraphDestroy(graph);
        (void)hipGetLastError();
        return rc ? rc : 1;
    }
    hipGraphExec_t exec = nullptr;
    if (hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0) != hipSuccess) {
        (void)hipGraphDestroy(graph);
        (void)hipGetLastError();
        return 1;
    }
    hipError_t e = hipSuccess;
    for (int r = 0; r < reps && e == hipSuccess; ++r) e = hipGraphLaunch(exec, g->stream);
    (void)hipGraphExecDestroy(exec);
    (void)hipGraphDestroy(graph);
    if (e != hipSuccess) return fail(LUMAGPU_EHIP, std::string("graph launch: ") + hipGetErrorString(e));
    g->t += 4 * reps;
    return 0;
}

// Small 2D grids take several steps per launch (k_multi2d): one level, no bodies, nothing that
// changes from step to step, and site types whose sources the window holds.  2^18 cells: above,
// a step fills the chip by itself, and the window's repeated cells cost more than launches.  FP64 and
// FP32-shifted storage: the kernel is built for these two, FP16-shifted grids of this size step singly.
bool multi_ok(const lumagpu_grid *g) {
    return !g->fuse_off && g->Q == 9 && (g->d.precision == LUMAGPU_FP64 || g->d.precision == LUMAGPU_FP32S) && !g->parent &&
           g->kids.empty() && ibm_marker_count(g) == 0 && !g->gravity_on && !(g->ramp_time > 0.0) &&
           !(g->re_ramp > 0.0) && g->nedge == 0 && g->simple_types && g->ncell <= (size_t(1) << 18) && g->has_state && (!g->masked || g->sites_ok);
}

// Fewer steps than these go one per launch: the first launches of a run follow each other every 3 us, and
// a window's start (its loads, 9 planes through LDS) costs 2 to 9 of them.  run(n) with the wait after it,
// single / several per launch, us: box FP32 48^2 n = 2 16.6 / 17.5, 4 22.1 / 18.9, 512^2 n = 2 22.7 / 26.5, 4
// 35.4 / 31.6; box FP64 256^2 n = 2 19.7 / 24.5, 4 29.3 / 29.5, 512^2 n = 2 30 / 38, 4 51 / 49; lid FP64 320^2
// n = 2 25.0 / 26.3, 4 39.8 / 33.1.  FP64 windows of a small box, whose single steps are launches and little
// else: 48^2 n = 4 22.4 / 25.6, 6 28.3 / 29.8, 128^2 n = 4 24.0 / 26.9, 6 30.8 / 30.4; from 8 steps on single
// ones are replayed as a graph, 48^2 54 / 33.
int multi_min(const lumagpu_grid *g) {
    return g->d.precision == LUMAGPU_FP64 && !g->masked && multi2d_blocks(g->d.N, g->d.M, 6) <= 64 ? 8 : 4;
}

// up to n steps from the post-local layout, as many as whole launches take; *done: steps run
int run_multi(lumagpu_grid *g, int n, int *done) {
    *done = 0;
    if (!f2_ensure(g)) return 0;   // one step per launch needs no second array
    const F2Use use(g);
    // begin_step's state for a grid without bodies
    g->all_forced = g->sweep1_zero = 0;
    while (n - *done >= multi_min(g)) {
        const int H = plan_multi2d(g->d.N, g->d.M, n - *done, g->d.precision == LUMAGPU_FP64);
        StepArgs a = make_args(g);
        if (!g->masked) {   // flag bytes that other calls made are not this step's
            a.flags = nullptr;
            a.link = nullptr;
        }
        const hipError_t e = g->d.precision == LUMAGPU_FP64 ? launch_multi2d_f64(a, g->f2, H, g->store_macro, g->stream)
                                                            : launch_multi2d_f32s(a, g->f2, H, g->store_macro, g->stream);
        if (e != hipSuccess) return fail(LUMAGPU_EHIP, std::string("multi-step launch: ") + hipGetErrorString(e));
        std::swap(g->f, g->f2);
        g->t += H;
        *done += H;
    }
    return 0;
}

// Two steps per launch on large D3Q19 grids in FP32-shifted storage (fused_kernels.hpp): one level, a
// step that is the same kernels every time (no gravity reset, no Reynolds ramp), site types of the
// list kernels, bodies rigid and settled (their supports flagged), outlet sources written by the
// step.  us per step, single -> pairs: periodic boxes 32^3 10.7 -> 3.4, 64^3 9.4 -> 6.5, 128^3 53 -> 37,
// 160^3 108 -> 77.  Labelled grids have three launches a pair and gain later: walls with a set force
// 48^3 11.3 -> 13.1, 64^3 14.2 -> 14.9, 65^3 22.9 -> 20.5, 96^3 42 -> 29, 160^3 129 -> 106.  Above 2^18 cells:
// there both take the same on rows of whole 64s (64 x 64 x 66 15.9 -> 15.5, 128 x 64 x 33 15.8 -> 15.8,
// 192 x 48 x 29 15.9 -> 16.3, 512 x 32 x 17 16.4 -> 16.5; rows of 1024, 15.9 -> 17.7, are the worst) and
// pairs less on others (300 x 30 x 30 21.3 -> 17.5).
constexpr size_t kPairMin = size_t(1) << 15, kPairMinLabelled = (size_t(1) << 18) + 1;
bool pair_ok(const lumagpu_grid *g) {
    if (g->fuse_off || g->Q != 19 || g->d.precision != LUMAGPU_FP32S || g->parent || !g->kids.empty() || g->zslab ||
        g->gravity_on || g->re_ramp > 0.0 || !g->has_state || g->ncell < (g->masked ? kPairMinLabelled : kPairMin) ||
        g->ps * g->elem >= (size_t(1) << 32))
        return false;
    if (g->has_outlet && !g->xr_fold) return false;
    if (g->masked && (!g->pair_types || !g->sites_ok)) return false;
    return !ibm_has_flexible(g) && !(g->host_forced && ibm_marker_count(g) > 0);
}

// the deep cells and the lists around them, from the flags on the device; LUMAGPU_ENOMEM where they do
// not fit
int pair_sets(lumagpu_grid *g) {
    // deep are cells by their types and, with bodies, by which sites these flag
    const uint64_t key[2] = {g->types_version, ibm_marker_count(g) > 0 ? g->flags_version : 0};
    if (!g->masked || (g->pair_key[0] == key[0] && g->pair_key[1] == key[1])) return 0;
    g->pair_key[0] = 0;
    const size_t nw = (g->ncell + 31) / 32 + 1;   // a whole pair of words at the end
    struct Buf {
        uint32_t *p = nullptr;
        ~Buf() { (void)hipFree(p); }
    } rest, near;
    if ((!g->pair_deep && dev_malloc(&g->pair_deep, nw * 4) != hipSuccess) ||
        dev_malloc(&rest.p, nw * 4) != hipSuccess || dev_malloc(&near.p, nw * 4) != hipSuccess)
        return fail(LUMAGPU_ENOMEM, "site set allocation failed");
    const StepArgs a = make_args(g);
    const unsigned nb = (unsigned)((g->ncell + 255) / 256);
    k_deep_bits<19><<<nb, 256, 0, g->stream>>>(a, ibm_marker_count(g) > 0, g->pair_deep, rest.p);
    k_near_bits<19><<<nb, 256, 0, g->stream>>>(a, g->pair_deep, rest.p, near.p);
    HIP_TRY(hipGetLastError());
    const size_t words = (g->ncell + 31) / 32;
    std::vector<uint32_t> hr(words), hn(words);
    HIP_TRY(hipMemcpyAsync(hr.data(), rest.p, words * 4, hipMemcpyDeviceToHost, g->stream));
    HIP_TRY(hipMemcpyAsync(hn.data(), near.p, words * 4, hipMemcpyDeviceToHost, g->stream));
    HIP_TRY(hipStreamSynchronize(g->stream));
    std::vector<int> cells;
    auto take = [&](const std::vector<uint32_t> &m) {
        const size_t before = cells.size();
        for (size_t w = 0; w < words; ++w)
            for (uint32_t b = m[w]; b; b &= b - 1) cells.push_back((int)(32 * w + __builtin_ctz(b)));
        return (int)(cells.size() - before);
    };
    g->n_near = take(hn);
    g->n_rest = take(hr);
    (void)hipFree(g->pair_cells);
    (void)hipFree(g->pair_links);
    g->pair_cells = nullptr;
    g->pair_links = nullptr;
    if (!cells.empty()) {
        if (dev_malloc(&g->pair_cells, cells.size() * sizeof(int)) != hipSuccess ||
            dev_malloc(&g->pair_links, cells.size() * sizeof(uint64_t)) != hipSuccess)
            return fail(LUMAGPU_ENOMEM, "site list allocation failed");
        HIP_TRY(hipMemcpyAsync(g->pair_cells, cells.data(), cells.size() * sizeof(int), hipMemcpyHostToDevice, g->stream));
        k_links<19><<<(unsigned)((cells.size() + 255) / 256), 256, 0, g->stream>>>(
            g->flags, g->d.N, g->d.M, g->d.K, g->d.regularised, g->pair_cells, cells.size(), g->pair_links);
        HIP_TRY(hipGetLastError());
        HIP_TRY(hipStreamSynchronize(g->stream));
    }
    g->pair_key[0] = key[0];
    g->pair_key[1] = key[1];
    return 0;
}

// One half of a pair for the listed sites: what apply_step does around its step kernel, the even half from
// f into f2 and before the deep cells, the odd half in place after them.
int pair_half(lumagpu_grid *g, bool odd, PairPlan plan) {
    if (int r = begin_step(g)) return r;
    if (g->ibm)
        if (int r = ibm_apply(g, true)) return r;
    StepArgs a = make_args(g);
    if (g->ib_fold) ibm_fold_args(g, a);
    g->ib_fold = 0;
    if (!odd) a.fo = g->f2;
    const bool store = g->store_macro != 0;
    auto check = [](hipError_t e) {
        return e == hipSuccess ? 0 : fail(LUMAGPU_EHIP, std::string("two-step launch: ") + hipGetErrorString(e));
    };
    if (g->nedge)
        if (int r = check(launch_edges(g, a, 0))) return r;
    if (g->masked) {
        const int *cells = odd ? g->pair_cells + g->n_near : g->pair_cells;
        const uint64_t *links = odd ? g->pair_links + g->n_near : g->pair_links;
        if (int r = check(launch_list_f32s(a, odd, odd && store, cells, links, odd ? g->n_rest : g->n_near, g->stream)))
            return r;
    }
    if (g->nedge)
        if (int r = check(launch_edges(g, a, 1))) return r;
    outlet_written(g, a);
    if (!odd) {
        if (int r = check(launch_pair_f32s(a, g->f2, plan, g->masked ? g->pair_deep : nullptr, g->host_forced != 0, store,
                                           g->stream)))
            return r;
        std::swap(g->f, g->f2);
    }
    g->parity ^= 1;
    g->t += 1;
    return 0;
}

// up to n steps from the post-neighbour layout, two at a time; *done: steps run
int run_pairs(lumagpu_grid *g, int n, int *done) {
    *done = 0;
    if (!f2_ensure(g)) return 0;
    const F2Use use(g);
    if (const int r = pair_sets(g)) {
        if (r != LUMAGPU_ENOMEM) return r;
        (void)hipGetLastError();
        return 0;   // single steps need no sets
    }
    if (g->masked && !g->pair_synced)
        HIP_TRY(hipMemcpyAsync(g->f2, g->f, g->ps * g->Q * g->elem, hipMemcpyDeviceToDevice, g->stream));
    g->pair_synced = 1;
    const PairPlan plan = plan_pair(g->d.N, g->d.M, g->d.K);
    while (n - *done >= 2) {
        for (bool odd : {false, true})
            if (int r = pair_half(g, odd, plan)) return r;
        *done += 2;
    }
    return 0;
}

// no host work inside a step anywhere in the hierarchy (flexible bodies download forces and
// run the FEM on the host every step)
bool graph_ok(const lumagpu_grid *g) {
    bool ok = !g->parent;
    for_each_level(g, [&](const lumagpu_grid *x) {
        if (ibm_has_flexible(x)) ok = false;
        if (x->ramp_time > 0.0) ok = false;   // the ramp factors change every step
        if (x->re_ramp > 0.0) ok = false;     // so does omega under a Reynolds ramp
        if (x->fuse_shape >= 0) ok = false;   // the two-step kernel alternates two arrays
    });
    return ok;
}

void add_time(lumagpu_grid *g, int steps) {
    g->t += steps;
    for (lumagpu_grid *k : g->kids) add_time(k, 2 * steps);
}

// Everything the two captured steps pass to their kernels, level by level: while it stays the
// same, the graph captured from them is the graph a new capture would give.
std::vector<uint8_t> graph_key(lumagpu_grid *g) {
    std::vector<uint8_t> key;
    auto put = [&](const void *p, size_t n) {
        const uint8_t *b = static_cast<const uint8_t *>(p);
        key.insert(key.end(), b, b + n);
    };
    for_each_level(g, [&](lumagpu_grid *x) {
        const StepArgs a = make_args(x);
        put(&a, sizeof a);
        const int misc[] = {x->Q, x->masked, x->store_macro, x->nmlist, x->nedge, x->zslab, x->has_outlet,
                            x->gravity_on, x->gravity_dir, (int)x->kids.size(), x->parity, (int)x->d.precision,
                            x->d.level, x->d.regularised, x->xr_sel, x->xr_ready, x->xr_fold,
                            x->host_forced, x->ibm != nullptr};
        put(misc, sizeof misc);
        const void *ptrs[] = {x->mlist, x->link, x->edge, x->erho, x->stream, x->force};
        put(ptrs, sizeof ptrs);
        put(&x->gravity, sizeof x->gravity);
        ibm_graph_key(x, key);
    });
    return key;
}

// Capture two steps of g (and its descendants) into a graph and launch it reps times; the
// executable graph is kept and launched again by later runs while its key holds.
// Returns 0 when the steps ran, 1 when the capture was not possible (nothing ran, host state
// restored), or an error code.
int run_graph(lumagpu_grid *g, int reps) {
    std::vector<int> t0;
    for_each_level(g, [&](lumagpu_grid *x) { t0.push_back(x->t); });
    auto restore = [&]() {
        size_t i = 0;
        for_each_level(g, [&](lumagpu_grid *x) {
            x->t = t0[i++];
            x->parity = 0;
        });
    };
    std::vector<uint8_t> key = graph_key(g);
    if (!g->gexec || key != g->gkey) {
        if (hipStreamBeginCapture(g->stream, hipStreamCaptureModeThreadLocal) != hipSuccess) {
            (void)hipGetLastError();
            return 1;
        }
        int rc = 0;
        for (int k = 0; k < 2 && !rc; ++k) rc = apply_step(g, 0, nullptr, nullptr);
        hipGraph_t graph = nullptr;
        const hipError_t ec = hipStreamEndCapture(g->stream, &graph);
        restore();
        if (rc || ec != hipSuccess) {
            if (graph) (void)hipGraphDestroy(graph);
            (void)hipGetLastError();
            return rc ? rc : 1;
        }
        hipGraphExec_t exec = nullptr;
        const hipError_t ei = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
        (void)hipGraphDestroy(graph);
        if (ei != hipSuccess) {
            (void)hipGetLastError();
            return 1;
        }
        if (g->gexec) (void)hipGraphExecDestroy(g->gexec);
        g->gexec = exec;
        // the key after the capture: its host-side effects (IB supports settling) are in it
        g->gkey = graph_key(g);
    }
    hipGraphExec_t exec = g->gexec;
    // the graph runs on g's stream: order it after whatever the descendants' streams hold,
    // and the descendants' later work after it
    hipError_t e = hipSuccess;
    for_each_level(g, [&](lumagpu_grid *x) {
        if (x->stream == g->stream || e != hipSuccess) return;
        e = hipEventRecord(x->ev_done, x->stream);
        if (e == hipSuccess) e = hipStreamWaitEvent(g->stream, x->ev_done, 0);
    });
    for (int r = 0; r < reps && e == hipSuccess; ++r) e = hipGraphLaunch(exec, g->stream);
    for_each_level(g, [&](lumagpu_grid *x) {
        if (x->stream == g->stream || e != hipSuccess) return;
        e = hipEventRecord(g->ev_ready, g->stream);
        if (e == hipSuccess) e = hipStreamWaitEvent(x->stream, g->ev_ready, 0);
    });
    if (e != hipSuccess) return fail(LUMAGPU_EHIP, std::string("graph launch: ") + hipGetErrorString(e));
    add_time(g, 2 * reps);
    return 0;
}

}  // namespace

namespace {
// Per-block partial sums of lumagpu_moments_noalloc: device memory fixed at load time, one copy
// per GPU, at most kScratchBlocks row blocks.  Host code never hands the symbol itself to a
// kernel (in host code it is a stand-in, not a device address): it takes each GPU's address
// from hipGetSymbolAddress once, with that GPU current, and passes that.
constexpr size_t kScratchBlocks = size_t(1) << 18;
static __device__ __align__(256) double scratch[kScratchBlocks * kMomentCount];
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
double *g_scratch_ptr[kMaxDevices] = {};

int scratch_on(int device, double **out) {
    if (device < 0 || device >= kMaxDevices) return fail(LUMAGPU_EINVAL, "device ordinal out of range");
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_ptr[device]) {
        void *p = nullptr;
        HIP_TRY(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        if (!p) return fail(LUMAGPU_EHIP, "hipGetSymbolAddress returned no address for the reduction scratch");
        g_scratch_ptr[device] = static_cast<double *>(p);
    }
    *out = g_scratch_ptr[device];
    return 0;
}
}  // namespace

namespace lumagpu {
int step_grid(lumagpu_grid *g, int subcycle) { return apply_step(g, subcycle, nullptr, nullptr); }
// the device table of g's refined regions, rewritten whenever the list changes
int upload_kids(lumagpu_grid *g) {
    (void)hipStreamSynchronize(g->stream);   // no queued step reads the old table
    (void)hipFree(g->d_kids);
    g->d_kids = nullptr;
    if (g->kids.empty()) return 0;
    std::vector<ChildRef> h(g->kids.size());
    for (size_t i = 0; i < g->kids.size(); ++i) {
        const lumagpu_grid *c = g->kids[i];
        ChildRef &r = h[i];
        r.f = c->f;
        r.ps = c->ps;
        r.nx = c->d.N;
        r.ny = c->d.M;
        r.nz = c->d.K;
        for (int a = 0; a < 3; ++a) {
            r.lo[a] = c->d.coarse_lims[2 * a];
            r.hi[a] = c->d.coarse_lims[2 * a + 1];
        }
        r.rho = c->rho;
        r.u = c->u;
        r.ncell = c->ncell;
    }
    if (dev_malloc(&g->d_kids, h.size() * sizeof(ChildRef)) != hipSuccess)
        return fail(LUMAGPU_ENOMEM, "refined-region table allocation failed");
    HIP_TRY(hipMemcpy(g->d_kids, h.data(), h.size() * sizeof(ChildRef), hipMemcpyHostToDevice));
    return 0;
}
namespace {
// f_v of the listed cells from the post-local layout (population v of a cell in its slot
// opp(v)), into out[v * n + k]
template <class W, int Q>
__global__ void k_copy_slots(const W *f, size_t ps, const int *cells, int n, W *out) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    for (int v = 0; v < Q; ++v) out[(size_t)v * n + k] = f[(size_t)Lattice<Q>::opp(v) * ps + (size_t)cells[k]];
}
struct Elem16 {
    uint64_t a, b;
};
template <class W>
void copy_slots(const lumagpu_grid *g) {
    const unsigned nb = (unsigned)((g->nstale + 127) / 128);
    const W *f = static_cast<const W *>(g->f);
    W *out = static_cast<W *>(g->stale);
    if (g->Q == 9) k_copy_slots<W, 9><<<nb, 128, 0, g->stream>>>(f, g->ps, g->stale_cells, g->nstale, out);
    else k_copy_slots<W, 19><<<nb, 128, 0, g->stream>>>(f, g->ps, g->stale_cells, g->nstale, out);
}
}  // namespace

int capture_stale(lumagpu_grid *g) {
    if (!g->nstale || !g->has_state) return 0;
    if (g->parity != 0) return fail(LUMAGPU_ESTATE, "refined-site capture needs the post-local layout");
    switch (g->elem) {
        case 2: copy_slots<uint16_t>(g); break;
        case 4: copy_slots<uint32_t>(g); break;
        case 8: copy_slots<uint64_t>(g); break;
        case 16: copy_slots<Elem16>(g); break;
        default: return fail(LUMAGPU_EUNSUPPORTED, "unexpected population element size");
    }
    HIP_TRY(hipGetLastError());
    return 0;
}

// refined sites read by a site that does not coalesce (anything but TL2F, solid or refined),
// with the periodic wrap of the step kernels
static int build_stale(lumagpu_grid *g, bool *fresh) {
    const int N = g->d.N, M = g->d.M, K = g->d.K;
    auto ty = [&](int i, int j, int k) {
        i = (i + N) % N; j = (j + M) % M; k = (k + K) % K;
        return g->hflags[(size_t)i + (size_t)N * ((size_t)j + (size_t)M * k)] & kTypeMask;
    };
    std::vector<int> idx(g->ncell, -1), cells;
    for (int k = 0; k < K; ++k)
        for (int j = 0; j < M; ++j)
            for (int i = 0; i < N; ++i) {
                const int t = ty(i, j, k);
                if (t == kTL2F || t == kRefined || t == kSolid) continue;
                // an outlet site's source two cells left (its side buffer, :246-251)
                if (t == kExtrapRight && i >= 2 && ty(i - 2, j, k) == kRefined) {
                    const size_t c = (size_t)(i - 2) + (size_t)N * ((size_t)j + (size_t)M * k);
                    if (idx[c] < 0) {
                        idx[c] = (int)cells.size();
                        cells.push_back((int)c);
                    }
                }
                for (int dk = (g->D == 3 ? -1 : 0); dk <= (g->D == 3 ? 1 : 0); ++dk)
                    for (int dj = -1; dj <= 1; ++dj)
                        for (int di = -1; di <= 1; ++di) {
                            if (ty(i + di, j + dj, k + dk) != kRefined) continue;
                            const int ii = (i + di + N) % N, jj = (j + dj + M) % M, kk = (k + dk + K) % K;
                            const size_t c = (size_t)ii + (size_t)N * ((size_t)jj + (size_t)M * kk);
                            if (idx[c] < 0) {
                                idx[c] = (int)cells.size();
                                cells.push_back((int)c);
                            }
                        }
            }
    // the same sites as before: keep what was captured
    *fresh = cells != g->stale_list;
    if (!*fresh) return 0;
    (void)hipStreamSynchronize(g->stream);
    (void)hipFree(g->stale);
    (void)hipFree(g->stale_idx);
    (void)hipFree(g->stale_cells);
    g->stale = nullptr;
    g->stale_idx = g->stale_cells = nullptr;
    g->nstale = 0;
    g->stale_list.clear();
    if (cells.empty()) return 0;
    if (dev_malloc(&g->stale, (size_t)g->Q * cells.size() * g->elem) != hipSuccess ||
        dev_malloc(&g->stale_idx, g->ncell * sizeof(int)) != hipSuccess ||
        dev_malloc(&g->stale_cells, cells.size() * sizeof(int)) != hipSuccess)
        return fail(LUMAGPU_ENOMEM, "refined-site buffer allocation failed");
    HIP_TRY(hipMemcpy(g->stale_idx, idx.data(), g->ncell * sizeof(int), hipMemcpyHostToDevice));
    HIP_TRY(hipMemcpy(g->stale_cells, cells.data(), cells.size() * sizeof(int), hipMemcpyHostToDevice));
    g->nstale = (int)cells.size();
    g->stale_list = std::move(cells);
    return 0;
}

// Large labelled grids step in two launches: k_aa_plain over the grid for the plain sites
// (fluid, every stencil neighbour fluid or TL2F: the k_plain_bits predicate) and the labelled
// kernel over the list of the other sites it steps.  Small grids, whose steps are launch-bound,
// keep one launch.
constexpr size_t kSplitMinCells = size_t(1) << 20;
static bool split_sites(const lumagpu_grid *g) { return g->ncell >= kSplitMinCells && !g->zslab; }
static int build_mlist(lumagpu_grid *g) {
    if (!split_sites(g)) return 0;
    const int N = g->d.N, M = g->d.M, K = g->d.K;
    auto ty = [&](int i, int j, int k) {
        i = (i + N) % N; j = (j + M) % M; k = (k + K) % K;
        return g->hflags[(size_t)i + (size_t)N * ((size_t)j + (size_t)M * k)] & kTypeMask;
    };
    std::vector<int> list;
    for (int k = 0; k < K; ++k)
        for (int j = 0; j < M; ++j)
            for (int i = 0; i < N; ++i) {
                const size_t c = (size_t)i + (size_t)N * ((size_t)j + (size_t)M * k);
                const unsigned fl = g->hflags[c];
                const int t = fl & kTypeMask;
                // the sites k_aa_masked leaves alone
                if (t == kSolid || t == kRefined || (!g->d.regularised && t == kVelocity)) continue;
                if (t == kPressure || (t == kVelocity && ((fl >> kNormalShift) & 7) == kNormalEdge)) continue;
                bool plain = t == kFluid;
                for (int dk = (g->D == 3 ? -1 : 0); plain && dk <= (g->D == 3 ? 1 : 0); ++dk)
                    for (int dj = -1; plain && dj <= 1; ++dj)
                        for (int di = -1; plain && di <= 1; ++di) {
                            if (g->D == 3 && di != 0 && dj != 0 && dk != 0) continue;   // D3Q19: no corners
                            const int tn = ty(i + di, j + dj, k + dk);
                            plain = tn == kFluid || tn == kTL2F;
                        }
                if (!plain) list.push_back((int)c);
            }
    if (!list.empty()) {
        if (dev_malloc(&g->mlist, list.size() * sizeof(int)) != hipSuccess)
            return fail(LUMAGPU_ENOMEM, "site list allocation failed");
        HIP_TRY(hipMemcpy(g->mlist, list.data(), list.size() * sizeof(int), hipMemcpyHostToDevice));
    }
    g->nmlist = (int)list.size();
    return 0;
}

// link words of the sites k_aa_masked or k_aa_masked_list steps, from the flags on the device
static int build_links(lumagpu_grid *g) {
    const size_t n = g->nmlist >= 0 ? (size_t)g->nmlist : g->ncell;
    if (n != g->link_n) {
        // a buffer of the same length is written over in stream order: on a 48 x 48 grid new labels take
        // 80 us with it, 121 with a wait, a free and an allocation
        (void)hipStreamSynchronize(g->stream);
        (void)hipFree(g->link);
        g->link = nullptr;
        g->link_n = 0;
        if (n > 0 && dev_malloc(&g->link, n * sizeof(uint64_t)) != hipSuccess)
            return fail(LUMAGPU_ENOMEM, "link word allocation failed");
        g->link_n = n;
    }
    if (n == 0) return 0;
    const unsigned nb = (unsigned)((n + 255) / 256);
    const int *cells = g->nmlist >= 0 ? g->mlist : nullptr;
    if (g->Q == 9)
        k_links<9><<<nb, 256, 0, g->stream>>>(g->flags, g->d.N, g->d.M, g->d.K, g->d.regularised, cells, n, g->link);
    else
        k_links<19><<<nb, 256, 0, g->stream>>>(g->flags, g->d.N, g->d.M, g->d.K, g->d.regularised, cells, n, g->link);
    HIP_TRY(hipGetLastError());
    return 0;
}

// The site list, its link words and the captured refined sites, from the flag bytes without the force
// bit and from which of the two layouts the grid steps in (one link word per cell, or per entry of
// the list).  Kept while both are the same.  sites_ok is 0 from here on until all of it is there:
// a step would read a list of one state with the link words of another, so it is refused meanwhile.
static int build_sites(lumagpu_grid *g, bool had) {
    std::vector<uint8_t> types(g->ncell);
    for (size_t c = 0; c < g->ncell; ++c) types[c] = g->hflags[c] & ~kForcedBit;
    if (had && types == g->site_types && split_sites(g) == (g->nmlist >= 0)) {
        g->sites_ok = 1;
        return 0;
    }
    ++g->types_version;
    g->pair_synced = 0;   // other cells may be the ones that never step
    if (g->mlist) {
        (void)hipStreamSynchronize(g->stream);
        (void)hipFree(g->mlist);
    }
    g->mlist = nullptr;
    g->nmlist = -1;
    if (int r = build_mlist(g)) return r;
    if (int r = build_links(g)) return r;
    bool fresh = false;
    if (int r = build_stale(g, &fresh)) return r;
    g->site_types = std::move(types);
    g->sites_ok = 1;
    return fresh ? capture_stale(g) : 0;
}

// the device's flag bytes and plain-site bitmap
static int alloc_flags(lumagpu_grid *g) {
    if (!g->flags && dev_malloc(&g->flags, g->ncell) != hipSuccess) {
        g->flags = nullptr;
        return fail(LUMAGPU_ENOMEM, "flag array allocation failed");
    }
    if (!g->plain && dev_malloc(&g->plain, (g->ncell + 31) / 32 * sizeof(uint32_t)) != hipSuccess) {
        g->plain = nullptr;
        return fail(LUMAGPU_ENOMEM, "plain-site bitmap allocation failed");
    }
    return 0;
}

int upload_flags(lumagpu_grid *g) {
    ++g->flags_version;
    if (g->hflags.size() != g->ncell) return fail(LUMAGPU_ESTATE, "host flag array does not cover the grid");
    if (int r = alloc_flags(g)) return r;
    // from here until the list and the link words are whole a step would read parts of two states:
    // begin_step refuses it
    const bool had = g->sites_ok != 0;
    g->sites_ok = 0;
    const size_t nw = (g->ncell + 31) / 32;
    HIP_TRY(hipMemcpyAsync(g->flags, g->hflags.data(), g->ncell, hipMemcpyHostToDevice, g->stream));
    g->simple_types = std::all_of(g->hflags.begin(), g->hflags.end(), [](uint8_t f) {
        const int t = f & kTypeMask;
        return t == kSolid || t == kFluid || t == kVelocity;
    });
    g->pair_types = std::all_of(g->hflags.begin(), g->hflags.end(), [](uint8_t f) {
        const int t = f & kTypeMask;
        return t == kSolid || t == kFluid || t == kVelocity || t == kPressure || t == kExtrapRight;
    });
    g->host_forced = std::any_of(g->hflags.begin(), g->hflags.end(), [](uint8_t f) { return (f & kForcedBit) != 0; });
    const unsigned nb = (unsigned)((nw + 255) / 256);
    if (g->Q == 9) k_plain_bits<9><<<nb, 256, 0, g->stream>>>(g->flags, g->d.N, g->d.M, g->d.K, g->ncell, g->plain);
    else k_plain_bits<19><<<nb, 256, 0, g->stream>>>(g->flags, g->d.N, g->d.M, g->d.K, g->ncell, g->plain);
    HIP_TRY(hipGetLastError());
    return build_sites(g, had);
}
hipError_t outlet_prepass(const lumagpu_grid *g) { return launch_extrap(g); }
}  // namespace lumagpu

extern "C" {

const char *lumagpu_last_error(void) { return g_last_error.c_str(); }
int lumagpu_abi_version(void) { return LUMAGPU_ABI_VERSION; }

int lumagpu_grid_create(const lumagpu_grid_desc *desc, lumagpu_grid **out) {
    if (!desc || !out) return fail(LUMAGPU_EINVAL, "null descriptor or output pointer");
    *out = nullptr;
    const lumagpu_grid_desc &d = *desc;
    if (!((d.dims == 2 && d.Q == 9) || (d.dims == 3 && d.Q == 19)))
        return fail(LUMAGPU_EUNSUPPORTED, "lattice must be D2Q9 or D3Q19");
    if (d.N < 3 || d.M < 3 || d.K < 1 || (d.dims == 2 && d.K != 1) || (d.dims == 3 && d.K < 3))
        return fail(LUMAGPU_EINVAL, "grid extents too small (need >= 3 per active dimension; K = 1 in 2D)");
    if (d.precision < LUMAGPU_FP64 || d.precision > LUMAGPU_FP32T)
        return fail(LUMAGPU_EINVAL, "unknown precision");
    // GridObj_init_grids.cpp:353-356
    if (!(d.omega > 0.0) || d.omega >= 2.0)
        return fail(LUMAGPU_EPHYS, "LBM relaxation frequency omega too large (must be 0 < omega < 2)");
    if (d.level < 0) return fail(LUMAGPU_EINVAL, "negative refinement level");
    // the shifted forms store f - w with the reference density 1 (their collision is written
    // for it); the plain forms do not use rho0
    if ((d.precision == LUMAGPU_FP32S || d.precision == LUMAGPU_FP16S || d.precision == LUMAGPU_FP32T) &&
        d.rho0 != 1.0)
        return fail(LUMAGPU_EINVAL, "the shifted forms use the reference density rho0 = 1");

    lumagpu_grid *g = new lumagpu_grid();
    g->d = d;
    g->Q = d.Q;
    g->D = d.dims;
    g->ncell = (size_t)d.N * d.M * d.K;
    g->ps = (g->ncell + 255) / 256 * 256 + kPlanePad;
    const bool tan = d.precision == LUMAGPU_FP64T || d.precision == LUMAGPU_FP32T;
    g->elem = d.precision == LUMAGPU_FP64T                                  ? 16
              : (d.precision == LUMAGPU_FP64 || d.precision == LUMAGPU_FP32T) ? 8
              : d.precision == LUMAGPU_FP32S                                 ? 4
                                                                             : 2;
    g->melem = tan ? 16 : 8;
    auto cleanup = [&](int code, const std::string &m) {
        lumagpu_grid_destroy(g);
        return fail(code, m);
    };
    if (hipGetDevice(&g->device) != hipSuccess) return cleanup(LUMAGPU_EHIP, "hipGetDevice failed");
    if (hipStreamCreateWithFlags(&g->own_stream, hipStreamNonBlocking) != hipSuccess)
        return cleanup(LUMAGPU_EHIP, "hipStreamCreate failed");
    g->stream = g->own_stream;
    if (hipEventCreateWithFlags(&g->ev_done, hipEventDisableTiming) != hipSuccess ||
        hipEventCreateWithFlags(&g->ev_ready, hipEventDisableTiming) != hipSuccess)
        return cleanup(LUMAGPU_EHIP, "hipEventCreate failed");
    if (dev_malloc(&g->f, g->ps * g->Q * g->elem) != hipSuccess)
        return cleanup(LUMAGPU_ENOMEM, "population array allocation failed");
    if (dev_malloc(&g->rho, g->ncell * g->melem) != hipSuccess ||
        dev_malloc(&g->u, g->ncell * g->D * g->melem) != hipSuccess)
        return cleanup(LUMAGPU_ENOMEM, "macro array allocation failed");
    if (dev_malloc(&g->uin, 3 * (size_t)d.M * sizeof(double)) != hipSuccess)
        return cleanup(LUMAGPU_ENOMEM, "inlet array allocation failed");
    if (hipMemsetAsync(g->uin, 0, 3 * (size_t)d.M * sizeof(double), g->stream) != hipSuccess)
        return cleanup(LUMAGPU_EHIP, "inlet array clear failed");
    const dim3 gr = cell_grid(d.N, d.M, d.K);
    const size_t nblocks = (size_t)gr.x * gr.y * gr.z;
    if (dev_malloc(&g->partials, nblocks * kMomentCount * sizeof(double)) != hipSuccess ||
        dev_malloc(&g->moments_out, kMomentCount * sizeof(double)) != hipSuccess)
        return cleanup(LUMAGPU_ENOMEM, "reduction buffers allocation failed");
    if (d.forced) {
        if (dev_malloc(&g->force, g->ncell * g->D * g->melem) != hipSuccess)
            return cleanup(LUMAGPU_ENOMEM, "force array allocation failed");
        if (hipMemsetAsync(g->force, 0, g->ncell * g->D * g->melem, g->stream) != hipSuccess)
            return cleanup(LUMAGPU_EHIP, "force array clear failed");
    }
    host_copy_grid_added();
    g->counted = 1;
    *out = g;
    return 0;
}

int lumagpu_grid_destroy(lumagpu_grid *g) {
    if (!g) return 0;
    if (g->stream) (void)hipStreamSynchronize(g->stream);
    if (g->counted) host_copy_grid_gone();
    (void)hipHostFree(g->pin);
    (void)hipFree(g->f);
    {
        std::lock_guard<std::mutex> lock(g_f2_grids_mu);
        scratch_set(g, 0);
    }
    (void)hipFree(g->f2);
    for (auto &b : g->blocks) (void)hipFree(b.p);
    (void)hipFree(g->pair_deep);
    (void)hipFree(g->pair_cells);
    (void)hipFree(g->pair_links);
    (void)hipFree(g->flags);
    (void)hipFree(g->plain);
    (void)hipFree(g->stale);
    (void)hipFree(g->stale_idx);
    (void)hipFree(g->stale_cells);
    (void)hipFree(g->mlist);
    (void)hipFree(g->link);
    (void)hipFree(g->force);
    (void)hipFree(g->uin);
    (void)hipFree(g->rho);
    (void)hipFree(g->u);
    (void)hipFree(g->partials);
    (void)hipFree(g->stage);
    (void)hipFree(g->moments_out);
    (void)hipFree(g->xr);
    (void)hipFree(g->edge);
    (void)hipFree(g->erho);
    ibm_destroy(g);
    if (g->parent) {
        auto &pk = g->parent->kids;
        pk.erase(std::remove(pk.begin(), pk.end(), g), pk.end());
        (void)upload_kids(g->parent);
    }
    for (lumagpu_grid *k : g->kids) {
        if (k->parent == g) k->parent = nullptr;
        // a detached subtree goes back to its own streams
        for_each_level(k, [](lumagpu_grid *x) { x->stream = x->own_stream; });
    }
    (void)hipFree(g->d_kids);
    if (g->ev_done) (void)hipEventDestroy(g->ev_done);
    if (g->ev_ready) (void)hipEventDestroy(g->ev_ready);
    if (g->gexec) (void)hipGraphExecDestroy(g->gexec);
    if (g->own_stream) (void)hipStreamDestroy(g->own_stream);
    delete g;
    return 0;
}

int lumagpu_set_labels(lumagpu_grid *g, const int *lattyp, const double *xpos, const double *ypos,
                       const double *zpos) {
    if (int r = check_grid(g)) return r;
    if (!lattyp) return fail(LUMAGPU_EINVAL, "null label array");
    // the grid's labels change only once the whole array has been accepted
    if (xpos && ypos && zpos) {
        g->xpos.assign(xpos, xpos + g->d.N);
        g->ypos.assign(ypos, ypos + g->d.M);
        g->zpos.assign(zpos, zpos + g->d.K);
    }
    const int N = g->d.N, M = g->d.M, K = g->d.K;
    // keep the force bits a previous lumagpu_set_force call placed
    std::vector<uint8_t> prev = g->hflags;
    if (prev.size() != g->ncell) prev.assign(g->ncell, 0);
    std::vector<uint8_t> nf(g->ncell, 0);
    int any = 0, outlet = 0;
    std::vector<int> ecell, enrm;   // edge/corner velocity sites (device cell, packed normal)
    for (int i = 0; i < N; ++i)
        for (int j = 0; j < M; ++j)
            for (int k = 0; k < K; ++k) {
                const size_t id = (size_t)k + (size_t)j * K + (size_t)i * K * M;
                const int ty = lattyp[id];
                uint8_t fl = 0;
                switch (ty) {
                    case kSolid:
                    case kFluid: fl = (uint8_t)ty; break;
                    case kVelocity: {
                        fl = (uint8_t)ty;
                        if (g->d.regularised) {
                            if (!xpos || !ypos || !zpos)
                                return fail(LUMAGPU_EINVAL, "positions are required for regularised velocity sites");
                            int code = 0, n[3];
                            const int cnt = wall_normal(g->d, xpos[i], ypos[j], zpos[k], &code, n);
                            if (cnt == 0)
                                return fail(LUMAGPU_EINVAL,
                                            "Velocity site not outside domain walls is currently not supported.");
                            if (cnt > 1) {
                                code = kNormalEdge;
                                ecell.push_back(i + N * (j + M * k));
                                enrm.push_back((n[0] + 1) | ((n[1] + 1) << 2) | ((n[2] + 1) << 4));
                            }
                            fl |= (uint8_t)(code << kNormalShift);
                        }
                        break;
                    }
                    case kPressure: {
                        // regularised pressure BC on a face (:389-402); LUMA has no other form
                        if (!g->d.regularised)
                            return fail(LUMAGPU_EUNSUPPORTED, "pressure sites need regularised boundaries");
                        if (!xpos || !ypos || !zpos)
                            return fail(LUMAGPU_EINVAL, "positions are required for regularised pressure sites");
                        int code = 0, n[3];
                        const int cnt = wall_normal(g->d, xpos[i], ypos[j], zpos[k], &code, n);
                        if (cnt == 0)
                            return fail(LUMAGPU_EINVAL,
                                        "Velocity site not outside domain walls is currently not supported.");
                        if (cnt > 1) return fail(LUMAGPU_EINVAL, "Pressure BC not supported at corner/edge site. Exiting.");
                        fl = (uint8_t)(ty | (code << kNormalShift));
                        ecell.push_back(i + N * (j + M * k));
                        enrm.push_back((n[0] + 1) | ((n[1] + 1) << 2) | ((n[2] + 1) << 4));
                        break;
                    }
                    case kRefined:
                    case kTL2C:
                    case kTL2F: fl = (uint8_t)ty; break;
                    case kExtrapRight:
                        // LUMA pulls from two sites to the left of the source (:246-251); the
                        // outlet must be the last x column for that to stay on the grid
                        if (i != N - 1 || N < 4)
                            return fail(LUMAGPU_EUNSUPPORTED, "ExtrapolateRight sites must form the last x column");
                        fl = (uint8_t)ty;
                        outlet = 1;
                        break;
                    default:
                        return fail(LUMAGPU_EUNSUPPORTED,
                                    "site label " + std::to_string(ty) + " is not supported by this build");
                }
                if (ty != kFluid) any = 1;
                const size_t cell = (size_t)i + (size_t)N * ((size_t)j + (size_t)M * k);
                nf[cell] = (uint8_t)(fl | (prev[cell] & kForcedBit));
            }
    // Edge/corner velocity sites extrapolate rho, pressure sites their tangential u, from x + n
    // and x + 2n (_LBM_updateAndExtrapolate, :1353-1412).  Those neighbours must be sites whose
    // sweep 1 computes rho and u (fluid, TL2F); for any other type LUMA reads a value left from
    // an earlier step or its initial state.
    const int ne = (int)ecell.size();
    std::vector<int> etab(4 * (size_t)ne);
    for (int e = 0; e < ne; ++e) {
        const int c = ecell[e];
        const int i = c % N, j = (c / N) % M, k = c / (N * M);
        const int n[3] = {(enrm[e] & 3) - 1, ((enrm[e] >> 2) & 3) - 1, ((enrm[e] >> 4) & 3) - 1};
        int nb[2];
        for (int s = 1; s <= 2; ++s) {
            const int ii = i + s * n[0], jj = j + s * n[1], kk = k + s * n[2];
            if (ii < 0 || ii >= N || jj < 0 || jj >= M || kk < 0 || kk >= K)
                return fail(LUMAGPU_EINVAL, "Extrapolation does not have enough available cells.");
            nb[s - 1] = ii + N * (jj + M * kk);
            const int nty = nf[nb[s - 1]] & kTypeMask;
            if (nty != kFluid && nty != kTL2F)
                return fail(LUMAGPU_EUNSUPPORTED,
                            "edge/corner velocity or pressure site whose extrapolation neighbours are not fluid "
                            "is not supported");
        }
        etab[e] = c;
        etab[ne + e] = enrm[e];
        etab[2 * ne + e] = nb[0];
        etab[3 * ne + e] = nb[1];
    }
    // the allocations before the first change: short of memory here, the grid stays as it was
    struct Freed {
        void *p = nullptr;
        ~Freed() { (void)hipFree(p); }
    } edge, erho;
    if (ne && (dev_malloc(&edge.p, etab.size() * sizeof(int)) != hipSuccess ||
               dev_malloc(&erho.p, 8 * (size_t)ne * g->melem) != hipSuccess))
        return fail(LUMAGPU_ENOMEM, "edge site table allocation failed");
    if (outlet && !g->xr && dev_malloc(&g->xr, 2 * (size_t)g->Q * g->d.M * g->d.K * g->melem) != hipSuccess) {
        g->xr = nullptr;
        return fail(LUMAGPU_ENOMEM, "outlet buffer allocation failed");
    }
    if (int r = alloc_flags(g)) return r;
    if (ne) HIP_TRY(hipMemcpyAsync(edge.p, etab.data(), etab.size() * sizeof(int), hipMemcpyHostToDevice, g->stream));
    // the old tables are freed on the way out
    void *const old_edge = g->edge, *const old_erho = g->erho;
    g->edge = static_cast<int *>(edge.p);
    g->erho = static_cast<double *>(erho.p);
    edge.p = old_edge;
    erho.p = old_erho;
    g->nedge = ne;
    g->hflags = std::move(nf);
    g->has_outlet = outlet;
    // the step kernels can write the next step's outlet sources when every outlet row's source
    // two cells left is a site they step (collided, or streamed only for TL2C)
    g->xr_fold = 0;
    g->xr_ready = 0;
    if (outlet) {
        bool ok = true;
        for (int k = 0; k < K && ok; ++k)
            for (int j = 0; j < M && ok; ++j) {
                const size_t row = (size_t)N * ((size_t)j + (size_t)M * k);
                if ((g->hflags[row + N - 1] & kTypeMask) != kExtrapRight) continue;
                const unsigned fl = g->hflags[row + N - 3];
                const int t = fl & kTypeMask;
                const bool stepped = t == kFluid || t == kTL2F || t == kTL2C ||
                                     (t == kVelocity && g->d.regularised && ((fl >> kNormalShift) & 7) != kNormalEdge);
                ok = stepped;
            }
        g->xr_fold = ok ? 1 : 0;
    }
    g->masked = any || g->d.forced;
    if (int r = upload_flags(g)) return r;
    HIP_TRY(hipStreamSynchronize(g->stream));
    return 0;
}

}  // extern "C"

namespace {
// The three arrays of a checkpoint in one launch: 16-byte pieces, the arrays one after another in
// the grid (their sizes and addresses are multiples of 16: hipMalloc'd, whole cells of 8 bytes
// counted in pairs with an odd one at the end).
struct Copy3 {
    const void *src[3];
    void *dst[3];
    size_t n[3];   // 8-byte words
};
__global__ __launch_bounds__(256) void k_copy3(Copy3 c) {
    const size_t stride = (size_t)gridDim.x * 256, i0 = (size_t)blockIdx.x * 256 + threadIdx.x;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const uint4 *s = static_cast<const uint4 *>(c.src[k]);
        uint4 *d = static_cast<uint4 *>(c.dst[k]);
        const size_t n = c.n[k] / 2;
        for (size_t i = i0; i < n; i += stride) d[i] = s[i];
        if ((c.n[k] & 1) && i0 == 0)
            static_cast<uint2 *>(c.dst[k])[c.n[k] - 1] = static_cast<const uint2 *>(c.src[k])[c.n[k] - 1];
    }
}
hipError_t copy3(const Copy3 &c, hipStream_t s) {
    const size_t most = std::max(c.n[0], std::max(c.n[1], c.n[2])) / 2;
    const unsigned nb = (unsigned)std::min<size_t>(8192, std::max<size_t>(1, (most + 255) / 256));
    k_copy3<<<nb, 256, 0, s>>>(c);
    return hipGetLastError();
}
}  // namespace

struct lumagpu_checkpoint {
    const lumagpu_grid *owner = nullptr;
    void *f = nullptr;
    double *rho = nullptr, *u = nullptr;
    size_t fbytes = 0;
    int parity = 0, t = 0, has_state = 0;
};

extern "C" {

int lumagpu_checkpoint_save(lumagpu_grid *g, lumagpu_checkpoint **out) {
    if (int r = check_grid(g)) return r;
    if (!out) return fail(LUMAGPU_EINVAL, "null output");
    if (g->parent || !g->kids.empty()) return fail(LUMAGPU_EUNSUPPORTED, "checkpoints cover single-level grids");
    if (ibm_has_flexible(g)) return fail(LUMAGPU_EUNSUPPORTED, "checkpoints do not hold flexible-body state");
    auto *ck = new lumagpu_checkpoint();
    ck->owner = g;
    ck->fbytes = g->ps * g->Q * g->elem;
    if (dev_malloc(&ck->f, ck->fbytes) != hipSuccess ||
        dev_malloc(&ck->rho, g->ncell * g->melem) != hipSuccess ||
        dev_malloc(&ck->u, g->ncell * g->D * g->melem) != hipSuccess) {
        lumagpu_checkpoint_free(ck);
        return fail(LUMAGPU_ENOMEM, "checkpoint allocation failed");
    }
    const size_t nm = g->ncell * g->melem / 8;
    const Copy3 c{{g->f, g->rho, g->u}, {ck->f, ck->rho, ck->u}, {ck->fbytes / 8, nm, nm * g->D}};
    if (copy3(c, g->stream) != hipSuccess || hipStreamSynchronize(g->stream) != hipSuccess) {
        lumagpu_checkpoint_free(ck);
        return fail(LUMAGPU_EHIP, "checkpoint copy failed");
    }
    ck->parity = g->parity;
    ck->t = g->t;
    ck->has_state = g->has_state;
    *out = ck;
    return 0;
}

int lumagpu_checkpoint_restore(lumagpu_grid *g, const lumagpu_checkpoint *ck) {
    if (int r = check_grid(g)) return r;
    if (!ck) return fail(LUMAGPU_EINVAL, "null checkpoint");
    if (ck->owner != g) return fail(LUMAGPU_EINVAL, "checkpoint belongs to another grid");
    // on the grid's stream, like the steps that follow; lumagpu_checkpoint_free waits for the device
    const size_t nm = g->ncell * g->melem / 8;
    HIP_TRY(copy3(Copy3{{ck->f, ck->rho, ck->u}, {g->f, g->rho, g->u}, {ck->fbytes / 8, nm, nm * g->D}}, g->stream));
    g->xr_ready = 0;
    g->parity = ck->parity;
    g->pair_synced = 0;
    g->t = ck->t;
    g->has_state = ck->has_state;
    return 0;
}

int lumagpu_checkpoint_free(lumagpu_checkpoint *ck) {
    if (!ck) return 0;
    (void)hipFree(ck->f);
    (void)hipFree(ck->rho);
    (void)hipFree(ck->u);
    delete ck;
    return 0;
}

int lumagpu_set_zslab(lumagpu_grid *g, int on) {
    if (int r = check_grid(g)) return r;
    if (!on) {
        g->zslab = 0;
        return 0;
    }
    if (g->d.dims != 3 || g->Q != 19 || g->d.K < 3)
        return fail(LUMAGPU_EINVAL, "a z-slab needs a D3Q19 grid with at least one interior and two halo planes");
    if (g->masked || g->d.forced || g->parent || !g->kids.empty() || g->ibm)
        return fail(LUMAGPU_EUNSUPPORTED, "z-slab halo exchange is implemented for unlabelled, unforced single-level grids");
    if (g->melem != sizeof(double)) return fail(LUMAGPU_EUNSUPPORTED, "z-slabs run in the FP64 and shifted forms");
    if (g->parity != 0) return fail(LUMAGPU_ESTATE, "switch to a z-slab between step pairs");
    g->zslab = 1;
    return 0;
}

int lumagpu_grid_add_child(lumagpu_grid *parent, lumagpu_grid *child) {
    if (int r = check_grid(parent)) return r;
    if (int r = check_grid(child)) return r;
    if (child->parent) return fail(LUMAGPU_ESTATE, "grid already has a parent");
    if (parent->kids.size() >= kMaxKids)
        return fail(LUMAGPU_EUNSUPPORTED, "at most " + std::to_string(kMaxKids) + " refined regions per grid");
    const lumagpu_grid_desc &p = parent->d, &c = child->d;
    if (c.level != p.level + 1) return fail(LUMAGPU_EINVAL, "child level must be parent level + 1");
    if (c.precision != p.precision || c.Q != p.Q) return fail(LUMAGPU_EINVAL, "child and parent must share lattice and precision");
    // LBM_initSubGrid (GridObj_init_grids.cpp:416-425): N = 2*(CoarseLimsMax - CoarseLimsMin + 1)
    const int ext[3] = {c.N, c.M, c.K};
    const int pext[3] = {p.N, p.M, p.K};
    for (int a = 0; a < c.dims; ++a) {
        const int lo = c.coarse_lims[2 * a], hi = c.coarse_lims[2 * a + 1];
        if (lo < 0 || hi >= pext[a] || hi < lo || ext[a] != 2 * (hi - lo + 1))
            return fail(LUMAGPU_EINVAL, "child extents do not match its coarse limits on the parent");
    }
    // regions of one grid are disjoint (GridUtils::getSubGrid takes the first that holds a site)
    for (const lumagpu_grid *o : parent->kids) {
        bool apart = false;
        for (int a = 0; a < c.dims; ++a)
            apart = apart || c.coarse_lims[2 * a + 1] < o->d.coarse_lims[2 * a] ||
                    o->d.coarse_lims[2 * a + 1] < c.coarse_lims[2 * a];
        if (!apart) return fail(LUMAGPU_EINVAL, "refined regions of one grid overlap");
    }
    parent->kids.push_back(child);
    child->parent = parent;
    if (int r = upload_kids(parent)) {
        parent->kids.pop_back();
        child->parent = nullptr;
        return r;
    }
    // The hierarchy's levels step one after another (each child reads its parent and the parent
    // its children), so they share the root's stream: one in-order queue instead of an event
    // hop between queues at every level change.
    HIP_TRY(hipStreamSynchronize(child->stream));
    HIP_TRY(hipStreamSynchronize(parent->stream));
    for_each_level(child, [&](lumagpu_grid *x) { x->stream = parent->stream; });
    return 0;
}

int lumagpu_set_inlet(lumagpu_grid *g, const double *ux, const double *uy, const double *uz) {
    if (int r = check_grid(g)) return r;
    const size_t M = g->d.M;
    std::vector<double> h(3 * M, 0.0);
    for (size_t j = 0; j < M; ++j) {
        h[j] = ux ? ux[j] : 0.0;
        h[M + j] = uy ? uy[j] : 0.0;
        h[2 * M + j] = uz ? uz[j] : 0.0;
    }
    HIP_TRY(hipMemcpyAsync(g->uin, h.data(), 3 * M * sizeof(double), hipMemcpyHostToDevice, g->stream));
    HIP_TRY(hipStreamSynchronize(g->stream));
    return 0;
}

int lumagpu_init_equilibrium(lumagpu_grid *g, const double *rho, const double *u) {
    if (int r = check_grid(g)) return r;
    if (!rho || !u) return fail(LUMAGPU_EINVAL, "null rho or u");
    const size_t nb = g->ncell * (1 + g->D) * sizeof(double);
    if (int r = ensure_stage(g, nb)) return r;
    double *drho = g->stage, *du = g->stage + g->ncell;
    HIP_TRY(hipMemcpyAsync(drho, rho, g->ncell * sizeof(double), hipMemcpyHostToDevice, g->stream));
    HIP_TRY(hipMemcpyAsync(du, u, g->ncell * g->D * sizeof(double), hipMemcpyHostToDevice, g->stream));
    HIP_TRY(launch_aux(g, kAuxInitFeq, drho, du, nullptr));
    HIP_TRY(macro_from_luma(g, drho, du));
    g->parity = 0;
    g->has_state = 1;
    g->pair_synced = 0;
    g->xr_ready = 0;
    if (int r = capture_stale(g)) return r;
    HIP_TRY(hipStreamSynchronize(g->stream));
    return 0;
}

int lumagpu_upload_f(lumagpu_grid *g, const double *f) {
    if (int r = check_grid(g)) return r;
    if (!f) return fail(LUMAGPU_EINVAL, "null f");
    const size_t nb = g->ncell * g->Q * sizeof(double);
    if (int r = ensure_stage(g, nb)) return r;
    HIP_TRY(hipMemcpyAsync(g->stage, f, nb, hipMemcpyHostToDevice, g->stream));
    HIP_TRY(launch_aux(g, kAuxUpload, g->stage, nullptr, nullptr));
    g->parity = 0;
    g->has_state = 1;
    g->pair_synced = 0;
    g->xr_ready = 0;
    if (int r = capture_stale(g)) return r;
    HIP_TRY(hipStreamSynchronize(g->stream));
    return 0;
}

int lumagpu_upload_macro(lumagpu_grid *g, const double *rho, const double *u) {
    if (int r = check_grid(g)) return r;
    if (!rho || !u) return fail(LUMAGPU_EINVAL, "null rho or u");
    const size_t nb = g->ncell * (1 + g->D) * sizeof(double);
    if (int r = ensure_stage(g, nb)) return r;
    double *drho = g->stage, *du = g->stage + g->ncell;
    HIP_TRY(hipMemcpyAsync(drho, rho, g->ncell * sizeof(double), hipMemcpyHostToDevice, g->stream));
    HIP_TRY(hipMemcpyAsync(du, u, g->ncell * g->D * sizeof(double), hipMemcpyHostToDevice, g->stream));
    HIP_TRY(macro_from_luma(g, drho, du));
    HIP_TRY(hipStreamSynchronize(g->stream));
    return 0;
}

int lumagpu_download_f(lumagpu_grid *g, double *f) {
    if (int r = check_grid(g)) return r;
    if (!f) return fail(LUMAGPU_EINVAL, "null f");
    if (!g->has_state) return fail(LUMAGPU_ESTATE, "no state to download");
    const size_t nb = g->ncell * g->Q * sizeof(double);
    if (int r = ensure_stage(g, nb)) return r;
    HIP_TRY(launch_aux(g, kAuxDownload, nullptr, nullptr, g->stage));
    if (int r = copy_to_host(g, f, g->stage, nb)) return r;
    HIP_TRY(hipStreamSynchronize(g->stream));
    return 0;
}

int lumagpu_download_macro(lumagpu_grid *g, double *rho, double *u) {
    if (int r = check_grid(g)) return r;
    if (!rho || !u) return fail(LUMAGPU_EINVAL, "null rho or u");
    const size_t nr = g->ncell * sizeof(double), nb = nr * (1 + g->D);
    if (nb <= kPinDownload && ensure_pin(g, nb)) {
        // a small grid's fields: the kernel writes them to host memory itself
        double *hr = static_cast<double *>(g->pin), *hu = hr + g->ncell;
        HIP_TRY(macro_to_luma(g, hr, hu, false));
        HIP_TRY(hipStreamSynchronize(g->stream));
        std::memcpy(rho, hr, nr);
        std::memcpy(u, hu, nb - nr);
        return 0;
    }
    if (int r = ensure_stage(g, nb)) return r;
    double *drho = g->stage, *du = g->stage + g->ncell;
    HIP_TRY(macro_to_luma(g, drho, du, false));
    if (int r = copy_to_host(g, rho, drho, nr)) return r;
    if (int r = copy_to_host(g, u, du, nb - nr)) return r;
    HIP_TRY(hipStreamSynchronize(g->stream));
    return 0;
}

int lumagpu_tangent_seed_omega(lumagpu_grid *g, double d_omega) {
    if (int r = check_grid(g)) return r;
    if (g->d.precision != LUMAGPU_FP64T)
        return fail(LUMAGPU_ESTATE, "an omega seed needs an FP64 tangent-form grid (LUMAGPU_FP64T)");
    g->d_omega = d_omega;
    return 0;
}

int lumagpu_download_tangent(lumagpu_grid *g, double *df, double *drho, double *du) {
    if (int r = check_grid(g)) return r;
    if (g->melem == sizeof(double)) return fail(LUMAGPU_ESTATE, "derivatives exist on tangent-form grids only");
    if (!g->has_state) return fail(LUMAGPU_ESTATE, "no state to download");
    const size_t nf = g->ncell * g->Q * sizeof(double), nm = g->ncell * (1 + g->D) * sizeof(double);
    if (int r = ensure_stage(g, nf > nm ? nf : nm)) return r;
    if (df) {
        HIP_TRY(launch_aux(g, kAuxDownloadTan, nullptr, nullptr, g->stage));
        if (int r = copy_to_host(g, df, g->stage, nf)) return r;
        HIP_TRY(hipStreamSynchronize(g->stream));
    }
    if (drho || du) {
        double *sr = g->stage, *su = g->stage + g->ncell;
        HIP_TRY(macro_to_luma(g, sr, su, true));
        if (drho)
            if (int r = copy_to_host(g, drho, sr, g->ncell * sizeof(double))) return r;
        if (du)
            if (int r = copy_to_host(g, du, su, g->ncell * g->D * sizeof(double))) return r;
        HIP_TRY(hipStreamSynchronize(g->stream));
    }
    return 0;
}

int lumagpu_set_force(lumagpu_grid *g, const double *force_xyz) {
    if (int r = check_grid(g)) return r;
    if (!g->d.forced) return fail(LUMAGPU_ESTATE, "grid was created without forcing (desc.forced = 0)");
    if (!force_xyz) return fail(LUMAGPU_EINVAL, "null force");
    const int N = g->d.N, M = g->d.M, K = g->d.K, D = g->D;
    if (g->hflags.empty()) g->hflags.assign(g->ncell, (uint8_t)kFluid);
    const size_t w = g->melem / sizeof(double);   // (value, derivative) pairs in the tangent form
    std::vector<double> soa(g->ncell * D * w, 0.0);
    for (int i = 0; i < N; ++i)
        for (int j = 0; j < M; ++j)
            for (int k = 0; k < K; ++k) {
                const size_t id = (size_t)k + (size_t)j * K + (size_t)i * K * M;
                const size_t cell = (size_t)i + (size_t)N * ((size_t)j + (size_t)M * k);
                bool nz = false;
                for (int d = 0; d < D; ++d) {
                    const double v = force_xyz[d + D * id];
                    soa[w * (d * g->ncell + cell)] = v;
                    nz = nz || v != 0.0;
                }
                g->hflags[cell] = (uint8_t)((g->hflags[cell] & ~kForcedBit) | (nz ? kForcedBit : 0));
            }
    if (int r = upload_flags(g)) return r;
    HIP_TRY(hipMemcpyAsync(g->force, soa.data(), soa.size() * sizeof(double), hipMemcpyHostToDevice, g->stream));
    HIP_TRY(hipStreamSynchronize(g->stream));
    g->masked = 1;
    return 0;
}

int lumagpu_set_velocity_ramp(lumagpu_grid *g, double ramp_time) {
    if (int r = check_grid(g)) return r;
    if (!(ramp_time >= 0.0)) return fail(LUMAGPU_EINVAL, "ramp time must be >= 0");
    if (ramp_time > 0.0 && !(g->d.dt > 0.0)) return fail(LUMAGPU_EINVAL, "a velocity ramp needs desc.dt > 0");
    g->ramp_time = ramp_time;
    return 0;
}

int lumagpu_set_temporal_blocking(lumagpu_grid *g, int shape, int zchunk) {
    if (int r = check_grid(g)) return r;
    std::lock_guard<std::recursive_mutex> lock(g->f2_mu);
    if (shape < 0) {
        g->f2_auto = 0;
        g->fuse_off = 1;
        if (g->f2) {
            HIP_TRY(hipStreamSynchronize(g->stream));
            HIP_TRY(hipFree(g->f2));
        }
        g->f2 = nullptr;
        g->fuse_shape = -1;
        scratch_note(g);
        return 0;
    }
    int tx, ty;
    if (!fused_tile(shape, tx, ty)) return fail(LUMAGPU_EINVAL, "unknown tile shape");
    if (g->Q != 19) return fail(LUMAGPU_EUNSUPPORTED, "the two-step kernel runs on D3Q19 grids");
    const int p = g->d.precision;
    if (p != LUMAGPU_FP64 && p != LUMAGPU_FP32S && p != LUMAGPU_FP16S)
        return fail(LUMAGPU_EUNSUPPORTED, "the two-step kernel runs in the FP64, FP32- and FP16-shifted forms");
    if ((shape & 8) && g->elem > 4)
        return fail(LUMAGPU_EINVAL, "double-buffered tiles need storage of at most 4 bytes (FP32- or FP16-shifted)");
    if (!fused_shape_fits(shape, g->d.N, g->d.M))
        return fail(LUMAGPU_EINVAL, "N and M must be whole numbers of the tile's x and y extents");
    if (zchunk < 1 || g->d.K < 3) return fail(LUMAGPU_EINVAL, "z chunk must be >= 1 and K >= 3");
    if (!g->f2 && dev_malloc(&g->f2, g->ps * g->Q * g->elem) != hipSuccess) {
        g->f2 = nullptr;
        return fail(LUMAGPU_ENOMEM, "second population array");
    }
    g->f2_auto = 0;   // asked for: no longer one to give back
    scratch_note(g);
    g->pair_synced = 0;
    g->fuse_off = 0;
    g->fuse_shape = shape;
    g->fuse_zc = zchunk;
    return 0;
}

int lumagpu_set_reynolds_ramp(lumagpu_grid *g, double re, double ramp_time) {
    if (int r = check_grid(g)) return r;
    if (!(ramp_time >= 0.0)) return fail(LUMAGPU_EINVAL, "Reynolds ramp time must be >= 0");
    if (ramp_time > 0.0 && !(re > 0.0)) return fail(LUMAGPU_EINVAL, "a Reynolds ramp needs L_RE > 0");
    bool dims_ok = true;
    for_each_level(g, [&](const lumagpu_grid *x) {
        if (ramp_time > 0.0 && !(x->d.dt > 0.0 && x->d.dh > 0.0)) dims_ok = false;
    });
    if (!dims_ok) return fail(LUMAGPU_EINVAL, "a Reynolds ramp needs desc.dt and desc.dh > 0 on every level");
    for_each_level(g, [&](lumagpu_grid *x) {
        x->re = re;
        x->re_ramp = ramp_time;
    });
    return 0;
}

int lumagpu_get_omega(const lumagpu_grid *g, double *omega) {
    if (int r = check_grid(g)) return r;
    if (omega) *omega = g->d.omega;
    return 0;
}

int lumagpu_set_pressure_delta(lumagpu_grid *g, double p) {
    if (int r = check_grid(g)) return r;
    if (!std::isfinite(p)) return fail(LUMAGPU_EINVAL, "pressure delta must be finite");
    if (p != 0.0 && !(g->d.dm > 0.0 && g->d.dt > 0.0 && g->d.dh > 0.0))
        return fail(LUMAGPU_EINVAL, "a pressure delta needs desc.dh, dt and dm > 0");
    // GridUnits::pd2dlbm (GridUnits.h:177-180)
    const double cs = 1.0 / std::sqrt(3.0);
    g->pressure_drho = p == 0.0 ? 0.0 : (p * g->d.dh * (g->d.dt * g->d.dt) / g->d.dm) / (cs * cs);
    return 0;
}

int lumagpu_set_gravity(lumagpu_grid *g, double gravity, int direction) {
    if (int r = check_grid(g)) return r;
    if (!g->d.forced) return fail(LUMAGPU_ESTATE, "gravity needs a grid created with desc.forced = 1");
    if (direction < 0 || direction >= g->D) return fail(LUMAGPU_EINVAL, "gravity direction out of range");
    g->gravity_on = 1;
    g->gravity = gravity;
    g->gravity_dir = direction;
    g->store_macro = 1;   // the reset reads every site's rho of the previous step
    return 0;
}

int lumagpu_set_store_macro(lumagpu_grid *g, int on) {
    if (int r = check_grid(g)) return r;
    g->store_macro = on ? 1 : 0;
    return 0;
}

int lumagpu_step(lumagpu_grid *g, int subcycle) {
    if (int r = check_grid(g)) return r;
    if (subcycle < 0 || subcycle > 1) return fail(LUMAGPU_EINVAL, "subcycle must be 0 or 1");
    return apply_step(g, subcycle, nullptr, nullptr);
}

int lumagpu_stream_bc_macro(lumagpu_grid *g, int subcycle) {
    if (int r = check_grid(g)) return r;
    if (subcycle < 0 || subcycle > 1) return fail(LUMAGPU_EINVAL, "subcycle must be 0 or 1");
    if (!g->has_state) return fail(LUMAGPU_ESTATE, "step before the populations were initialised");
    if (g->half) return fail(LUMAGPU_ESTATE, "a split step is already open on this grid");
    if (g->re_ramp > 0.0) update_reynolds(g);
    if (int r = begin_step(g)) return r;
    // sweep 1's rho, u at every fluid, TL2F and regularised-face site, as LUMA's arrays hold them
    // between the sweeps (edge/corner and pressure sites get theirs in the second half)
    const StepArgs a = make_args(g);
    hipError_t e = launch_sites(g, a, g->parity == 0, (int)g->ncell, nullptr, 0);
    if (e != hipSuccess) return fail(LUMAGPU_EHIP, std::string("macro launch: ") + hipGetErrorString(e));
    g->half = 1;
    g->half_sub = subcycle;
    return 0;
}

int lumagpu_force_collide_swap(lumagpu_grid *g) {
    if (int r = check_grid(g)) return r;
    if (!g->half) return fail(LUMAGPU_ESTATE, "no split step open: call lumagpu_stream_bc_macro first");
    g->half = 0;
    return end_step(g, g->half_sub, nullptr, nullptr);
}

int lumagpu_reset_forces(lumagpu_grid *g) {
    if (int r = check_grid(g)) return r;
    if (!g->d.forced) return fail(LUMAGPU_ESTATE, "grid was created without forcing (desc.forced = 0)");
    const StepArgs a = make_args(g);
    const unsigned nb = (unsigned)((g->ncell + 255) / 256);
    if (g->gravity_on) {
        // _LBM_resetForces (:1327-1337) with L_GRAVITY_ON: the gravity component from rho
        const double rr = 1.0 / std::pow(2.0, (double)g->d.level);
        if (g->melem == sizeof(double))
            k_gravity_reset<double><<<nb, 256, 0, g->stream>>>(a, g->force, g->gravity, rr, g->gravity_dir);
        else
            k_gravity_reset<Dual><<<nb, 256, 0, g->stream>>>(a, g->force, g->gravity, rr, g->gravity_dir);
        HIP_TRY(hipGetLastError());
        return 0;
    }
    // every component of every site zeroed, the force bits with it
    if (g->melem == sizeof(double))
        k_force_clear<double><<<nb, 256, 0, g->stream>>>(a, g->force, g->flags, g->D);
    else
        k_force_clear<Dual><<<nb, 256, 0, g->stream>>>(a, g->force, g->flags, g->D);
    HIP_TRY(hipGetLastError());
    for (auto &f : g->hflags) f &= (uint8_t)~kForcedBit;
    ++g->flags_version;
    ibm_forget_flags(g);
    return 0;
}

int lumagpu_run(lumagpu_grid *g, int nsteps) {
    if (int r = check_grid(g)) return r;
    std::lock_guard<std::recursive_mutex> lock(g->f2_mu);
    if (nsteps < 0) return fail(LUMAGPU_EINVAL, "negative step count");
    if (g->half) return fail(LUMAGPU_ESTATE, "a split step is open on this grid: finish it with lumagpu_force_collide_swap");
    int s = 0;
    if (g->fuse_shape >= 0) {
        if (g->parity == 0 && nsteps >= 3) {
            if (int r = apply_step(g, 0, nullptr, nullptr)) return r;
            ++s;
        }
        // long runs replay a captured pair of two-step launches (the two arrays trade places
        // twice, so the graph's pointers hold for every replay)
        const int reps = fused_ready(g) ? (nsteps - s) / 4 : 0;
        if (reps >= 2) {
            const int r = run_fused_graph(g, reps);
            if (r < 0) return r;
            if (r == 0) s += 4 * reps;
        }
        while (nsteps - s >= 2 && fused_ready(g)) {
            if (int r = fused_pair(g, nullptr, nullptr)) return r;
            s += 2;
        }
    }
    if (nsteps - s >= 5 && pair_ok(g)) {
        // single steps until the bodies' supports are flagged and the layout is the one pairs start from
        for (int k = 0; k < 2 && (g->parity == 0 || !ibm_settled(g)); ++k, ++s)
            if (int r = apply_step(g, 0, nullptr, nullptr)) return r;
        int done = 0;
        if (g->parity != 0 && ibm_settled(g) && pair_ok(g))
            if (int r = run_pairs(g, nsteps - s, &done)) return r;
        s += done;
    }
    if (nsteps - s >= multi_min(g) && multi_ok(g)) {
        if (g->parity != 0) {
            if (int r = apply_step(g, 0, nullptr, nullptr)) return r;
            ++s;
        }
        int done = 0;
        if (int r = run_multi(g, nsteps - s, &done)) return r;
        s += done;
    }
    // Long runs of a hierarchy without host work per step replay a captured pair of steps: the
    // step alternates between the two AA kernels, so two steps are the period (the child's
    // four sub-steps included).  One eager step first settles the IB support flags.
    if (nsteps - s >= 8 && graph_ok(g)) {
        while (s < nsteps && (s == 0 || g->parity != 0)) {
            if (int r = apply_step(g, 0, nullptr, nullptr)) return r;
            ++s;
        }
        const int reps = (nsteps - s) / 2;
        if (reps >= 2) {
            int r = run_graph(g, reps);
            if (r < 0) return r;
            if (r == 0) s += 2 * reps;   // r > 0: not capturable here, steps continue eagerly
        }
    }
    for (; s < nsteps; ++s)
        if (int r = apply_step(g, 0, nullptr, nullptr)) return r;
    return 0;
}

int lumagpu_run_timed(lumagpu_grid *g, int nsteps, double *ms_total, double *ms_kernel_mean) {
    if (int r = check_grid(g)) return r;
    if (nsteps <= 0) return fail(LUMAGPU_EINVAL, "step count must be positive");
    std::vector<hipEvent_t> ev(2 * (size_t)nsteps);
    for (auto &e : ev) HIP_TRY(hipEventCreate(&e));
    int rc = 0;
    // launches: event pairs in use, each covering one step or (two-step kernel) two
    int nl = 0;
    for (int s = 0; s < nsteps && !rc;) {
        if (nsteps - s >= 2 && fused_ready(g)) {
            rc = fused_pair(g, ev[2 * nl], ev[2 * nl + 1]);
            s += 2;
        } else {
            rc = apply_step(g, 0, ev[2 * nl], ev[2 * nl + 1]);
            s += 1;
        }
        ++nl;
    }
    if (!rc) {
        HIP_TRY(hipEventSynchronize(ev[2 * nl - 1]));
        float tot = 0.f;
        HIP_TRY(hipEventElapsedTime(&tot, ev.front(), ev[2 * nl - 1]));
        double sum = 0.0;
        for (int l = 0; l < nl; ++l) {
            float k = 0.f;
            HIP_TRY(hipEventElapsedTime(&k, ev[2 * l], ev[2 * l + 1]));
            sum += k;
        }
        if (ms_total) *ms_total = tot;
        // per step: a two-step launch counts half its duration for each of its steps
        if (ms_kernel_mean) *ms_kernel_mean = sum / nsteps;
    }
    for (auto &e : ev) (void)hipEventDestroy(e);
    return rc;
}

int lumagpu_get_time(const lumagpu_grid *g, int *t) {
    if (int r = check_grid(g)) return r;
    if (t) *t = g->t;
    return 0;
}

int lumagpu_sync(lumagpu_grid *g) {
    if (int r = check_grid(g)) return r;
    HIP_TRY(hipStreamSynchronize(g->stream));
    return 0;
}

int lumagpu_moments(lumagpu_grid *g, double out[LUMAGPU_NUM_MOMENTS]) {
    if (int r = check_grid(g)) return r;
    if (!out) return fail(LUMAGPU_EINVAL, "null output");
    if (!g->has_state) return fail(LUMAGPU_ESTATE, "no state");
    HIP_TRY(launch_aux(g, kAuxMoments, nullptr, nullptr, g->partials));
    const dim3 gr = cell_grid(g->d.N, g->d.M, g->d.K);
    const size_t nblocks = (size_t)gr.x * gr.y * gr.z;
    k_sum_partials<<<1, 256, 0, g->stream>>>(g->partials, nblocks, g->moments_out);
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipMemcpyAsync(out, g->moments_out, kMomentCount * sizeof(double), hipMemcpyDeviceToHost, g->stream));
    HIP_TRY(hipStreamSynchronize(g->stream));
    return 0;
}

int lumagpu_moments_noalloc(lumagpu_grid *g, double *out_dev) {
    if (int r = check_grid(g)) return r;
    if (!out_dev) return fail(LUMAGPU_EINVAL, "null output");
    if (!g->has_state) return fail(LUMAGPU_ESTATE, "no state");
    const dim3 gr = cell_grid(g->d.N, g->d.M, g->d.K);
    const size_t nblocks = (size_t)gr.x * gr.y * gr.z;
    if (nblocks > kScratchBlocks)
        return fail(LUMAGPU_EINVAL, "grid too large for lumagpu_moments_noalloc: " + std::to_string(nblocks) +
                                        " row blocks of 256 cells, at most " + std::to_string(kScratchBlocks));
    int dev = -1;
    HIP_TRY(hipGetDevice(&dev));
    if (dev != g->device) return fail(LUMAGPU_EINVAL, "call lumagpu_moments_noalloc with the grid's GPU current");
    double *partials = nullptr;
    if (int r = scratch_on(dev, &partials)) return r;
    // every block writes its own partials and the sum writes every output: nothing to clear
    HIP_TRY(launch_aux(g, kAuxMoments, nullptr, nullptr, partials));
    k_sum_partials<<<1, 256, 0, g->stream>>>(partials, nblocks, out_dev);
    HIP_TRY(hipGetLastError());
    return 0;
}

int lumagpu_footprint(const lumagpu_grid *g, size_t *bytes_per_cell, size_t *f_bytes) {
    if (int r = check_grid(g)) return r;
    if (bytes_per_cell) *bytes_per_cell = g->elem * g->Q;
    if (f_bytes) *f_bytes = g->ps * g->Q * g->elem;
    return 0;
}

}  // extern "C"
