"""Several steps per launch on small 2D grids (lumagpu_run): against single steps bit for bit in
every population slot that a download reads, and against the oracle in FP64.  Sizes from less than
one window to several tiles with a remainder; step counts with every remainder; solid walls,
regularised and forced-equilibrium lids, a periodic box, a set force field."""
import dataclasses

import numpy as np
import pytest

from luma_amd import setups
from luma_amd.grid import GpuGrid
from oracle.oracle import OracleGrid

pytestmark = pytest.mark.gpu


def _case(kind, n, m):
    if kind == "periodic":
        return setups.taylor_green((n, m, 1), u0=0.04, tau=0.7, dims=2)
    if kind == "force":
        case = setups.body_force_channel(n, m, 1, 2, g=1e-5)
        case.force[..., 1] = 1e-6 * np.sin(np.arange(m))[None, :, None]
        case.force[3::5] = 0.0
        return case
    case = setups.lid_driven_cavity(max(n, m), re=5.0 * max(n, m), regularised=kind == "regularised")
    return case


@pytest.mark.parametrize("kind", ["periodic", "force", "regularised", "forced_eq"])
@pytest.mark.parametrize("shape", [(3, 3), (7, 33), (24, 24), (65, 40), (131, 131)])
@pytest.mark.parametrize("form", ["fp64", "fp32s"])
def test_matches_single_steps(kind, shape, form):
    case = _case(kind, *shape)
    print(f"[multi2d] {kind} {case.N}x{case.M} {form}", flush=True)
    with GpuGrid.from_case(case, form, store_macro=True) as a, GpuGrid.from_case(case, form, store_macro=True) as b:
        for steps in (2, 5, 8, 19, 3):      # the odd counts leave the other layout for the next run
            a.run(steps)
            for _ in range(steps):
                b.LBM_multi_opt()
            assert a.t == b.t
            for p, q in zip((a.download_f(),) + a.download_macro(), (b.download_f(),) + b.download_macro()):
                assert np.array_equal(p, q), steps
        if form == "fp64":
            o = OracleGrid(2, 9, case.N, case.M, 1, omega=case.omega, regularised=case.regularised, forced=case.forced,
                           edges=case.edges, wall_thk=case.wall_thk)
            if case.lattyp is not None:
                o.set_labels(case.lattyp)
            if case.xpos is not None:
                o.set_positions(case.xpos, case.ypos, case.zpos)
            if case.ux_in is not None:
                o.set_inlet(case.ux_in, case.uy_in, case.uz_in)
            if case.force is not None:
                o.set_force(case.force)
            o.init_feq(case.rho, case.u)
            o.run(37, 1)
            m = np.ones((case.N, case.M, 1), bool) if case.lattyp is None else \
                (case.lattyp == setups.FLUID) | ((case.lattyp == setups.VELOCITY) & case.regularised)
            for p, q in zip(a.download_macro(), o.get_macro()):
                assert np.array_equal(p[m], q[m])


def test_new_state_and_labels_between_runs():
    # an upload, a checkpoint and new labels between runs: nothing of the other array comes back
    case = _case("regularised", 40, 40)
    case2 = dataclasses.replace(case, lattyp=case.lattyp.copy())
    case2.lattyp[10:15, 12:20] = setups.SOLID
    with GpuGrid.from_case(case, "fp64", store_macro=True) as a, GpuGrid.from_case(case, "fp64", store_macro=True) as b:
        a.run(12)
        ck = a.checkpoint()
        a.run(11)
        a.restore(ck)
        GpuGrid.free_checkpoint(ck)
        for _ in range(12):
            b.LBM_multi_opt()
        f = b.download_f()
        assert np.array_equal(a.download_f(), f)
        for g in (a, b):
            g.set_labels(case2.lattyp, case2.xpos, case2.ypos, case2.zpos)
            g.upload_f(f * (1.0 + 1e-3 * np.arange(9)))
        a.run(10)
        for _ in range(10):
            b.LBM_multi_opt()
        assert np.array_equal(a.download_f(), b.download_f())


# runs on both sides of the least counts (4, and 8 for small FP64 boxes), from both layouts, with the steps
# that are left over one at a time
@pytest.mark.parametrize("kind", ["periodic", "regularised"])
@pytest.mark.parametrize("n", [40, 330])
@pytest.mark.parametrize("form", ["fp64", "fp32s"])
def test_short_runs(kind, n, form):
    case = _case(kind, n, n)
    print(f"[multi2d] short {kind} {n} {form}", flush=True)
    with GpuGrid.from_case(case, form, store_macro=True) as a, GpuGrid.from_case(case, form, store_macro=True) as b:
        for steps in (4, 6, 7, 8, 9, 1, 5, 10, 13, 3):
            a.run(steps)
            for _ in range(steps):
                b.LBM_multi_opt()
            for p, q in zip((a.download_f(),) + a.download_macro(), (b.download_f(),) + b.download_macro()):
                assert np.array_equal(p, q), steps
