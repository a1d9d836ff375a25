"""Grid kernels that take the cells in linear order (rows that no block size divides): every row
length class, both AA parities and macro store, bit for bit against the oracle in FP64, and the
shifted forms against FP64 within their storage."""
import numpy as np
import pytest

from luma_amd import setups
from luma_amd.grid import GpuGrid
from oracle.oracle import OracleGrid

pytestmark = pytest.mark.gpu


def _pair(case, form, steps):
    o = OracleGrid(case.dims, case.Q, case.N, case.M, case.K, omega=case.omega, forced=case.forced)
    if case.lattyp is not None:
        o.set_labels(case.lattyp)
    if case.force is not None:
        o.set_force(case.force)
    o.init_feq(case.rho, case.u)
    o.run(steps, 8)
    with GpuGrid.from_case(case, form, store_macro=True) as g:
        g.run(steps)
        return (g.download_f(),) + g.download_macro(), (o.get_f(),) + o.get_macro()


# one lane over a wave, a block and a row; aligned rows (48, 96 doubles) and others
@pytest.mark.parametrize("shape", [(3, 3, 3), (65, 3, 4), (48, 5, 7), (96, 3, 5), (250, 4, 3), (257, 3, 3)])
@pytest.mark.parametrize("form", ["fp64", "fp32s", "fp16s"])
def test_periodic_box(shape, form):
    case = setups.taylor_green(shape, u0=0.04, tau=0.7)
    for steps in (1, 2, 5):
        print(f"[order] {shape} {form} {steps}", flush=True)
        got, want = _pair(case, form, steps)
        for a, b in zip(got, want):
            if form == "fp64":
                assert np.array_equal(a, b)
            else:
                # a few roundings of populations below 0.05 (their deviations) per step
                eps = 2.0 ** -24 if form == "fp32s" else 2.0 ** -11
                assert np.abs(a - b).max() <= 19 * 8 * steps * 0.05 * eps


# the plain-site kernel needs 2^20 cells; rows of 90 start off the cache lines, rows of 96 on them
@pytest.mark.parametrize("shape", [(90, 120, 98), (96, 121, 91)])
def test_labelled_channel(shape):
    case = setups.body_force_channel(*shape, dims=3, g=1e-5)
    case.u[..., 0] = 0.01 * np.sin(np.arange(shape[2]))
    case.u[case.lattyp == setups.SOLID] = 0.0
    print(f"[order] channel {shape}", flush=True)
    got, want = _pair(case, "fp64", 3)
    m = case.lattyp != setups.SOLID
    for a, b in zip(got, want):
        assert np.array_equal(a[m], b[m])


# the site list of large labelled grids (2^20 cells and more): walls, a forced-equilibrium inlet and an
# outlet (their sources and the outlet's own populations), by link words, one wave per block
def test_listed_sites():
    case = setups.uniform_inflow_3d(131, 92, 88, 0.03, 0.6)
    case.lattyp[1:-1, 0, :] = setups.SOLID
    case.lattyp[40:47, 30:37, 20:31] = setups.SOLID
    case.forced = False
    o = OracleGrid(3, 19, case.N, case.M, case.K, omega=case.omega, regularised=False, edges=case.edges)
    o.set_labels(case.lattyp)
    o.set_positions(case.xpos, case.ypos, case.zpos)
    o.set_inlet(case.ux_in, case.uy_in, case.uz_in)
    o.init_feq(case.rho, case.u)
    o.run(4, 8)
    print("[order] listed sites", flush=True)
    with GpuGrid.from_case(case, "fp64", store_macro=True) as g:
        g.run(4)
        got = (g.download_f(),) + g.download_macro()
    # an outlet row behind a solid x = N-3 site takes that site's own populations, which this build
    # does not keep: four steps carry them four columns from the outlet
    m = (case.lattyp == setups.FLUID) & (np.arange(case.N) < case.N - 4)[:, None, None]
    for a, b in zip(got, (o.get_f(),) + o.get_macro()):
        assert np.array_equal(a[m], b[m])
