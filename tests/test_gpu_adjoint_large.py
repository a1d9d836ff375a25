"""The discrete adjoint on grids whose reversed step takes the plain sites and a list of the others
(2^17 cells and more): omega, inlet-scale and initial-population gradients against central differences of
the forward, with the body near the inlet and near the outlet (whose sources are pulled twice); the run
along the tape against checkpoint intervals that give one, several and a partial last segment, bit for
bit; the state it leaves; and a second run on the kept buffers."""
import dataclasses

import numpy as np
import pytest

from luma_amd import setups
from luma_amd.grid import GpuGrid

pytestmark = pytest.mark.gpu


def _inlet():
    return setups.uniform_inflow_3d(72, 46, 44, 0.03, 0.6), setups.sphere_markers((7.2, 23.1, 21.9), 3.0, 1.0)


def _outlet():
    case = setups.uniform_inflow_3d(72, 46, 44, 0.03, 0.6)
    case.lattyp[30:33, 10:14, 10:14] = setups.SOLID
    return case, setups.sphere_markers((64.2, 23.1, 21.9), 3.0, 1.0)


def _walls():
    case = setups.channel_2d(560, 240, 20.0, 0.04, 20.0, regularised=True)
    dh = case.info["dh"]
    return case, setups.circle_markers((8.3 * dh, 120.4 * dh, 0.0), 4.0 * dh, dh)


def _grid(case, pos, omega=None, scale=1.0, f0=None):
    g = GpuGrid.from_case(case if omega is None else dataclasses.replace(case, omega=omega), "fp64", store_macro=True)
    if scale != 1.0:
        g.set_inlet(case.ux_in * scale, case.uy_in * scale, case.uz_in * scale)
    if f0 is not None:
        g.upload_f(f0)
    g.ibm_add_body(pos)
    g.ibm_initialise()
    return g


T = 14


def _J(case, pos, **kw):
    with _grid(case, pos, **kw) as g:
        return g.adj_run(T, T, backward=False)["J"]


@pytest.mark.parametrize("build", [_inlet, _outlet, _walls])
def test_gradients_and_tape(build):
    case, pos = build()
    print(f"[adjoint] {build.__name__} {case.N}x{case.M}x{case.K}", flush=True)
    with _grid(case, pos) as g:
        f0 = g.download_f()
        adj = g.adj_run(T, 5, initial=True)
        end = (g.download_f(),) + g.download_macro()
        more = g.adj_run(3, 2, initial=True)
        g.upload_f(f0)
        assert g.t == T + 3
        again = g.adj_run(T, 1, initial=True)
    with _grid(case, pos) as g:
        whole = g.adj_run(T, T, initial=True)
        for a, b in zip(end, (g.download_f(),) + g.download_macro()):
            assert np.array_equal(a, b)
    with _grid(case, pos) as g:
        for _ in range(T):
            g.LBM_multi_opt()
        for a, b in zip(end, (g.download_f(),) + g.download_macro()):
            assert np.array_equal(a, b)
    assert more["J"] != 0.0
    for key in ("J", "dJ_domega", "dJ_dinlet", "dJ_dpos", "lambda0"):
        assert np.array_equal(adj[key], whole[key]) and np.array_equal(adj[key], again[key]), key

    # central differences as in the small grids' test: 1e-4 bounds their truncation and rounding
    h = 1e-5 * case.omega
    fd = (_J(case, pos, omega=case.omega + h) - _J(case, pos, omega=case.omega - h)) / (2 * h)
    print("dJ/domega", adj["dJ_domega"], fd, flush=True)
    assert abs(adj["dJ_domega"] - fd) <= 1e-4 * abs(fd)
    if build is not _outlet:       # no inlet signal reaches the body at the far end
        h = 1e-5
        fd = (_J(case, pos, scale=1 + h) - _J(case, pos, scale=1 - h)) / (2 * h)
        print("dJ/dinlet", adj["dJ_dinlet"], fd, flush=True)
        assert abs(adj["dJ_dinlet"] - fd) <= 1e-4 * abs(fd)
    else:
        assert adj["dJ_dinlet"] == 0.0
    live = np.isin(case.lattyp, (setups.FLUID, setups.VELOCITY))
    dirn = np.random.default_rng(5).standard_normal(f0.shape) * live[..., None]
    h = 1e-6
    fd = (_J(case, pos, f0=f0 + h * dirn) - _J(case, pos, f0=f0 - h * dirn)) / (2 * h)
    pred = float((adj["lambda0"] * dirn).sum())
    print("dJ/df0 . d", pred, fd, flush=True)
    assert abs(pred - fd) <= 1e-4 * abs(fd)


# the state a gradient leaves is that of plain steps at every site, those of a forced-equilibrium inlet (which
# never step) included: last segments of one, two and more steps, ending on either kind of step, from either
# layout
@pytest.mark.parametrize("dims,form", [(2, "fp64"), (2, "fp32s"), (3, "fp64"), (3, "fp32s")])
def test_state_at_sites_that_never_step(dims, form):
    if dims == 2:
        case = setups.channel_2d(60, 30, 10.0, 0.04, 20.0, regularised=False)
        case.lattyp[20:24, 10:16] = setups.SOLID
        case.lattyp[30:33, 4:9] = setups.VELOCITY
    else:
        case = setups.uniform_inflow_3d(24, 12, 11, 0.03, 0.6)
        case.lattyp[10:13, 3:7, 2:5] = setups.VELOCITY
    for before, t, every in ((0, 3, 4), (1, 2, 7), (0, 2, 2), (1, 3, 3), (0, 5, 2), (0, 6, 5), (1, 7, 4), (0, 1, 1)):
        print(f"[adjoint] state {dims}D {form} {before} {t} {every}", flush=True)
        with GpuGrid.from_case(case, form) as a, GpuGrid.from_case(case, form) as b:
            for g in (a, b):
                for _ in range(before):
                    g.LBM_multi_opt()
            a.adj_run(t, every, initial=True)
            for _ in range(t):
                b.LBM_multi_opt()
            assert a.t == b.t and np.array_equal(a.download_f(), b.download_f()), (before, t, every)
