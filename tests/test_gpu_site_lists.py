"""Grids large enough for the site list (2^20 cells): with labels set again, the list and its link words
are those of a grid that never had other labels, whatever the earlier calls left; and the outlet's
rows, which the list steps by their link words' outlet bits, against the oracle."""
import numpy as np
import pytest

from luma_amd import setups
from luma_amd.grid import GpuGrid
from oracle.oracle import OracleGrid

pytestmark = pytest.mark.gpu


def _after(g, rho, u):
    g.init_equilibrium(rho, u)
    g.set_store_macro(True)
    for _ in range(3):
        g.LBM_multi_opt()
    return (g.download_f(),) + g.download_macro()


def _flow(shape):
    x, y, z = np.meshgrid(*(np.arange(n) for n in shape), indexing="ij")
    u = np.stack([0.02 * np.sin(0.3 * y), 0.02 * np.sin(0.2 * z), 0.02 * np.cos(0.25 * x)], axis=-1)
    return np.ones(shape) + 0.01 * np.cos(0.1 * x), u


def test_labels_from_a_z_slab():
    # on a z-slab a grid is labelled as a whole; the same labels on the plain grid go by the list
    shape = (104, 101, 102)
    rho, u = _flow(shape)
    lt = np.full(shape, setups.FLUID)
    lt[:, 0, :] = lt[:, -1, :] = setups.SOLID
    lt[30:40, 20:31, 50:62] = setups.SOLID
    u[lt == setups.SOLID] = 0.0
    print("[lists] z-slab", flush=True)
    with GpuGrid(3, 19, *shape, precision="fp64", omega=1.3) as a, GpuGrid(3, 19, *shape, precision="fp64", omega=1.3) as b:
        a.set_zslab(True)
        a.set_labels(lt)
        a.set_zslab(False)
        a.set_labels(lt)
        b.set_labels(lt)
        for p, q in zip(_after(a, rho, u), _after(b, rho, u)):
            assert np.array_equal(p, q)


def test_same_labels_at_other_positions():
    # the positions decide which sites of an inlet plane are faces (stepped by the list) and which edges
    shape = (104, 101, 102)
    rho, u = _flow(shape)
    lt = np.full(shape, setups.FLUID)
    lt[0] = setups.VELOCITY
    x, y, z = (0.5 + np.arange(n) for n in shape)
    inside = 10.0 + np.arange(shape[1]) / 10.0       # no row of this y lies in a wall
    kw = dict(precision="fp64", omega=1.3, edges=(104.0, 101.0, 102.0), wall_thk=(1.0, 1.0, 1.0, 1.0, 0.0, 0.0))
    print("[lists] positions", flush=True)
    with GpuGrid(3, 19, *shape, **kw) as a, GpuGrid(3, 19, *shape, **kw) as b:
        for g in (a, b):
            g.set_inlet(np.full(shape[1], 0.02), np.zeros(shape[1]), np.zeros(shape[1]))
        a.set_labels(lt, x, np.concatenate([[0.5], inside[1:]]), z)
        a.set_labels(lt, x, inside, z)
        b.set_labels(lt, x, inside, z)
        for p, q in zip(_after(a, rho, u), _after(b, rho, u)):
            assert np.array_equal(p, q)


def test_outlet_rows():
    # every fluid and outlet site up to the last column, behind fluid rows as the flow has them and with
    # a solid block on the way
    case = setups.uniform_inflow_3d(131, 92, 88, 0.03, 0.6)
    case.lattyp[60:67, 30:37, 20:31] = setups.SOLID
    case.forced = False
    case.u[..., 1] = 0.01 * np.sin(np.arange(92))[None, :, None]
    case.u[..., 2] = 0.01 * np.cos(0.3 * np.arange(131))[:, None, None]
    case.u[0] = (0.03, 0.0, 0.0)        # the inlet's, which is what its sites hold
    case.u[case.lattyp == setups.SOLID] = 0.0
    o = OracleGrid(3, 19, case.N, case.M, case.K, omega=case.omega, regularised=False, edges=case.edges)
    o.set_labels(case.lattyp)
    o.set_positions(case.xpos, case.ypos, case.zpos)
    o.set_inlet(case.ux_in, case.uy_in, case.uz_in)
    o.init_feq(case.rho, case.u)
    o.run(5, 8)
    print("[lists] outlet", flush=True)
    with GpuGrid.from_case(case, "fp64", store_macro=True) as g:
        g.run(5)
        got = (g.download_f(),) + g.download_macro()
    m = (case.lattyp == setups.FLUID) | (case.lattyp == setups.EXTRAP_RIGHT)
    assert m[-1].any()
    for a, b in zip(got, (o.get_f(),) + o.get_macro()):
        assert np.array_equal(a[m], b[m])
