"""Epsilon systems solved on the device in the position gradient (bodies of 192 markers and more): the
gradient against central differences of the forward, as in the other gradient tests, for body
sizes around the device's lower limit, multiples of the factorisation's 16-column panels and its
1024 rows per block; and a singular system's refusal."""
import ctypes as C

import numpy as np
import pytest

from luma_amd import _abi, setups
from luma_amd.grid import GpuGrid
from oracle.oracle import OracleGrid, OracleIBM

pytestmark = pytest.mark.gpu


def _grid(pos, shape):
    case = setups.uniform_inflow_3d(*shape, 0.03, 0.6)
    g = GpuGrid.from_case(case, "fp64")
    g.ibm_add_body(pos)
    g.ibm_initialise()
    return g


# 191 is solved on the host; 192 = 12 panels, 193 leaves one column; 1040 takes two rows per thread
@pytest.mark.parametrize("n", [191, 192, 193, 300, 1040])
def test_position_gradient_against_differences(n):
    radius = float(np.sqrt(n / (4.0 * np.pi)))      # one marker per unit area
    shape = (int(2 * radius) + 16,) + (int(2 * radius) + 10,) * 2
    centre = tuple(0.5 * s + 0.13 for s in shape)
    pos = setups.sphere_markers(centre, radius, 1.0, n=n) + np.random.default_rng(n).normal(0.0, 0.03, (n, 3))
    print(f"[eps] {n}", flush=True)
    with _grid(pos, shape) as g:
        out = g.adj_run(6, 3, initial=False)
    grad = out["dJ_dpos"]
    # a random direction over all markers.  Among n spacings some lie within the moves of a kink (the
    # nearest marker changes, a support enters), which enters J by O(h) of those markers' share:
    # h = 1e-5 keeps that at 1e-8 here, and the rounding of J over h at 1e-11 (h = 1e-4 is 5e-3
    # off at 192 markers for a host-solved gradient too)
    d = np.random.default_rng(n + 1).standard_normal((n, 3))
    h, J = 1e-5, []
    for s in (1.0, -1.0):
        with _grid(pos + s * h * d, shape) as g:
            J.append(g.adj_run(6, 3, backward=False)["J"])
    fd = (J[0] - J[1]) / (2.0 * h)
    assert abs((grad * d).sum() - fd) <= 1e-4 * abs(fd) + 1e-9


# the systems of ibm_initialise go the same way: epsilon bit for bit the oracle's LU
@pytest.mark.parametrize("n", [192, 207, 500, 1100])
def test_epsilon_bitwise(n):
    radius = float(np.sqrt(n / (4.0 * np.pi)))
    shape = (int(2 * radius) + 10,) * 3
    pos = setups.sphere_markers(tuple(0.5 * s + 0.13 for s in shape), radius, 1.0, n=n) + \
        np.random.default_rng(n).normal(0.0, 0.03, (n, 3))
    case = setups.uniform_inflow_3d(*shape, 0.03, 0.6)
    print(f"[eps] bitwise {n}", flush=True)
    o = OracleGrid(3, 19, case.N, case.M, case.K, omega=case.omega, regularised=False, forced=True, edges=case.edges)
    o.set_labels(case.lattyp)
    o.set_positions(case.xpos, case.ypos, case.zpos)
    ib = OracleIBM(o, 1.0)
    ib.add_body(pos)
    ib.initialise()
    with _grid(pos, shape) as g:
        m = g.ibm_markers(0)
    want = ib.markers(0)
    assert np.array_equal(m["ds"], want["ds"]) and np.array_equal(m["eps"], want["eps"])


def test_singular_system_is_refused():
    # two markers at one place give two equal rows
    pos = setups.sphere_markers((12.0, 11.0, 11.0), 4.0, 1.0, n=200)
    pos[150] = pos[20]
    case = setups.uniform_inflow_3d(26, 22, 22, 0.03, 0.6)
    with GpuGrid.from_case(case, "fp64") as g:
        g.ibm_add_body(pos)
        with pytest.raises(Exception, match="singular|epsilon"):
            g.ibm_initialise()
            g.adj_run(2, 2, initial=False)
            raise RuntimeError("epsilon system accepted")


# a chain of markers couples to its neighbours alone: its matrix is made on the device and solved in the
# band, up to the length where a panel of the dense factorisation takes two rows per thread and beyond
@pytest.mark.parametrize("n", [192, 1030])
def test_position_gradient_of_a_chain(n):
    case = setups.channel_2d(n + 40, 34, 12.0, 0.04, 20.0)
    dh = case.info["dh"]
    r = np.random.default_rng(n)
    pos = np.zeros((n, 3))
    pos[:, 0] = (20.2 + np.arange(n) + r.uniform(-0.2, 0.2, n)) * dh
    pos[:, 1] = (17.3 + r.uniform(-0.2, 0.2, n)) * dh

    def run(p, **kw):
        with GpuGrid.from_case(case, "fp64") as g:
            g.ibm_add_body(p)
            g.ibm_initialise()
            return g.adj_run(6, 3, **kw)
    print(f"[eps] chain {n}", flush=True)
    grad = run(pos, initial=False)["dJ_dpos"]
    d = np.zeros((n, 3))
    d[:, :2] = r.standard_normal((n, 2)) * dh
    h = 1e-5
    fd = (run(pos + h * d, backward=False)["J"] - run(pos - h * d, backward=False)["J"]) / (2.0 * h)
    assert abs((grad * d).sum() - fd) <= 1e-4 * abs(fd) + 1e-9


# ---- the factorisation itself --------------------------------------------------------------------
# lu_factor_device is no entry of the C ABI: it is called by its C++ name, in buffers of the runtime that
# the library links
def _factor(a):
    lib, hip = _abi.load(), C.CDLL("libamdhip64.so.7")
    n = a.shape[0]
    f = lib["_ZN7lumagpu16lu_factor_deviceEiPdPiS1_P12ihipStream_t"]
    f.argtypes = [C.c_int, C.c_void_p, C.c_void_p, C.c_void_p, C.c_void_p]
    da, dp = C.c_void_p(), C.c_void_p()
    assert hip.hipMalloc(C.byref(da), C.c_size_t(8 * n * n)) == 0
    assert hip.hipMalloc(C.byref(dp), C.c_size_t(4 * (n + 1))) == 0
    m = np.asfortranarray(a, dtype=np.float64)     # column-major
    piv = np.full(n + 1, -1, np.int32)
    ptr = lambda x: C.c_void_p(x.ctypes.data)
    try:
        assert hip.hipMemcpy(da, ptr(m), C.c_size_t(m.nbytes), 1) == 0
        assert f(n, da, dp, C.c_void_p(dp.value + 4 * n), None) == 0
        assert hip.hipDeviceSynchronize() == 0
        assert hip.hipMemcpy(ptr(m), da, C.c_size_t(m.nbytes), 2) == 0
        assert hip.hipMemcpy(ptr(piv), dp, C.c_size_t(piv.nbytes), 2) == 0
    finally:
        hip.hipFree(da)
        hip.hipFree(dp)
    return m, piv[:n], int(piv[n])


# one column, a panel of 16 and its neighbours, several panels, two rows per thread
@pytest.mark.parametrize("n", [1, 15, 16, 17, 200, 1030])
def test_factors_in_the_order_of_dgetf2(n):
    a = np.random.default_rng(n).standard_normal((n, n))
    print(f"[eps] factors {n}", flush=True)
    got, piv, info = _factor(a)
    m, want = a.copy(order="F"), np.empty(n, int)
    for j in range(n):
        p = j + int(np.argmax(np.abs(m[j:, j])))
        want[j] = p
        m[[j, p]] = m[[p, j]]
        m[j + 1:, j] *= 1.0 / m[j, j]
        m[j + 1:, j + 1:] -= m[j + 1:, j, None] * m[j, j + 1:]
    assert info == 0 and np.array_equal(piv, want) and np.array_equal(got, m)


# a column of zeros stays one under every update: the pivot of that column is exactly zero, in the first
# panel, at a panel's first and last column, in the last panel, with one, two and four rows per thread
@pytest.mark.parametrize("n,col", [(1, 0), (40, 0), (40, 15), (40, 16), (40, 39), (1100, 700), (2100, 8), (2100, 2099)])
def test_zero_pivot_is_reported(n, col):
    a = np.random.default_rng(n + col).standard_normal((n, n))
    a[:, col] = 0.0
    print(f"[eps] zero pivot {n} {col}", flush=True)
    assert _factor(a)[2] == col + 1
