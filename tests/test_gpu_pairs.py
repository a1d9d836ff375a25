"""Two steps per launch on large 3D grids (lumagpu_run in FP32-shifted storage) against single steps,
bit for bit in every population a download reads and in the macro arrays: extents off the tiles,
walls with a set force field, an inflow with outlet and an immersed sphere, velocity walls meeting
at edges and corners, a pressure outlet; odd and even counts from both layouts; a restored state,
new labels and new populations between runs; and the switch that turns it off."""
import numpy as np
import pytest

from luma_amd import setups
from luma_amd.grid import GpuGrid

pytestmark = pytest.mark.gpu


def _walls():
    case = setups.body_force_channel(90, 83, 75, 3, g=1e-5)
    case.force[..., 2] = 1e-6 * np.cos(np.arange(case.K))
    case.lattyp[20:30, 40:44, 30:33] = setups.SOLID
    case.u[..., 0] = 0.02 * np.sin(np.arange(case.M))[None, :, None]
    case.u[case.lattyp == setups.SOLID] = 0.0
    return case


def _sphere():
    case = setups.uniform_inflow_3d(121, 70, 66, 0.03, 0.6)
    case.lattyp[60:64, 5:9, 7:12] = setups.SOLID
    return case


CASES = {
    "ragged": lambda: setups.taylor_green((85, 81, 79), u0=0.04, tau=0.6),
    "tiles": lambda: setups.taylor_green((128, 64, 65), u0=0.04, tau=0.6),
    "thin": lambda: setups.taylor_green((700, 250, 3), u0=0.04, tau=0.6),
    "walls": _walls,
    "sphere": _sphere,
    "corners": lambda: setups.velocity_corner_box(84, 80, 79, dims=3),
    "ramp": lambda: setups.uniform_inflow_3d(121, 70, 66, 0.03, 0.6),
    "pressure": lambda: setups.pressure_outlet_duct(90, 80, 75, dims=3),
}


def _grid(name, case):
    g = GpuGrid.from_case(case, "fp32s", store_macro=True)
    if name == "sphere":
        g.ibm_add_body(setups.sphere_markers((40.3, 35.1, 33.2), 6.0, 1.0))
        g.ibm_initialise()
    if name == "ramp":
        g.set_velocity_ramp(21.0)   # ends within the third run
    return g


def _same(a, b):
    return all(np.array_equal(p, q) for p, q in zip((a.download_f(),) + a.download_macro(),
                                                   (b.download_f(),) + b.download_macro()))


@pytest.mark.parametrize("name", list(CASES))
def test_matches_single_steps(name):
    case = CASES[name]()
    print(f"[pairs] {name} {case.N}x{case.M}x{case.K}", flush=True)
    with _grid(name, case) as a, _grid(name, case) as b:
        for steps in (7, 6, 5, 12):
            a.run(steps)
            for _ in range(steps):
                b.LBM_multi_opt()
            assert a.t == b.t
            assert _same(a, b), steps
        if name == "sphere":
            assert np.array_equal(a.ibm_markers(0)["force"], b.ibm_markers(0)["force"])
        # a restored state, other populations, other labels: nothing of the second array comes back
        ck = a.checkpoint()
        a.run(9)
        a.restore(ck)
        GpuGrid.free_checkpoint(ck)
        assert _same(a, b)
        f = b.download_f() * (1.0 + 1e-4 * np.arange(19))
        if case.lattyp is not None and name != "sphere":
            lt = case.lattyp.copy()
            lt[10:16, 20:24, 30:35] = setups.SOLID
            for g in (a, b):
                g.set_labels(lt, case.xpos, case.ypos, case.zpos)
        for g in (a, b):
            g.upload_f(f)
        a.run(8)
        for _ in range(8):
            b.LBM_multi_opt()
        assert _same(a, b)
        a.set_temporal_blocking(-1)
        a.run(7)
        for _ in range(7):
            b.LBM_multi_opt()
        assert _same(a, b)
