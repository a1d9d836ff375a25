"""Programs that run the library short of device memory, or with a failing launch, one per name, each in a process of its own
(test_gpu_memory.py): the limiter has to be loaded before the library.  A scenario raises where it
fails and prints its name at the end."""
import ctypes as C
import dataclasses
import sys
import threading
from pathlib import Path

import numpy as np

HERE = Path(__file__).resolve().parent
sys.path.insert(0, str(HERE.parent))
limit = C.CDLL(str(HERE / "cpp" / "_build" / "alloc_limit.so"), mode=C.RTLD_GLOBAL)
limit.limit_budget.argtypes = [C.c_longlong]
limit.limit_refuse_size.argtypes = limit.limit_refuse_until_freed.argtypes = [C.c_size_t]
limit.limit_show_total.argtypes = [C.c_size_t]
limit.limit_held.restype = C.c_size_t

from luma_amd import setups  # noqa: E402
from luma_amd._abi import LumaGpuError  # noqa: E402
from luma_amd.grid import GpuGrid  # noqa: E402

MB = 1 << 20


def walls(n=70):
    """FP32-shifted labelled box of n^3 cells with a set force: run() takes two steps per launch."""
    case = setups.body_force_channel(n, n, n, 3, g=1e-5)
    case.u[..., 0] = 0.02 * np.sin(np.arange(n))[None, :, None]
    case.u[case.lattyp == setups.SOLID] = 0.0
    return case


def grid(case, form="fp32s"):
    return GpuGrid.from_case(case, form, store_macro=True)


def state(g):
    return (g.download_f(),) + g.download_macro()


def single_steps(case, n, form="fp32s"):
    with grid(case, form) as g:
        for _ in range(n):
            g.LBM_multi_opt()
        return state(g)


def same(a, b):
    assert all(np.array_equal(x, y) for x, y in zip(a, b))


def labels_cut_short():
    # the link words of new labels do not fit: the call fails and steps are refused, until the labels
    # have been set; nothing reads a part of them
    case = setups.lid_driven_cavity(40, re=200.0)
    box = dataclasses.replace(case, lattyp=None)
    with grid(box) as g, grid(box) as h:
        g.run(4)
        h.run(4)
        limit.limit_refuse_size(8 * 40 * 40)
        try:
            g.set_labels(case.lattyp, case.xpos, case.ypos, case.zpos)
            raise AssertionError("link words allocated")
        except LumaGpuError as e:
            assert "allocation" in str(e)
        for step in (lambda: g.run(6), lambda: g.run(1), g.LBM_multi_opt, g.stream_bc_macro):
            try:
                step()
                raise AssertionError("stepped")
            except LumaGpuError as e:
                assert "set them again" in str(e)
        limit.limit_refuse_size(0)
        for x in (g, h):
            x.set_labels(case.lattyp, case.xpos, case.ypos, case.zpos)
            x.run(6)
        same(state(g), state(h))


def sets_do_not_fit():
    # two steps per launch need bitmaps and lists of sites; single steps do not
    case = walls()
    words = (70 ** 3 + 31) // 32 + 1
    with grid(case) as g:
        limit.limit_refuse_size(4 * words)
        g.run(9)
        assert limit.limit_refusals() > 0
        same(state(g), single_steps(case, 9))
        limit.limit_refuse_size(0)
        g.run(9)
        same(state(g), single_steps(case, 18))


def sets_take_back():
    # an allocation inside a run takes the arrays of other grids back, and spares the one in use
    case = walls()
    words = (70 ** 3 + 31) // 32 + 1
    with grid(case) as a, grid(case) as b:
        b.run(9)
        limit.limit_refuse_until_freed(4 * words)
        a.run(9)
        assert limit.limit_refusals() == 1
        want = single_steps(case, 9)
        same(state(a), want)
        same(state(b), want)
        for g in (a, b):
            g.run(8)
        want = single_steps(case, 17)
        same(state(a), want)
        same(state(b), want)


def others_give_way():
    # with no memory left but another grid's second array: labels, outlet, bodies and their steps
    case = setups.uniform_inflow_3d(60, 50, 44, 0.03, 0.6)
    pos = setups.sphere_markers((20.3, 25.1, 22.2), 5.0, 1.0)

    class Tight(GpuGrid):
        def set_labels(self, *a):
            limit.limit_budget(0)
            super().set_labels(*a)

    def flow(cls):
        with cls.from_case(case, "fp64", store_macro=True) as g:
            limit.limit_budget(-1)
            if cls is Tight:
                b2 = grid(walls())
                b2.run(9)
                limit.limit_budget(0)
            g.ibm_add_body(pos)
            g.ibm_initialise()
            g.run(4)
            limit.limit_budget(-1)
            return state(g)

    want = flow(GpuGrid)
    with grid(walls()) as b:
        b.run(9)
        same(flow(Tight), want)
        assert limit.limit_refusals() >= 2
        b.run(8)
        same(state(b), single_steps(walls(), 17))


def epsilon_on_the_host():
    # ibm_initialise needs no device memory for its marker system
    n = 300
    case = setups.uniform_inflow_3d(30, 26, 26, 0.03, 0.6)
    pos = setups.sphere_markers((13.1, 13.2, 13.3), 5.0, 1.0, n=n)
    limit.limit_refuse_size(8 * n * n)
    with grid(case, "fp64") as g:
        g.ibm_add_body(pos)
        g.ibm_initialise()
        assert np.isfinite(g.ibm_markers(0)["eps"]).all() and limit.limit_refusals() == 0


def position_gradient_on_the_host():
    # the same sums in another order: n markers' terms, each rounded at 1e-16 of the largest
    n = 200
    case = setups.uniform_inflow_3d(30, 26, 26, 0.03, 0.6)
    pos = setups.sphere_markers((13.1, 13.2, 13.3), 4.0, 1.0, n=n)
    out = []
    for size in (0, 8 * n * n):
        limit.limit_refuse_size(size)
        with grid(case, "fp64") as g:
            g.ibm_add_body(pos)
            g.ibm_initialise()
            out.append(g.adj_run(5, 3))
        assert limit.limit_refusals() == (2 if size else 0)      # tried again after taking back
    a, b = out
    assert a["J"] == b["J"]
    g = np.abs(a["dJ_dpos"]).max()
    assert g > 0 and np.abs(a["dJ_dpos"] - b["dJ_dpos"]).max() <= 1e-11 * g


def force_set_again():
    # other forces leave the site types, and with them the sets of two steps per launch, as they are
    case = walls()
    force = [case.force, 2.0 * case.force, case.force.copy()]
    force[2][20:40, 10:30] = 0.0                # other force bits
    with grid(case) as a, grid(case) as b:
        for f in force:
            calls = limit.limit_calls()
            for g in (a, b):
                g.set_force(f)
            a.run(9)
            if f is not force[0]:
                assert limit.limit_calls() == calls, "sets or arrays made again"
            for _ in range(9):
                b.LBM_multi_opt()
            same(state(a), state(b))


def labels_set_again():
    # new labels of a small grid go into the arrays that it has
    case = setups.lid_driven_cavity(40, re=200.0)
    lt = [case.lattyp, case.lattyp.copy()]
    lt[1][10:15, 12:20] = setups.SOLID
    with grid(case, "fp64") as g:
        calls = limit.limit_calls()
        for k in (1, 0, 1):
            g.set_labels(lt[k], case.xpos, case.ypos, case.zpos)
        assert limit.limit_calls() == calls
        for _ in range(5):
            g.LBM_multi_opt()
        got = state(g)
    case.lattyp = lt[1]
    same(got, single_steps(case, 5, "fp64"))


def short_runs_step_singly():
    # too short for several steps per launch: no second array for them
    for n, form, steps in ((48, "fp64", 7), (400, "fp64", 3), (48, "fp32s", 3)):
        with GpuGrid.from_case(setups.taylor_green((n, n, 1), u0=0.04, tau=0.6, dims=2), form) as g:
            calls = limit.limit_calls()
            for _ in range(3):
                g.run(steps)
            assert limit.limit_calls() == calls, (n, form)
            g.run(40)
            assert limit.limit_calls() == calls + 1, (n, form)


def current_device_stays():
    # a large download copies on the caller's thread too: its current device is what it was
    f = np.random.default_rng(1).standard_normal((60, 70, 64, 19))      # 40 MB: several pieces
    with GpuGrid(3, 19, 60, 70, 64, precision="fp64", omega=1.2) as g:
        g.upload_f(f)
        limit.limit_show_device(-1)
        assert np.array_equal(g.download_f(), f) and limit.limit_set_device_calls() == 0
        limit.limit_show_device(1)
        assert np.array_equal(g.download_f(), f) and limit.limit_shown_device() == 1
        limit.limit_show_device(-1)


def run_from_another_device():
    # what a run takes for itself would lie on the caller's device: single steps need nothing there
    case, box = walls(), setups.taylor_green((64, 50, 1), u0=0.04, tau=0.6, dims=2)
    want = single_steps(case, 18), single_steps(box, 40)
    with grid(case) as g, grid(box) as h:
        g.run(9)
        calls = limit.limit_calls()
        limit.limit_show_device(1)
        g.run(9)
        h.run(40)
        assert limit.limit_calls() == calls
        limit.limit_show_device(-1)
        same(state(g), want[0])
        same(state(h), want[1])


def kept_memory_is_bounded():
    # second arrays and adjoint blocks of all grids together: a sixteenth of the device's memory
    case = walls()
    f2 = (-(-70 ** 3 // 256) * 256) * 19 * 4          # and the planes' padding: below 1 % more
    limit.limit_show_total(int(16 * 1.5 * f2))
    want = single_steps(case, 9)
    with grid(case) as a:
        before = limit.limit_held()
        a.run(9)
        assert limit.limit_held() > before + f2, "no second array"
        with grid(case) as b:
            state(b)                                  # its staging
            before = limit.limit_held()
            b.run(9)
            assert limit.limit_held() == before, "a second array beyond the bound"
            same(state(b), want)
            a.close()
            b.init_equilibrium(case.rho, case.u)
            before = limit.limit_held()
            b.run(9)
            assert limit.limit_held() > before + f2
            same(state(b), want)
    box = setups.channel_2d(90, 40, 10.0, 0.04, 20.0)
    grads = []
    for total in (1 << 40, 16 << 10):
        limit.limit_show_total(total)
        with grid(box, "fp64") as g:
            g.ibm_add_body(setups.circle_markers((3.0, 2.0, 0.0), 0.5, box.info["dh"]))
            g.ibm_initialise()
            start = g.checkpoint()
            state(g)
            before = limit.limit_held()
            for _ in range(2):
                g.restore(start)
                grads.append(g.adj_run(20, 6, initial=True))
                if total < 1 << 40:
                    assert limit.limit_held() == before, "blocks beyond the bound"
            assert total < 1 << 40 or limit.limit_held() > before
            GpuGrid.free_checkpoint(start)
    for r in grads[1:]:
        assert r["J"] == grads[0]["J"] and np.array_equal(r["lambda0"], grads[0]["lambda0"])


def threads_short_of_memory():
    # one thread steps while another's grids come, run and go in memory that holds one second array less
    case = walls(66)
    want = {n: single_steps(case, n) for n in (9, 18, 27)}
    size = 66 ** 3 * 19 * 4
    with grid(case) as a, grid(case) as b:
        state(a)
        limit.limit_budget(int(7.2 * size))       # b's grids (f, rho, u, force, staging): 5 x size, and two arrays
        out, errors = {}, []

        def stepping():
            try:
                for n in (9, 18, 27):
                    a.run(9)
                    out[n] = state(a)
            except Exception as e:
                errors.append(e)

        def coming_and_going():
            try:
                for _ in range(4):
                    b.init_equilibrium(case.rho, case.u)
                    b.run(9)
                    same(state(b), want[9])
                    with grid(case) as c:
                        c.run(9)
                        same(state(c), want[9])
            except Exception as e:
                errors.append(e)
        threads = [threading.Thread(target=t) for t in (stepping, coming_and_going)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        limit.limit_budget(-1)
    assert not errors, errors
    for n in out:
        same(out[n], want[n])


def second_array_refused():
    # a second array that would take more than half of what is free: single steps
    case, box = walls(), setups.taylor_green((64, 50, 1), u0=0.04, tau=0.6, dims=2)
    want = single_steps(case, 9), single_steps(box, 40)
    with grid(case) as g, grid(box) as h:
        for x, cells, q, steps in ((g, 70 ** 3, 19, 9), (h, 64 * 50, 9, 40)):
            calls = limit.limit_calls()
            limit.limit_budget(int(1.9 * cells * q * 4))
            x.run(steps)
            assert limit.limit_calls() == calls
            limit.limit_budget(-1)
        same(state(g), want[0])
        same(state(h), want[1])


def gradient_cut_short():
    # a gradient that runs out of memory between its forward and its reversed steps, then the same again
    case = setups.channel_2d(90, 40, 10.0, 0.04, 20.0)
    with grid(case, "fp64") as g:
        g.ibm_add_body(setups.circle_markers((3.0, 2.0, 0.0), 0.5, case.info["dh"]))
        g.ibm_initialise()
        start = g.checkpoint()
        limit.limit_refuse_size(3 * 8 * 90 * 40)      # the force adjoint
        for _ in range(3):
            g.restore(start)
            try:
                g.adj_run(20, 6, initial=True)
                raise AssertionError("allocated")
            except LumaGpuError as e:
                assert "adjoint buffer" in str(e)
        limit.limit_refuse_size(0)
        got = []
        for _ in range(2):
            g.restore(start)
            got.append(g.adj_run(20, 6, initial=True))
        GpuGrid.free_checkpoint(start)
    with grid(case, "fp64") as g:
        g.ibm_add_body(setups.circle_markers((3.0, 2.0, 0.0), 0.5, case.info["dh"]))
        g.ibm_initialise()
        want = g.adj_run(20, 6, initial=True)
    assert np.abs(want["lambda0"]).max() > 0
    for r in got:
        for k in want:
            assert np.array_equal(r[k], want[k]), k


def launch_errors_are_reported():
    # a grid of plain sites alone steps in one launch, without a list after it
    shape = (104, 101, 102)
    case = setups.taylor_green(shape, u0=0.04, tau=0.7)
    case.forced, case.force = True, np.full(shape + (3,), 1e-6)
    with GpuGrid.from_case(case, "fp64") as g:
        g.run(2)
        limit.limit_fail_launch(1)
        try:
            g.LBM_multi_opt()
            raise AssertionError("a failed launch was taken for a step")
        except LumaGpuError as e:
            assert "launch" in str(e)
        assert g.t == 2


if __name__ == "__main__":
    print(f"[memory] {sys.argv[1]}", flush=True)
    globals()[sys.argv[1]]()
    assert limit.limit_calls() > 0, "the library's allocations do not come through the limiter"
    print(f"done {sys.argv[1]}", flush=True)
