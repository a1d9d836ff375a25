"""State and fields to the host: what was uploaded comes back bit for bit, for sizes on both sides of
the pinned small download, of one staging slot and of the threaded copy's start, with a short
last piece, with rows and depths off the transposing tiles, and from two threads at once."""
import threading

import numpy as np
import pytest

from luma_amd.grid import GpuGrid

pytestmark = pytest.mark.gpu


def _round_trip(dims, n, m, k, seed):
    r = np.random.default_rng(seed)
    with GpuGrid(dims, 9 if dims == 2 else 19, n, m, k, precision="fp64", omega=1.2) as g:
        f = r.standard_normal((n, m, k, g.Q))
        rho, u = r.standard_normal((n, m, k)), r.standard_normal((n, m, k, dims))
        g.upload_f(f)
        g.upload_macro(rho, u)
        ck = g.checkpoint()
        out = (g.download_f(),) + g.download_macro()
        g.upload_f(-f)
        g.upload_macro(-rho, -u)
        g.restore(ck)
        GpuGrid.free_checkpoint(ck)
        again = (g.download_f(),) + g.download_macro()
    return all(np.array_equal(a, b) and np.array_equal(c, b) for a, c, b in zip(out, again, (f, rho, u)))


@pytest.mark.parametrize("size", [(2, 3, 3, 1), (2, 31, 33, 1), (2, 209, 209, 1), (2, 210, 209, 1), (2, 400, 700, 1),
                                  (3, 3, 3, 3), (3, 33, 5, 65), (3, 50, 41, 40), (3, 71, 60, 64), (3, 97, 101, 103)])
def test_what_went_up_comes_down(size):
    print(f"[copy] {size}", flush=True)
    assert _round_trip(*size, seed=1)


def test_two_threads():
    ok = [False, False]

    def work(i):
        ok[i] = all(_round_trip(3, 64, 70, 61 + i, seed=s) for s in range(3))
    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert ok == [True, True]
