"""State transfers between the host layout u[elem][var][node] and the device
layout: what was uploaded comes back bit for bit, below and above the size at
which the staged copy takes over, with a last chunk that is not full, for
every degree and equation system, and from two threads at once."""
import threading

import numpy as np
import pytest

from nemo_amd import _lib, mesh as meshmod, solver

pytestmark = pytest.mark.gpu


def _solver(N, eq, n):
    mhd = eq == _lib.EQ_GLM_MHD
    cfg = solver.make_config(N=N, volume=_lib.VOL_EC, surface=_lib.SURF_HLLD if mhd else _lib.SURF_HLLC,
                             indicator=_lib.IND_PP, timedisc=_lib.TD_LSRK54, repair=1, equations=eq)
    s = solver.Solver(cfg)
    s.upload_mesh(meshmod.uniform_periodic(*n))
    return s


# one element; 4 MB less and more than a row; odd sizes through each chunk size
@pytest.mark.parametrize("N,eq,n", [
    (2, _lib.EQ_EULER, (1, 1, 1)), (3, _lib.EQ_EULER, (3, 5, 7)), (4, _lib.EQ_EULER, (29, 29, 1)),
    (2, _lib.EQ_EULER, (17, 19, 12)), (2, _lib.EQ_EULER, (17, 19, 13)), (4, _lib.EQ_GLM_MHD, (5, 7, 17)),
    (3, _lib.EQ_GLM_MHD, (23, 19, 17)), (3, _lib.EQ_EULER, (41, 37, 43)),
])
def test_round_trip(N, eq, n):
    with _solver(N, eq, n) as s:
        rng = np.random.default_rng(3)
        for _ in range(2):  # the second pass finds the buffers in use before
            u = rng.standard_normal((s.nelem, s.nvars, s.M3))
            s.set_state(u)
            assert np.array_equal(s.get_state(), u)


def test_two_threads_at_once():
    ok = [False, False]

    def body(k):
        with _solver(3, _lib.EQ_EULER, (19, 17, 16 + k)) as s:
            rng = np.random.default_rng(k)
            good = True
            for _ in range(4):
                u = rng.standard_normal((s.nelem, 5, s.M3))
                s.set_state(u)
                good = good and np.array_equal(s.get_state(), u)
            ok[k] = good

    th = [threading.Thread(target=body, args=(k,)) for k in range(2)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert all(ok)
