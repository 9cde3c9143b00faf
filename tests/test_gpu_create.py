"""A handle's first calls find its buffers cleared, however soon they come:
creation clears them on the handle's own stream, ahead of every later call."""
import numpy as np
import pytest

from nemo_amd import _lib, indicator_mlp, mesh as meshmod, setups, solver

pytestmark = pytest.mark.gpu


def test_first_calls_of_new_handles():
    # each handle is likely to get the memory that the last one left full
    for k in range(8):
        p = indicator_mlp.init_params(k)
        with solver.Solver(solver.make_config()) as s:
            s.mlp_set_params(p)
            assert np.array_equal(s.mlp_get_params(), p), k
            assert s.get_glm() == (0.0, 0.0)
            s.set_glm(3.0, 5.0)


def test_first_run_of_new_batches():
    m = meshmod.uniform_periodic(3)
    cfg = solver.make_config(N=3, volume=_lib.VOL_EC, surface=_lib.SURF_HLLC, indicator=_lib.IND_PP,
                             timedisc=_lib.TD_SSPRK54, repair=1)
    u0 = setups.planar_riemann(m, 3, np.random.default_rng(1))
    first = None
    for k in range(4):
        with solver.Batch(cfg, [m], [3]) as b:
            b.upload(0, u0)
            dt = b.run(3, record_dt=True)
            u = b.download(0)
        first = (dt, u) if first is None else first
        assert (dt > 0.0).all(), k
        assert np.array_equal(dt, first[0]) and np.array_equal(u, first[1]), k
