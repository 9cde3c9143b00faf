"""An error belongs to the call that caused it: state transfers and launches of
one handle work after an allocation of another one has failed in the same
thread."""
import numpy as np
import pytest

from nemo_amd import _lib, indicator_mlp, mesh as meshmod, setups, solver

pytestmark = pytest.mark.gpu


def test_transfers_after_a_failed_allocation():
    with solver.Solver(solver.make_config(N=3)) as s, solver.Solver(solver.make_config()) as other:
        s.upload_mesh(meshmod.uniform_periodic(3))
        other.mlp_set_params(indicator_mlp.init_params(1))
        u = np.random.default_rng(1).standard_normal((s.nelem, 5, s.M3))
        x = np.zeros(4, np.float32)

        def fail():
            with pytest.raises(_lib.NemoGpuError):  # 2^48 bytes of features
                other._call("nemo_gpu_mlp_forward", other._h, 1 << 44, solver.fptr(x), solver.fptr(x))

        for _ in range(2):
            fail()
            s.set_state(u)
            fail()
            assert np.array_equal(s.get_state(), u)


def test_launches_after_a_failed_allocation():
    with solver.Solver(solver.make_config(N=3)) as s, solver.Solver(solver.make_config()) as other:
        m = meshmod.uniform_periodic(3)
        s.upload_mesh(m)
        s.set_state(setups.isentropic_vortex(m, 3))
        other.mlp_set_params(indicator_mlp.init_params(1))
        x = np.zeros(4, np.float32)
        for call in (s.kernel_calc_flux, s.hook_calc_timestep, lambda: s.run(1)):
            with pytest.raises(_lib.NemoGpuError):
                other._call("nemo_gpu_mlp_forward", other._h, 1 << 44, solver.fptr(x), solver.fptr(x))
            call()
