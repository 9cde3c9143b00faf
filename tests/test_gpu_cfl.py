"""The CFL reduction at the block counts where it changes: up to 2048 blocks
the last block of the launch reduces the partials (256 at a time), beyond them
a launch of its own.  The three extrema sit in elements of their own, in the
first, a middle and the last block in turn, so that no partial can be missed:
the largest signal speed, the largest velocity, and the smallest time step (by
the smallest element)."""
import itertools

import numpy as np
import pytest

from nemo_amd import _lib, mesh as meshmod, setups, solver
from oracle import oracle as O

pytestmark = pytest.mark.gpu

TILE = {2: 7, 3: 4, 4: 2}


def _state(nelem, N, fast, moving):
    M3 = (N + 1) ** 3
    rng = np.random.default_rng(nelem)
    rho = 1.0 + 0.1 * rng.random((nelem, M3))
    v = 0.1 * rng.standard_normal((3, nelem, M3))
    p = np.full((nelem, M3), 1.0)
    p[fast] = 6.0     # sound speed 2.9 against 1.2
    v[1, moving] = 1.5  # signal speed 2.7
    return np.ascontiguousarray(setups.prim2cons(rho, v[0], v[1], v[2], p, 1.4))


@pytest.mark.parametrize("N", [2, 3, 4])
@pytest.mark.parametrize("blocks", [1, 3, 257, 743, 2047, 2048, 2049])
def test_extrema_in_any_block(N, blocks):
    n = blocks * TILE[N] - (1 if blocks > 1 else 0)  # the last block is not full
    m = meshmod.uniform_periodic(n, 1, 1)
    kw = dict(N=N, volume=_lib.VOL_EC, surface=_lib.SURF_HLLC, timedisc=_lib.TD_LSRK54, repair=1)
    g, o = solver.make_config(indicator=_lib.IND_PP, **kw), O.make_cfg(indicator=O.IND_PP, **kw)
    places = sorted({0, n // 2, n - 1})
    print(f"CFL N={N} blocks={blocks}: elements {places}", flush=True)
    with solver.Solver(g) as s:
        for fast, moving, small in itertools.permutations(places) if len(places) == 3 else [(0, 0, 0)]:
            m.delta[:] = 1.0
            m.delta[small] = 0.25
            u0 = _state(n, N, fast, moving)
            s.upload_mesh(m)
            s.set_state(u0)
            ref = O.calc_timestep(o, m.delta, u0)
            # (the parity bound of the time step)
            assert all(abs(x - y) <= 1e-15 * y for x, y in zip(s.hook_calc_timestep(), ref))
            for form in (_lib.FORM_ONE_WAVE, _lib.FORM_FOUR_WAVES):
                s.set_form(form)
                s.set_state(u0)
                s.run(1)
                dt, lm, vm = O.calc_timestep(o, m.delta, s.get_state())
                # the reduction behind the first of two steps
                s.set_state(u0)
                hist = s.run(2, record_dt=True)
                assert abs(hist[0] - ref[0]) <= 1e-15 * ref[0]
                assert abs(hist[1] - dt) <= 1e-15 * dt, form
                assert abs(s.get_glm()[0] - 2.0 * abs(lm - vm)) <= 4e-15 * lm, form
