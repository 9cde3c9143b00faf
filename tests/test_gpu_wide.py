"""The two forms of the stage kernel against each other: a state repeated
periodically on a mesh of so many blocks that the one-wavefront form runs must
evolve, repeat by repeat, like the state on the small mesh, where a block is
spread over four wavefronts.  Euler: the same bits (each form adds the same
terms in the same order; the learned indicator is left out, since its network
returns other last bits for another place of an element in its block, in
either form); GLM-MHD sums its rotated states in another order, so
its time derivative is compared to rounding.  The small meshes end in a block
that is not full (tiles of 7, 4 and 2 elements)."""
import numpy as np
import pytest

from nemo_amd import _lib, mesh as meshmod, setups, solver

pytestmark = pytest.mark.gpu

SMALL = (5, 3, 3)


def _tiled(n, reps):
    """Mesh of `reps` copies of the n box side by side in x (elements of the
    same size), and the small element of each of its elements."""
    small = meshmod.uniform_periodic(*n)
    big = meshmod.uniform_periodic(reps * n[0], n[1], n[2])
    at = lambda m, size: np.rint(m.lower / m.delta[0]).astype(int) % np.array(size)
    index = {tuple(c): e for e, c in enumerate(at(small, n))}
    src = np.array([index[tuple(c)] for c in at(big, n)])
    big.delta[:] = small.delta[0]
    return small, big, src


def _solvers(n, reps, ind, **kw):
    small, big, src = _tiled(n, reps)
    cfg = solver.make_config(indicator=ind, repair=1, **kw)
    out = []
    for m in (small, big):
        s = solver.Solver(cfg)
        s.upload_mesh(m)
        out.append(s)
    return small, out[0], out[1], src


EULER = [(N, prec, vol, surf, td, ind) for N in (2, 3, 4) for prec in (0, 1) for vol, surf, td, ind in (
    (_lib.VOL_EC, _lib.SURF_HLLC, _lib.TD_LSRK54, _lib.IND_PP),
    (_lib.VOL_CENTRAL, _lib.SURF_RUSANOV, _lib.TD_SSPRK54, _lib.IND_PP),
    (_lib.VOL_WEAK, _lib.SURF_RUSANOV, _lib.TD_SSPRK54, _lib.IND_NONE))]


@pytest.mark.parametrize("N,prec,vol,surf,td,ind", EULER)
def test_euler_same_bits(N, prec, vol, surf, td, ind):
    # one element more than the largest limit of blocks
    limit, tile = {2: (2048, 7), 3: (6144, 4), 4: (1536, 2)}[N]
    reps = limit * tile // int(np.prod(SMALL)) + 1
    mesh, s, b, src = _solvers(SMALL, reps, ind, N=N, volume=vol, surface=surf, timedisc=td, precision=prec)
    u = setups.planar_riemann(mesh, N, np.random.default_rng(N))
    u = u * (1.0 + 1e-3 * np.random.default_rng(7).standard_normal(u.shape))
    print(f"forms N={N} precision={prec} volume={vol} elements={len(src)}", flush=True)
    with s, b:
        s.set_state(u)
        b.set_state(u[src])
        assert np.array_equal(b.kernel_calc_flux(), s.kernel_calc_flux()[src])
        assert np.array_equal(b.run(3, record_dt=True), s.run(3, record_dt=True))
        assert np.array_equal(b.get_state(), s.get_state()[src])


@pytest.mark.parametrize("N", [2, 3, 4])
@pytest.mark.parametrize("prec", [0, 1])
def test_walls_and_open_sides(N, prec):
    """Boundary faces, whose fluxes both forms take from a launch before them:
    walls across y, open sides across z."""
    limit, tile = {2: (2048, 7), 3: (6144, 4), 4: (1536, 2)}[N]
    reps = limit * tile // int(np.prod(SMALL)) + 1
    small, big, src = _tiled(SMALL, reps)
    kinds = [None, None, meshmod.BC_SLIP_WALL, meshmod.BC_SLIP_WALL, meshmod.BC_TRANSMISSIVE, meshmod.BC_TRANSMISSIVE]
    cfg = solver.make_config(N=N, volume=_lib.VOL_EC, surface=_lib.SURF_HLLC, indicator=_lib.IND_PP, repair=1,
                             timedisc=_lib.TD_LSRK54, precision=prec)
    rng = np.random.default_rng(N)
    u = np.zeros((small.nelem, 5, (N + 1) ** 3))
    u[:, 0] = 1.0 + 0.2 * rng.random(u[:, 0].shape)
    u[:, 1:4] = 0.3 * rng.standard_normal(u[:, 1:4].shape)
    u[:, 4] = 2.5 + 0.5 * (u[:, 1:4] ** 2).sum(1)
    print(f"forms walls N={N} precision={prec} elements={len(src)}", flush=True)
    out = []
    for m, v in ((small, u), (big, u[src])):
        with solver.Solver(cfg) as s:
            s.upload_mesh(meshmod.with_boundaries(m, kinds))
            s.set_state(v)
            out.append(s.kernel_calc_flux())
    # the faces' fluxes are FP64 in both, to rounding (1e-12 and, through the
    # FP32 operator, 1e-5 of the largest value: the bounds of the boundary tests)
    tol = 1e-5 if prec else 1e-12
    for h in range(5):
        assert np.abs(out[1][:, h] - out[0][src][:, h]).max() <= tol * np.abs(out[1][:, h]).max(), h


@pytest.mark.parametrize("N,surf", [(2, _lib.SURF_HLLD), (3, _lib.SURF_HLLD), (3, _lib.SURF_RUSANOV),
                                    (4, _lib.SURF_RUSANOV)])
@pytest.mark.parametrize("prec", [0, 1])
def test_mhd_to_rounding(N, surf, prec):
    limit, tile = {2: (1200, 7), 3: (1536, 4), 4: (1536, 2)}[N]
    reps = limit * tile // int(np.prod(SMALL)) + 1
    mesh, s, b, src = _solvers(SMALL, reps, _lib.IND_PP, N=N, volume=_lib.VOL_EC, surface=surf,
                               timedisc=_lib.TD_LSRK54, precision=prec, equations=_lib.EQ_GLM_MHD, gamma=5.0 / 3.0)
    rng = np.random.default_rng(N)
    u = np.zeros((mesh.nelem, 9, (N + 1) ** 3))
    u[:, 0] = 1.0 + 0.2 * rng.random(u[:, 0].shape)
    u[:, 1:4] = 0.3 * rng.standard_normal(u[:, 1:4].shape)
    u[:, 5:9] = 0.2 * rng.standard_normal(u[:, 5:9].shape)
    u[:, 4] = 3.0 + 0.5 * (u[:, 1:4] ** 2).sum(1) + 0.5 * (u[:, 5:9] ** 2).sum(1)
    print(f"forms MHD N={N} precision={prec} surface={surf} elements={len(src)}", flush=True)
    with s, b:
        for x, v in ((s, u), (b, u[src])):
            x.set_state(v)
            x.set_glm(1.5, 8.0)
        r, q = s.kernel_calc_flux()[src], b.kernel_calc_flux()
    # both forms are within 1e-12 (FP64) and 4e-5 (FP32) of the exact result
    # relative to its largest value, per variable (tests of the MHD operator)
    tol = 8e-5 if prec else 2e-12
    for h in range(9):
        assert np.abs(r[:, h] - q[:, h]).max() <= tol * np.abs(q[:, h]).max(), h
