"""The parity tests of the stage kernel in each of its two forms.

Which form a mesh takes depends on its number of blocks, and the meshes of the
parity tests are small: by themselves they reach the form of four wavefronts
per block only.  Here those tests run again with the form given
(Solver.set_form): the near-1 log-means and the update fused into the x pass,
partial blocks, repair, mortars, boundary faces, the learned indicator and
GLM-MHD on one wavefront per block, which large meshes take, and the same on
four, whatever the rule's limits are."""
import itertools

import numpy as np
import pytest

import test_gpu_amr
import test_gpu_boundaries
import test_gpu_fp32
import test_gpu_mhd
import test_gpu_mlp
import test_gpu_parity
from nemo_amd import _lib, mesh as meshmod, setups, solver
from oracle import oracle as O

pytestmark = pytest.mark.gpu

FORMS = {"one": _lib.FORM_ONE_WAVE, "four": _lib.FORM_FOUR_WAVES}

SUITE = [(test_gpu_parity, ["test_rhs_parity", "test_run_100_steps", "test_stage_api_matches_run",
                            "test_repair_parity", "test_partial_last_block", "test_near1_log_means_at_their_bound"]),
         (test_gpu_amr, ["test_amr_rhs_parity", "test_amr_run_parity_and_conservation", "test_amr_fp32_operator",
                         "test_mhd_amr_rhs_parity", "test_mhd_amr_run_parity", "test_mhd_amr_fp32_operator"]),
         (test_gpu_boundaries, ["test_boundary_rhs_parity", "test_boundary_run_parity", "test_boundary_fp32_operator",
                                "test_mhd_transmissive_parity"]),
         (test_gpu_fp32, ["test_fp32_rhs_against_fp64_oracle", "test_fp32_100_steps_l1_density_error"]),
         (test_gpu_mhd, ["test_mhd_rhs_parity", "test_mhd_fp32_rhs_against_fp64_oracle",
                         "test_mhd_run_parity_100_steps", "test_mhd_other_degrees_rhs_and_run"]),
         (test_gpu_mlp, ["test_features_and_fused_inference", "test_judge_and_fallback", "test_sampled_judge_fraction",
                         "test_trained_network_gain_on_sedov",
                         "test_diagnostics_between_stages_leave_the_step_untouched"])]


def _expand():
    """Every test of the suite with the arguments of its parametrize marks."""
    for mod, names in SUITE:
        for name in names:
            fn = getattr(mod, name)
            marks = getattr(fn, "pytestmark", [])
            axes = []
            for m in marks:
                if m.name == "parametrize":
                    keys = [k.strip() for k in m.args[0].split(",")]
                    axes.append([dict(zip(keys, v if len(keys) > 1 else (v,))) for v in m.args[1]])
            skips = [m for m in marks if m.name in ("skip", "skipif")]
            for i, combo in enumerate(itertools.product(*axes)):
                kw = {k: v for part in combo for k, v in part.items()}
                yield pytest.param(fn, kw, id=f"{mod.__name__[9:]}-{name[5:]}-{i}", marks=skips)


def _one_wave_built(cfg):
    return not (cfg.equations == _lib.EQ_GLM_MHD and cfg.surface == _lib.SURF_HLLD and cfg.n_poly == 4)


@pytest.fixture(params=list(FORMS))
def forced(request, monkeypatch):
    """Every solver made in the test has the form."""
    class Forced(solver.Solver):
        def __init__(self, cfg):
            super().__init__(cfg)
            if _one_wave_built(cfg):
                self.set_form(FORMS[request.param])

    monkeypatch.setattr(solver, "Solver", Forced)
    return request.param


@pytest.mark.parametrize("fn,kw", list(_expand()))
def test_parity(forced, fn, kw):
    print(f"form {forced}: {fn.__name__} {kw}", flush=True)
    fn(**kw)


def test_invalid_forms_are_refused():
    with solver.Solver(solver.make_config()) as s:
        for form in (-1, 3):
            with pytest.raises(_lib.NemoGpuError):
                s.set_form(form)
    cfg = solver.make_config(N=4, volume=_lib.VOL_EC, surface=_lib.SURF_HLLD, equations=_lib.EQ_GLM_MHD, gamma=5 / 3)
    with solver.Solver(cfg) as s:
        with pytest.raises(_lib.NemoGpuError, match="four wavefronts"):
            s.set_form(_lib.FORM_ONE_WAVE)


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("surf", [_lib.SURF_HLLC, _lib.SURF_RUSANOV])
def test_learned_stages_in_both_forms(prec, surf):
    """The learned indicator's first stage (network) and its others (stored
    factor): a network of one constant output has no rounding of its own, so
    both forms give the same bits, and the time derivative is the oracle's
    with that factor.  45 elements end in a block that is not full."""
    m = meshmod.uniform_periodic(5, 3, 3)
    m.delta[:] = m.delta[0]
    kw = dict(N=3, volume=_lib.VOL_EC, surface=surf, timedisc=_lib.TD_LSRK54, repair=1)
    u0 = setups.planar_riemann(m, 3, np.random.default_rng(2))
    u0 = u0 * (1.0 + 1e-3 * np.random.default_rng(3).standard_normal(u0.shape))
    p = np.zeros(_lib.MLP_NPARAMS, np.float32)
    p[-1] = -1.0  # the output's bias
    factor = 1.0 / (1.0 + np.exp(1.0))
    print(f"learned forms precision={prec} surface={surf}", flush=True)
    out = []
    for form in FORMS.values():
        with solver.Solver(solver.make_config(indicator=_lib.IND_MLP, precision=prec, **kw)) as s:
            s.set_form(form)
            s.upload_mesh(m)
            s.set_state(u0)
            s.mlp_set_params(p)
            s.mlp_set_policy(0.0, 0.05)
            out.append((s.kernel_calc_flux(), s.run(4, record_dt=True), s.get_state()))
            a = s.indicator()
    assert all(np.array_equal(x, y) for x, y in zip(*out))
    # the factor is FP32 (5 roundings of its sigmoid); the operator's bounds are
    # those of the parity tests, and a factor's error enters with a weight below one
    assert np.abs(a - factor).max() <= 5 * 2.0 ** -24
    if prec == 0:
        s0 = O.make_cfg(N=3, volume=_lib.VOL_EC, surface=surf, indicator=O.IND_PP, timedisc=_lib.TD_LSRK54, repair=1)
        ref = O.rhs(s0, m.nbr, m.delta, u0, a)
        assert np.abs(out[0][0] - ref).max() <= 1e-12 * np.abs(ref).max()


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("N", [2, 3, 4])
def test_mortars_same_bits(N, prec):
    f = test_gpu_amr._forest()
    u0 = test_gpu_amr._state(f, N)
    cfg, _ = test_gpu_amr._cfgs(f, N, _lib.VOL_EC, _lib.SURF_HLLC, _lib.IND_PP, repair=1, precision=prec)
    print(f"mortar forms N={N} precision={prec}", flush=True)
    out = []
    for form in FORMS.values():
        with solver.Solver(cfg) as s:
            s.set_form(form)
            s.upload_mesh(f)
            s.set_state(u0)
            out.append((s.kernel_calc_flux(), s.run(3, record_dt=True), s.get_state()))
    assert all(np.array_equal(x, y) for x, y in zip(*out))


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("use_graph", [True, False])
@pytest.mark.parametrize("form", list(FORMS))
def test_batch_groups_match_single_runs(form, use_graph, precision):
    """Degree groups with launches of their own, side by side, in each form:
    run by run the bits of single solvers of that form."""
    import test_gpu_batch
    meshes, npolys, states = test_gpu_batch._runs()
    cfg = solver.make_config(N=3, precision=precision, **test_gpu_batch.KW)
    print(f"batch form {form} graph={use_graph} precision={precision}", flush=True)
    with solver.Batch(cfg, meshes, npolys) as b:
        b.set_launch(0, xcd_map=False, one_launch=False)
        b.set_form(FORMS[form])
        for r, u in enumerate(states):
            b.upload(r, u)
        dts = np.concatenate([b.run(4, use_graph=use_graph, record_dt=True) for _ in range(2)])
        ub = [b.download(r) for r in range(len(states))]
    for r, (m, N, u0) in enumerate(zip(meshes, npolys, states)):
        with solver.Solver(solver.make_config(N=N, precision=precision, **test_gpu_batch.KW)) as s:
            s.set_form(FORMS[form])
            s.upload_mesh(m)
            s.set_state(u0)
            d = np.concatenate([s.run(4, record_dt=True) for _ in range(2)])
            us = s.get_state()
        assert np.array_equal(d, dts[:, r]), r
        assert np.array_equal(us, ub[r]), r
