"""Outputs and gradients of the learned indicator's batch kernels (tiles of 16
samples, up to 256 gradient workgroups, 1024 output workgroups) at the sizes
where a tile or a round of workgroups ends, against the FP64 reference; the
bounds are those of the indicator's other tests."""
import numpy as np
import pytest

from nemo_amd import indicator_mlp, solver
from oracle import mlp_ref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 15, 16, 17, 4096, 4097, 16384, 16399])
def test_tiles(n):
    rng = np.random.default_rng(n)
    p = indicator_mlp.init_params(5)
    X = rng.normal(-1.0, 0.7, (n, 4)).astype(np.float32)
    t = rng.uniform(0, 0.5, n).astype(np.float32)
    print(f"mlp tiles n={n}", flush=True)
    with solver.Solver(solver.make_config()) as s:
        s.mlp_set_params(p)
        loss, g = s.mlp_grad(X, t)
        y = s.mlp_forward(X)
    p64, X64 = p.astype(np.float64), X.astype(np.float64)
    lref, gref = mlp_ref.loss_grad(p64, X64, t.astype(np.float64))
    yref, _ = mlp_ref.forward(p64, X64)
    assert np.abs(y - yref).max() <= 2e-6
    assert abs(loss - lref) <= 1e-5 * lref
    assert np.abs(g - gref).max() <= 1e-4 * np.abs(gref).max()
