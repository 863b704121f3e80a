"""The gradient kernel at the edges of its rounds of 64 samples and of its grid of 256 workgroups,
against the numpy restatement (the tolerances of the gradient test at other sizes)."""
import numpy as np
import pytest

from oracle import mlp_oracle as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 15, 63, 64, 65, 129, 16383, 16384, 16385, 33000])
def test_gradient_at_round_and_grid_edges(n):
    import torch
    if torch.cuda.device_count() < 1:
        pytest.fail("no GPU visible: the gpu tests need an MI355X")
    from akuaengine_amd import learned
    rng = np.random.default_rng(n)
    F = (rng.normal(size=(n, 16)) * rng.uniform(0.1, 10, 16) + rng.normal(size=16)).astype(np.float32)
    T = (rng.normal(size=(n, 4)) * np.array([0.3, 1.0, 0.1, 2.0])).astype(np.float32)
    p = M.random_params(rng, np.concatenate([F, -F]), np.concatenate([T, -T])).astype(np.float32)
    w = (1.0, 0.5, 2.0, 0.25)
    print(f"[mlp grad] n={n}", flush=True)
    loss, g = learned.mlp_gradient(p, F, T, w)
    le, ge = M.loss_and_grad(p, F, T, w, exact=False)
    assert loss == pytest.approx(le, rel=2e-3)
    assert np.linalg.norm(g - ge) < 2e-3 * np.linalg.norm(ge)
    for a, b in ((M.OFF_W1, M.OFF_B1), (M.OFF_W2, M.OFF_B2), (M.OFF_W3, M.OFF_B3), (M.OFF_B1, M.OFF_W2)):
        assert np.linalg.norm(g[a:b] - ge[a:b]) < 5e-3 * np.linalg.norm(ge[a:b]) + 1e-9, (a, b)
