"""Crowded scenes against the FP32 oracle, order by order and list by list: some thousands of coincident
particles, a crowded cell and its neighbours beside ordinary ones, in single scenes of both orderings, with
caps from a few entries to more than a cell holds."""
import dataclasses

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
DT = 0.004


@pytest.fixture(scope="module")
def gpu():
    import torch
    if torch.cuda.device_count() < 1:
        pytest.fail("no GPU visible: the gpu tests need an MI355X")
    from akuaengine_amd.solver import PBFSolver
    return PBFSolver


def _crowd(n, coincident, seed):
    """n particles in a box of 4 x 4 x 4: some at one point, as many in that cell's surroundings, a few
    pairs at one point, the others anywhere."""
    rng = np.random.default_rng(seed)
    pos = rng.uniform(0.1, 3.9, (n, 3))
    pos[:coincident] = (1.03, 1.07, 1.02)
    pos[coincident:2 * coincident] = 1.0 + rng.uniform(-0.1, 0.2, (coincident, 3))
    pos[2 * coincident:2 * coincident + 40:2] = pos[2 * coincident + 1:2 * coincident + 41:2]
    return rng.permutation(pos).astype(np.float32)


def _check(gpu, oracle_mod, cfg, corr, pos, steps):
    lo, hi = (0.0, 0.0, 0.0), (4.0, 4.0, 4.0)
    vel = np.random.default_rng(len(pos)).uniform(-0.5, 0.5, pos.shape).astype(np.float32)
    s = gpu(len(pos), cfg, corr)
    o = oracle_mod.Oracle(len(pos), cfg, corr, 32)
    s.set_state(pos, vel)
    o.set_state(pos, vel)
    full = 0  # the most full lists after a step
    for k in range(steps):
        s.step(DT, lo, hi)
        o.step(DT, lo, hi)
        t = o.taps()
        np.testing.assert_array_equal(s.debug_hashes(), t["sorted_hash"])
        np.testing.assert_array_equal(s.debug_permutation(), t["perm"])
        assert np.array_equal(np.sort(s.debug_physical_order()), np.arange(len(pos)))
        nbr, cnt = s.debug_neighbours()
        np.testing.assert_array_equal(cnt, t["cnt"])
        np.testing.assert_array_equal(nbr, t["nbr"])
        full = max(full, int((cnt == cfg.maxNeighbours).sum()))
    g, r = s.get_state(), o.state()
    for k in ("pos", "vel", "density", "lam", "ids"):
        np.testing.assert_array_equal(g[k], r[k].astype(g[k].dtype), err_msg=k)
    return full


@pytest.mark.parametrize("n,coincident", [(12000, 4000), (40000, 5000), (160001, 7001)])
@pytest.mark.parametrize("cap", [3, 64, 128, 321])
def test_lists_at_the_cap(gpu, oracle_mod, dam_params, n, coincident, cap):
    """Runs whose lists are all full long before their candidates end (streams of several windows),
    beside runs that take all of theirs."""
    cfg, corr = dam_params
    print(f"[crowded] n={n}, coincident={coincident}, cap={cap}", flush=True)
    full = _check(gpu, oracle_mod, dataclasses.replace(cfg, maxNeighbours=cap), corr, _crowd(n, coincident, cap), 2)
    assert full >= coincident  # the crowd disperses after the first step
