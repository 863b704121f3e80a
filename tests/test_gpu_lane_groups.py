"""Lane groups in the neighbour sweeps (several lanes per particle, sums in list order), bit for bit
against the FP32 oracle: lists that end inside, at and past a group's round, uneven masses, wall
samples whose windows take several rounds, and the sizes at which the default changes its group."""
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


def _check(gpu, oracle_mod, cfg, corr, pos, mass, lo, hi, layers, lanes, steps):
    s = gpu(len(pos), cfg, corr)
    o = oracle_mod.Oracle(len(pos), cfg, corr, 32)
    for x in (s, o):
        x.set_state(pos, np.zeros_like(pos), mass)
        if layers:
            x.set_boundary(layers, 0.0)
    if lanes:
        s.set_tuning(laneGroup=lanes)
    longest = 0
    for _ in range(steps):
        s.step(DT, lo, hi)
        o.step(DT, lo, hi)
        longest = max(longest, int(s.debug_neighbours()[1].max()))
    g, r = s.get_state(), o.state()
    for k in ("pos", "vel", "density", "lam", "ids"):
        np.testing.assert_array_equal(g[k], r[k].astype(g[k].dtype), err_msg=k)
    return longest


@pytest.mark.parametrize("layers", [0, 1, 3])
@pytest.mark.parametrize("cap", [3, 8, 9, 31, 32, 33, 64, 65, 90])
@pytest.mark.parametrize("lanes", [2, 4, 8, 16])
def test_list_lengths(gpu, oracle_mod, dam_params, lanes, cap, layers):
    from akuaengine_amd import scenes
    cfg, corr = dam_params
    cfg = dataclasses.replace(cfg, maxNeighbours=cap)
    rng = np.random.default_rng(cap)
    pos = scenes.lattice(11, 9, 7, 0.035, (0.02, 0.02, 0.02))  # about 95 neighbours inside
    pos = (pos + rng.uniform(-0.004, 0.004, pos.shape)).astype(np.float32)
    mass = rng.uniform(0.5, 1.5, len(pos)).astype(np.float32) if cap % 2 else None
    print(f"[lane groups] {lanes} lanes, cap {cap}, {layers} layers", flush=True)
    longest = _check(gpu, oracle_mod, cfg, corr, pos, mass, (0.0, 0.0, 0.0), (0.7, 0.5, 0.27), layers, lanes, 2)
    assert longest == cap  # in the first step; later ones spread


@pytest.mark.parametrize("n", [1, 2, 31, 32767, 32769, 262145])
def test_default_group_by_size(gpu, oracle_mod, dam_params, n):
    from akuaengine_amd import scenes
    cfg, corr = dam_params
    sc = scenes.batched_scene(n, index=n % 5)
    print(f"[lane groups] n={n}", flush=True)
    _check(gpu, oracle_mod, cfg, corr, sc.pos, None, sc.box_min, sc.box_max, 0, 0, 2)


@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("cap", [30, 64, 91])
def test_uneven_lists_in_large_scenes(gpu, oracle_mod, dam_params, cap, mixed):
    """Above 262,144 particles a wave shares its long lists: dense blobs (about 95 neighbours) between
    sparse particles in the same waves, lists of 0 to the cap, a last wave that is not full."""
    from akuaengine_amd import scenes
    cfg, corr = dam_params
    cfg = dataclasses.replace(cfg, maxNeighbours=cap)
    rng = np.random.default_rng(cap)
    blob = scenes.lattice(7, 7, 7, 0.035, (0.0, 0.0, 0.0))
    at = rng.uniform(0.5, 7.5, (300, 1, 3))
    pos = np.concatenate([(blob[None] + at).reshape(-1, 3), rng.uniform(0.05, 7.95, (160001, 3))])
    pos = (pos + rng.uniform(-0.004, 0.004, pos.shape)).astype(np.float32)
    assert len(pos) > 1 << 18 and len(pos) % 64
    mass = rng.uniform(0.5, 1.5, len(pos)).astype(np.float32) if mixed else None
    print(f"[lane groups] uneven lists, cap {cap}, masses {mixed}", flush=True)
    longest = _check(gpu, oracle_mod, cfg, corr, pos, mass, (0.0, 0.0, 0.0), (8.0, 8.0, 8.0), 0, 0, 2)
    assert longest == cap
