"""The list build's edges, list by list against the FP32 oracle: runs of particles in one cell that
are shorter and longer than the rows a wave keeps, waves of 8 to 64 slots that end inside a cell or a
scene, candidate streams longer than one bitmap window, caps around the row sizes of each form, buckets
that several cells share."""
import dataclasses

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
DT = 0.0083


@pytest.fixture(scope="module")
def gpu():
    import torch
    if torch.cuda.device_count() < 1:
        pytest.fail("no GPU visible: the gpu tests need an MI355X")
    from akuaengine_amd.solver import PBFSolver
    return PBFSolver


def _check(gpu, oracle_mod, cfg, corr, pos, lo, hi):
    vel = np.zeros_like(pos)
    s = gpu(len(pos), cfg, corr)
    o = oracle_mod.Oracle(len(pos), cfg, corr)
    s.set_state(pos, vel)
    o.set_state(pos, vel)
    s.step(DT, lo, hi)
    o.step(DT, lo, hi)
    nbr, cnt = s.debug_neighbours()
    t = o.taps()
    np.testing.assert_array_equal(cnt, t["cnt"])
    np.testing.assert_array_equal(nbr, t["nbr"])
    return cnt


# wave sizes change at 2^13 (below), 2^17 and 2^19 slots
@pytest.mark.parametrize("n", [1, 2, 7, 8, 9, 63, 65, 257, 4099, 65535, 65537, 131071, 131073, 524287, 524289])
def test_counts_around_the_wave_sizes(gpu, oracle_mod, dam_params, n):
    from akuaengine_amd import scenes
    cfg, corr = dam_params
    sc = scenes.batched_scene(n, index=n % 7)
    print(f"[list build] n={n}", flush=True)
    _check(gpu, oracle_mod, cfg, corr, sc.pos, sc.box_min, sc.box_max)


@pytest.mark.parametrize("cap", [1, 3, 4, 31, 33, 63, 64, 65, 128, 319, 320, 321, 900, 1792, 1793])
def test_caps_in_crowded_cells(gpu, oracle_mod, dam_params, cap):
    """2,400 particles in one cell and its neighbours beside a sparse spray: streams past 2,048
    candidates, lists at the cap, runs of one particle."""
    cfg, corr = dam_params
    cfg = dataclasses.replace(cfg, maxNeighbours=cap)
    rng = np.random.default_rng(cap)
    pos = np.concatenate([1.0 + rng.uniform(0.0, 0.099, (1500, 3)), 1.0 + rng.uniform(-0.1, 0.2, (900, 3)),
                          rng.uniform(0.1, 3.9, (700, 3))]).astype(np.float32)
    print(f"[list build] cap={cap}", flush=True)
    cnt = _check(gpu, oracle_mod, cfg, corr, pos, (0.0, 0.0, 0.0), (4.0, 4.0, 4.0))
    assert (cnt == 0).any()
    if cap <= 900:  # no particle has more than about 1,700 neighbours here
        assert (cnt == cap).any()


def test_shared_buckets_and_search_cells(gpu, oracle_mod, dam_params):
    """A hash table of one entry per particle (cells share buckets, whose particles then lie apart in
    memory and are listed twice) and a search cell size that is not the hash's."""
    cfg, corr = dam_params
    rng = np.random.default_rng(5)
    pos = rng.uniform(0.1, 1.9, (5003, 3)).astype(np.float32)
    for over in (dict(maxNeighbours=1), dict(maxNeighbours=2), dict(spatialHashCellSize=0.13),
                 dict(spatialHashCellSize=0.07, maxNeighbours=40)):
        _check(gpu, oracle_mod, dataclasses.replace(cfg, **over), corr, pos, (0.0, 0.0, 0.0), (2.0, 2.0, 2.0))


@pytest.mark.parametrize("n", [8191, 8192, 8193])
def test_counts_around_the_smallest_waves(gpu, oracle_mod, dam_params, n):
    """Waves of four slots below 2^13, of eight from there on."""
    from akuaengine_amd import scenes
    cfg, corr = dam_params
    sc = scenes.batched_scene(n, index=n % 7)
    print(f"[list build] n={n}", flush=True)
    _check(gpu, oracle_mod, cfg, corr, sc.pos, sc.box_min, sc.box_max)
