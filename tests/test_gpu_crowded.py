"""Crowded scenes against the FP32 oracle, order by order and list by list: some thousands of coincident
particles, a crowded cell and its neighbours beside ordinary ones, in single scenes of both orderings, with
caps from a few entries to more than a cell holds; groups of hashes around the size from which they are
sorted, whose particles share a cell, a bucket or the group only, inside the box and far out; records whose
positions are not finite."""
import dataclasses
import math

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


def _cells(oracle_mod, table, shift, far, want):
    """Up to three cells of one hash (want "bucket") or of hashes that differ within one group ("group"), among
    those of the box or, far, 400 cells off."""
    by = {}
    for c in ((far + i, j, k) for i in range(1, 39) for j in range(1, 39) for k in range(1, 39)):
        h = oracle_mod.cell_hash(*c, table)
        like = by.setdefault(h if want == "bucket" else h >> shift, {})
        like.setdefault(len(like) if want == "bucket" else h, c)
        if len(like) == 3:
            return list(like.values())
    return list(max(by.values(), key=len).values())


@pytest.mark.parametrize("n", [9001, 33003, 140001])
@pytest.mark.parametrize("crowd", [511, 512, 513, 1024, 1025, 3333])
@pytest.mark.parametrize("want,far", [("cell", 0), ("bucket", 0), ("group", 0), ("group", 400)])
def test_crowded_groups(gpu, oracle_mod, dam_params, n, crowd, want, far):
    """One crowd, in one cell or shuffled over up to three that share a bucket or only the group; far: out of
    the box, beyond the cells that have bins."""
    cfg, corr = dam_params
    cap = 1 if want == "bucket" else 16  # the table has cap entries per particle: few make buckets be shared
    cfg = dataclasses.replace(cfg, maxNeighbours=cap)
    lg = max(8 if n <= 32768 else 6, math.ceil(math.log2((n + 3) // 4)))
    shift = max(0, math.ceil(math.log2(n * cap)) - lg)
    cells = _cells(oracle_mod, n * cap, shift, far, want) if want != "cell" else [(3, 5, 2)]
    rng = np.random.default_rng(crowd + n)
    pos = rng.uniform(0.05, 3.95, (n, 3))
    at = np.array([cells[k % len(cells)] for k in range(crowd)], np.float64)
    pos[:crowd] = (at + rng.uniform(0.2, 0.8, (crowd, 3))) * cfg.spatialHashCellSize
    print(f"[crowded] n={n}, crowd={crowd}, {want}, far={far}, {len(cells)} cells", flush=True)
    _check(gpu, oracle_mod, cfg, corr, rng.permutation(pos).astype(np.float32), 2)


@pytest.mark.parametrize("n", [9001, 40003])
def test_crowd_in_a_step_without_iterations(gpu, oracle_mod, dam_params, n):
    """Density, lambda and the position delta are carried along."""
    cfg, corr = dam_params
    _check(gpu, oracle_mod, dataclasses.replace(cfg, solverIterations=0), corr, _crowd(n, 2500, 1), 2)


@pytest.mark.parametrize("n", [9001, 40003])
@pytest.mark.parametrize("value", [float("nan"), float("inf")])
def test_records_that_are_not_finite(gpu, oracle_mod, dam_params, n, value):
    """2,000 records without a finite position: one cell, and no neighbours of the others, which step as
    beside particles far away.  Records are told apart by their colour."""
    import torch
    cfg, corr = dam_params
    lo, hi, lost = (0.0, 0.0, 0.0), (4.0, 4.0, 4.0), 2000
    rng = np.random.default_rng(n)
    pos = rng.uniform(0.1, 3.9, (n, 3)).astype(np.float32)
    pos[rng.permutation(n)[:lost]] = value
    ok = np.isfinite(pos).all(axis=1)
    buf = np.zeros((n, 27), np.float32)
    buf[:, 0:3], buf[:, 18], buf[:, 22] = pos, 1.0, np.arange(n)
    dev = torch.from_numpy(buf).cuda()
    print(f"[crowded] n={n}, {value}", flush=True)
    gpu(n, cfg, corr).step_device(dev.data_ptr(), DT, lo, hi)
    torch.cuda.synchronize()
    out = dev.cpu().numpy()
    assert np.array_equal(np.sort(out[:, 22]), np.arange(n))
    out = out[np.argsort(out[:, 22])]
    far = pos.copy()
    far[~ok] = 1000.0
    o = oracle_mod.Oracle(n, cfg, corr, 32)
    o.set_state(far, np.zeros_like(far))
    o.step(DT, lo, hi)
    w = o.state()
    back = np.argsort(w["ids"])
    np.testing.assert_array_equal(out[ok, 0:3], w["pos"][back][ok].astype(np.float32))
    np.testing.assert_array_equal(out[ok, 3:6], w["vel"][back][ok].astype(np.float32))
