"""Tuning cache files written for other kernels: their lines are kept but not applied."""
import re

import pytest

pytestmark = pytest.mark.gpu
DT = 0.0083


def test_lines_of_other_kernels_are_not_applied(dam_params, tmp_path):
    import torch
    if torch.cuda.device_count() < 1:
        pytest.fail("no GPU visible: the gpu tests need an MI355X")
    from akuaengine_amd import scenes
    from akuaengine_amd.solver import PBFSolver
    sc = scenes.dam_break_scaled(10, seed=1)

    def tune(cache):
        s = PBFSolver(sc.n, *dam_params)
        s.set_state(sc.pos, sc.vel, sc.mass)
        return s.autotune(DT, sc.box_min, sc.box_max, trialSteps=1, cachePath=str(cache))

    fresh = tmp_path / "fresh.txt"
    tune(fresh)
    key, _ = fresh.read_text().split(" | ")
    assert re.search(r" kernels\d+", key)
    old = tmp_path / "old.txt"
    stale = "512 3 8 8 8 2048 8 1 1 2 2"  # a setting that no trial prefers
    for line in (re.sub(r" kernels\d+", "", key), re.sub(r" kernels\d+", " kernels1", key)):
        old.write_text(f"{line} | {stale}\n")
        print(f"[tuning cache] {line}", flush=True)
        tune(old)
        lines = old.read_text().splitlines()
        assert lines[0] == f"{line} | {stale}" and len(lines) == 2 and lines[1].startswith(f"{key} | ")
