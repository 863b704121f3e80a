"""Masses of device records: scenes large enough that the kernels look at them, stepped with unit
masses, with one that is not, and with unit masses again, each step against the FP32 oracle started
from the buffer before it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
DT = 0.004


@pytest.mark.parametrize("n", [32769, 40000, 131073, 262145])
def test_masses_change_between_steps(oracle_mod, dam_params, n):
    import torch
    if torch.cuda.device_count() < 1:
        pytest.fail("no GPU visible: the gpu tests need an MI355X")
    from akuaengine_amd import scenes
    from akuaengine_amd.solver import PBFSolver
    cfg, corr = dam_params
    sc = scenes.batched_scene(n, index=n % 5)
    buf = np.zeros((n, 27), np.float32)
    buf[:, 0:3] = sc.pos
    buf[:, 18] = 1.0
    buf[:, 25] = np.arange(n)
    s = PBFSolver(n, cfg, corr)
    dev = torch.from_numpy(buf).cuda()
    for step, where in enumerate((None, n - 1, None, 256 * (n // 512))):
        print(f"[record masses] n={n}, step {step}", flush=True)
        if where is not None:
            dev[where, 18] = 0.75
        else:
            dev[:, 18] = 1.0
        before = dev.cpu().numpy()
        o = oracle_mod.Oracle(n, cfg, corr, 32)
        o.set_state(before[:, 0:3], before[:, 3:6], before[:, 18])
        o.step(DT, sc.box_min, sc.box_max)
        s.step_device(dev.data_ptr(), DT, sc.box_min, sc.box_max, torch.cuda.current_stream().cuda_stream)
        g, st, sa, t = dev.cpu().numpy(), o.state(), o.stage_arrays(), o.taps()
        want = (("pos", 0, st["pos"]), ("vel", 3, st["vel"]), ("new_pos", 6, st["pos"]), ("new_vel", 9, sa["vs"]),
                ("dp", 12, sa["dp"]), ("vort", 15, sa["vort"]), ("mass", 18, st["mass"]),
                ("density", 19, st["density"]), ("lambda", 20, st["lam"]))
        for name, at, w in want:
            w = np.asarray(w, np.float32).reshape(n, -1)
            np.testing.assert_array_equal(g[:, at:at + w.shape[1]], w, err_msg=f"{name}, step {step}")
        np.testing.assert_array_equal(g.view(np.uint32)[:, 21], t["sorted_hash"])
        np.testing.assert_array_equal(g[:, 25], before[st["ids"].astype(np.int64), 25])
