"""Record steps run on the caller's stream: steps on two streams and on the null stream, with steps,
uploads and reads on the solver's own stream between them and no host synchronisation, equal the FP32
oracle's; a changed box, a failed step and a destroyed stream on the way."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
DT = 0.004


@pytest.mark.parametrize("n", [1000, 140000])
def test_streams_in_turn(oracle_mod, dam_params, n):
    import torch
    if torch.cuda.device_count() < 1:
        pytest.fail("no GPU visible: the gpu tests need an MI355X")
    from akuaengine_amd import scenes
    from akuaengine_amd.solver import PBFSolver
    cfg, corr = dam_params
    sc = scenes.batched_scene(n, index=1)
    lo, hi = sc.box_min, sc.box_max
    buf = np.zeros((n, 27), np.float32)
    buf[:, 0:3] = sc.pos
    buf[:, 18] = 1.0
    s = PBFSolver(n, cfg, corr)
    o = oracle_mod.Oracle(n, cfg, corr, 32)
    o.set_state(sc.pos, np.zeros_like(sc.pos))
    s.set_state(sc.pos, np.zeros_like(sc.pos))
    s.step_n(DT, lo, hi, 2)  # the solver's own stream first: its state is then replaced by the records
    dev = torch.from_numpy(buf).cuda()
    torch.cuda.synchronize()
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    busy = torch.ones(1 << 24, device="cuda")
    torch.cuda.synchronize()
    last = None
    for step, stream in enumerate((a, a, None, b, "own", a, b, None)):
        print(f"[record streams] n={n}, step {step}", flush=True)
        if step == 3:
            hi = tuple(h * 1.25 for h in hi)
        o.step(DT, lo, hi)
        if stream == "own":  # steps on from the state that the last record step left
            s.step_n(DT, lo, hi, 1)
            got = s.get_state()
            for k, w in (("pos", o.state()["pos"]), ("vel", o.state()["vel"])):
                np.testing.assert_array_equal(got[k], w.astype(np.float32), err_msg=f"{k}, step {step}")
            buf = np.zeros((n, 27), np.float32)
            buf[:, 0:3], buf[:, 3:6], buf[:, 18] = got["pos"], got["vel"], 1.0
            dev = torch.from_numpy(buf).cuda()
            torch.cuda.synchronize()
            o = oracle_mod.Oracle(n, cfg, corr, 32)
            o.set_state(got["pos"], got["vel"])
            last = None
            continue
        st = stream if stream is not None else torch.cuda.default_stream()
        with torch.cuda.stream(st):
            if last is not None and last is not st:
                st.wait_stream(last)  # the caller orders its own buffer
            busy.mul_(1.0000001)      # queued work ahead of the step
            s.step_device(dev.data_ptr(), DT, lo, hi, stream=0 if stream is None else st.cuda_stream)
        last = st
    with pytest.raises(Exception):
        s.step_device(dev.data_ptr(), float("nan"), lo, hi, stream=0)
    with torch.cuda.stream(last):
        out = dev.to("cpu")
    torch.cuda.synchronize()
    w = o.state()
    np.testing.assert_array_equal(out[:, 0:3].numpy(), w["pos"].astype(np.float32))
    np.testing.assert_array_equal(out[:, 3:6].numpy(), w["vel"].astype(np.float32))
    t = torch.cuda.Stream()
    s.step_device(dev.data_ptr(), DT, lo, hi, stream=t.cuda_stream)
    o.step(DT, lo, hi)
    del t  # the state is still the step's
    np.testing.assert_array_equal(s.get_state()["pos"], o.state()["pos"].astype(np.float32))
