"""Record steps of one solver on several streams, each with a record buffer of its own: nothing but the
solver orders what the steps share.  Two host threads on hipStreamPerThread (one handle, two streams), two
streams and the null stream in turn, a stream created on the handle of a destroyed one, and steps on the
solver's own stream between them, all without host synchronisation and equal to the FP32 oracle's."""
import ctypes
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
DT = 0.004
PER_THREAD = 2  # hipStreamPerThread


def _records(pos):
    import torch
    buf = np.zeros((len(pos), 27), np.float32)
    buf[:, 0:3] = pos
    buf[:, 18] = 1.0
    return torch.from_numpy(buf).cuda()


def _setup(oracle_mod, cfg, corr, n, buffers):
    """A solver, and for each buffer a scene, its records and its oracle."""
    import torch
    if torch.cuda.device_count() < 1:
        pytest.fail("no GPU visible: the gpu tests need an MI355X")
    from akuaengine_amd import scenes
    from akuaengine_amd.solver import PBFSolver
    s = PBFSolver(n, cfg, corr)
    sets = []
    for k in range(buffers):
        sc = scenes.batched_scene(n, index=k + 1)
        o = oracle_mod.Oracle(n, cfg, corr, 32)
        o.set_state(sc.pos, np.zeros_like(sc.pos))
        sets.append((sc, _records(sc.pos), o))
    torch.cuda.synchronize()
    return s, sets


def _equal(dev, o):
    out, w = dev.cpu().numpy(), o.state()
    np.testing.assert_array_equal(out[:, 0:3], w["pos"].astype(np.float32))
    np.testing.assert_array_equal(out[:, 3:6], w["vel"].astype(np.float32))


@pytest.mark.parametrize("n", [1000, 140000])
def test_two_threads_on_their_own_streams(oracle_mod, dam_params, n):
    import torch
    cfg, corr = dam_params
    s, sets = _setup(oracle_mod, cfg, corr, n, 2)
    steps = 4
    turn = [threading.Semaphore(1), threading.Semaphore(0)]
    finished = threading.Barrier(3)
    errors = []

    def work(k):
        sc, dev, _ = sets[k]
        try:
            for step in range(steps):
                turn[k].acquire()  # the host calls are serialised, the device's work is not
                print(f"[record order] n={n}, thread {k}, step {step}", flush=True)
                s.step_device(dev.data_ptr(), DT, sc.box_min, sc.box_max, stream=PER_THREAD)
                turn[1 - k].release()
        except Exception as e:  # noqa: BLE001 - reported by the test's thread
            errors.append(e)
            turn[1 - k].release()
        finished.wait(60)  # both threads, and so their streams, live until the device is done
        finished.wait(60)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(2)]
    for t in threads:
        t.start()
    finished.wait(60)
    torch.cuda.synchronize()
    finished.wait(60)
    for t in threads:
        t.join()
    assert not errors, errors
    for sc, dev, o in sets:
        o.step(DT, sc.box_min, sc.box_max, steps)
        _equal(dev, o)


@pytest.mark.parametrize("n", [1000, 140000])
def test_streams_and_buffers_in_turn(oracle_mod, dam_params, n):
    import torch
    from akuaengine_amd import _lib
    cfg, corr = dam_params
    s, sets = _setup(oracle_mod, cfg, corr, n, 3)
    hip = _lib.load()  # the HIP runtime's symbols, through the library that is linked to it
    stream_of = [torch.cuda.Stream(), torch.cuda.Stream(), None]
    busy = [torch.ones(1 << 24, device="cuda") for _ in sets]
    torch.cuda.synchronize()

    def step(k, handle=None):
        sc, dev, o = sets[k]
        st = stream_of[k]
        if handle is None:
            with torch.cuda.stream(st if st is not None else torch.cuda.default_stream()):
                busy[k].mul_(1.0000001)  # queued work ahead of the step
            handle = 0 if st is None else st.cuda_stream
        s.step_device(dev.data_ptr(), DT, sc.box_min, sc.box_max, stream=handle)
        o.step(DT, sc.box_min, sc.box_max)

    # buffers in turn, each on its stream only
    for k in (0, 1, 0, 2, 1, 2, 0):
        print(f"[record order] n={n}, buffer {k}", flush=True)
        step(k)
    # on from the last records on the solver's own stream, at once behind the caller's
    sc, dev, o = sets[0]
    s.step_n(DT, sc.box_min, sc.box_max, 2)
    own = oracle_mod.Oracle(n, cfg, corr, 32)
    own.set_state(o.state()["pos"], o.state()["vel"])
    own.step(DT, sc.box_min, sc.box_max, 2)
    # records again, at once behind the solver's own steps; the state is then the records'
    step(1)
    np.testing.assert_array_equal(s.get_state()["pos"], sets[1][2].state()["pos"].astype(np.float32))
    # and the solver's own steps once more, read back
    step(0)
    s.step_n(DT, sc.box_min, sc.box_max, 1)
    own.set_state(o.state()["pos"], o.state()["vel"])
    own.step(DT, sc.box_min, sc.box_max, 1)
    np.testing.assert_array_equal(s.get_state()["pos"], own.state()["pos"].astype(np.float32))

    # streams that are created and destroyed between the steps: a handle may come again
    for k in (2, 1, 2):
        h = ctypes.c_void_p()
        assert hip.hipStreamCreate(ctypes.byref(h)) == 0
        print(f"[record order] n={n}, buffer {k}, a new stream", flush=True)
        torch.cuda.synchronize()  # buffer k's earlier work is on another stream
        step(k, handle=h.value)
        step(1 - (k == 1), handle=h.value)  # and another buffer behind it
        assert hip.hipStreamDestroy(h) == 0
    torch.cuda.synchronize()
    for _, dev, o in sets:
        _equal(dev, o)
