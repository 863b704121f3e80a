"""Reading back from several solvers, whose copies share one pinned ring: first and later calls on both sides
of the size up to which a first call does without it, several threads at once on solvers of their own, solvers
that go while others read, and states and images in turn."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    import torch
    if torch.cuda.device_count() < 1:
        pytest.fail("no GPU visible: the gpu tests need an MI355X")
    from akuaengine_amd import solver
    return solver


def _given(n, seed):
    rng = np.random.default_rng(seed)
    return tuple(rng.uniform(0.5, 39.5, k).astype(np.float32) for k in ((n, 3), (n, 3), n, n, n))


def _equal(s, given):
    out = s.get_state()
    for name, a in zip(("pos", "vel", "mass", "density", "lam"), given):
        np.testing.assert_array_equal(out[name], a)
    np.testing.assert_array_equal(out["ids"], np.arange(len(given[2]), dtype=np.uint32))


# 40 B per particle, 4 MB at 104,857 particles
@pytest.mark.parametrize("n", [5, 27000, 104857, 104858, 500000])
def test_first_and_later_calls_of_new_solvers(gpu, dam_params, n):
    image = None
    for k in range(3):
        s = gpu.PBFSolver(n, *dam_params)
        given = _given(n, 1)
        s.set_state(*given)
        print(f"[shared readback] n={n}, solver {k}", flush=True)
        if k == 1:  # an image first
            image = s.render(width=640, height=360)
        for _ in range(3):
            _equal(s, given)
        again = s.render(width=640, height=360)
        assert image is None or np.array_equal(image, again)
        image = again
        del s


def test_threads_on_solvers_of_their_own(gpu, dam_params):
    sizes = [3000, 60000, 150000, 400000]
    start, errors = threading.Barrier(len(sizes)), []

    def work(n, seed):
        try:
            start.wait(60)
            for k in range(4):
                s = gpu.PBFSolver(n, *dam_params)
                given = _given(n, seed + k)
                s.set_state(*given)
                for _ in range(3):
                    _equal(s, given)
                del s
        except BaseException as e:  # noqa: BLE001 - reported by the test's thread
            errors.append((n, e))

    threads = [threading.Thread(target=work, args=(n, 10 * i)) for i, n in enumerate(sizes)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(100)
    assert not errors, errors
    assert not any(t.is_alive() for t in threads)
