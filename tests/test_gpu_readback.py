"""Reading the particles back: sizes on both sides of each of the copy's limits (one pinned chunk, the
calling thread alone, the ring of chunks), scenes with padding between their slots, absent arrays, a
solver without particles, and the arrays against the records of the same step."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
LO, HI = (0.0, 0.0, 0.0), (40.0, 40.0, 40.0)


@pytest.fixture(scope="module")
def gpu():
    import torch
    if torch.cuda.device_count() < 1:
        pytest.fail("no GPU visible: the gpu tests need an MI355X")
    from akuaengine_amd import solver
    return solver


def _state(n, seed):
    rng = np.random.default_rng(seed)
    f = lambda *s: rng.uniform(0.5, 39.5, s).astype(np.float32)  # noqa: E731
    return f(n, 3), f(n, 3), f(n), f(n), f(n)


# 40 B per particle: 64 KB, 1 MB and 4 MB lie at 1,638, 26,214 and 104,857 particles, the ring at 419,430
@pytest.mark.parametrize("n", [1, 1638, 1639, 26214, 26215, 104857, 104858, 419431, 1000003])
def test_state_returns_what_was_set(gpu, dam_params, n):
    print(f"[readback] n={n}", flush=True)
    s = gpu.PBFSolver(n, *dam_params)
    given = _state(n, n)
    for _ in range(2):  # the second call reuses the chunks
        s.set_state(*given)
        out = s.get_state()
        for name, a in zip(("pos", "vel", "mass", "density", "lam"), given):
            np.testing.assert_array_equal(out[name], a)
        np.testing.assert_array_equal(out["ids"], np.arange(n, dtype=np.uint32))
        given = _state(n, n + 1)


@pytest.mark.parametrize("n", [333, 70001, 450001])
def test_state_equals_the_records_of_a_step(gpu, dam_params, n):
    from akuaengine_amd import _lib
    s = gpu.PBFSolver(n, *dam_params)
    pos, vel, mass, dens, lam = _state(n, 7)
    s.set_state(pos, 0.01 * vel, mass)
    s.step(0.001, LO, HI)
    out = s.get_state()
    rec = np.frombuffer(s.get_particles(), np.float32).reshape(n, 27)
    for name, a in (("pos", rec[:, 0:3]), ("vel", rec[:, 3:6]), ("mass", rec[:, 18]), ("density", rec[:, 19]),
                    ("lam", rec[:, 20])):
        np.testing.assert_array_equal(out[name], a)
    np.testing.assert_array_equal(out["mass"], mass[out["ids"]])
    only = np.zeros(n, np.uint32)  # one array alone
    p = only.ctypes.data_as(ctypes.c_void_p)
    _lib.check(s._L.akua_solver_get_state(s._h, None, None, None, None, None, p, n))
    np.testing.assert_array_equal(only, out["ids"])


def test_scenes_without_their_padding(gpu, dam_params):
    counts = [1, 255, 256, 257, 1000, 40000, 3]
    b = gpu.BatchSolver(counts, *dam_params)
    given = _state(sum(counts), 3)
    b.set_state(*given)
    out = b.get_state()
    for name, a in zip(("pos", "vel", "mass", "density", "lam"), given):
        np.testing.assert_array_equal(out[name], a)
    for i in range(len(counts)):
        b.set_box(i, LO, HI)
    b.step_batch(0.001, 1)
    out = b.get_state()
    at = np.cumsum([0] + counts)
    for a, e in zip(at[:-1], at[1:]):
        np.testing.assert_array_equal(np.sort(out["ids"][a:e]), np.arange(a, e, dtype=np.uint32))
    np.testing.assert_array_equal(out["mass"], given[2][out["ids"]])


def test_a_solver_without_particles_is_zero(gpu, dam_params):
    for s in (gpu.PBFSolver(500, *dam_params), gpu.BatchSolver([5, 300], *dam_params)):
        assert all(not a.any() for a in s.get_state().values())
