"""akua_mlp_adam_step_device on arrays that begin at any float (the features, read four at a time since ever,
excepted): the results of the same call on arrays that begin at 256 bytes."""
import ctypes

import numpy as np
import pytest

from oracle import mlp_oracle as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("off", [1, 2, 3])
def test_arrays_at_any_float(off):
    import torch
    if torch.cuda.device_count() < 1:
        pytest.fail("no GPU visible: the gpu tests need an MI355X")
    from akuaengine_amd import _lib
    L = _lib.load()
    rng = np.random.default_rng(off)
    n = 1000
    F = (rng.normal(size=(n, 16)) * rng.uniform(0.1, 5, 16)).astype(np.float32)
    T = (rng.normal(size=(n, 4)) * np.array([0.3, 1.0, 0.1, 2.0])).astype(np.float32)
    p = M.random_params(rng, F, T).astype(np.float32)
    w = np.array([1.0, 0.5, 2.0, 0.25], np.float32)
    dF = torch.from_numpy(F).cuda()

    def call(at):
        def put(a):
            d = torch.zeros(a.size + 8, dtype=torch.float32, device="cuda")
            d[at:at + a.size] = torch.from_numpy(a.ravel()).cuda()
            return d, ctypes.c_void_p(d.data_ptr() + 4 * at)
        arrays = [put(a) for a in (p, np.zeros(M.TRAINABLE, np.float32), np.zeros(M.TRAINABLE, np.float32), T,
                                   np.zeros(1, np.float32))]
        P, m, v, targets, loss = (q for _, q in arrays)
        assert L.akua_mlp_adam_step_device(P, m, v, 1, 1e-3, ctypes.c_void_p(dF.data_ptr()), targets, n,
                                           w.ctypes.data_as(ctypes.c_void_p), loss, None) == 0, L.akua_last_error()
        torch.cuda.synchronize()
        return [d[at:at + k].cpu().numpy() for (d, _), k in
                zip(arrays, (p.size, M.TRAINABLE, M.TRAINABLE, T.size, 1))]

    for got, want in zip(call(off), call(0)):
        np.testing.assert_array_equal(got, want)
