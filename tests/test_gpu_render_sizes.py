"""The same sprites, of one pixel to a third of the image, in scenes of as many particles as wanted (the
others behind the camera): each number of particles that a wave projects draws the image that the numpy
restatement draws, whichever lanes draw a sprite."""
import ctypes

import numpy as np
import pytest

from test_gpu_render import _reference_render

pytestmark = pytest.mark.gpu


def _scene(n, rng):
    """n particles, the visible ones among them (in draw order), colours and sizes."""
    vis = np.sort(rng.permutation(n)[:min(n, 260)])
    pos = np.tile(np.array([3.0, 2.0, 30.0], np.float32), (n, 1))  # behind the camera
    pos[vis] = np.stack([rng.uniform(0.5, 5.5, len(vis)), rng.uniform(0.0, 4.0, len(vis)),
                         rng.uniform(-4.0, 4.5, len(vis))], 1)
    twin = len(vis) // 4 * 2
    pos[vis[1:twin:2]] = pos[vis[0:twin:2]]  # pairs at one point: draw order decides
    col = np.ones((n, 4), np.float32)
    col[:, :3] = rng.uniform(0, 1, (n, 3))
    size = np.exp(rng.uniform(np.log(2.0), np.log(300.0), n)).astype(np.float32)
    size[vis[1:twin:2]] = size[vis[0:twin:2]]
    return vis, pos, col, size


@pytest.mark.parametrize("n", [1, 3, 4, 5, 255, 32767, 32768, 32769, 32785, 131071, 131072, 131073, 131137,
                               (1 << 21) - 1, (1 << 21) + 1])
def test_image_does_not_depend_on_the_number_of_particles(n):
    import torch
    if torch.cuda.device_count() < 1:
        pytest.fail("no GPU visible: the gpu tests need an MI355X")
    from akuaengine_amd import _lib, solver as S
    from akuaengine_amd.config import LambdaCorrParams, PBFConfig
    vis, pos, col, size = _scene(n, np.random.default_rng(n))
    buf = np.zeros((n, 27), np.float32)
    buf[:, 0:3], buf[:, 18], buf[:, 22:26], buf[:, 26] = pos, 1.0, col, size
    recs = (_lib.AkuaParticle * n)()
    ctypes.memmove(recs, buf.ctypes.data, buf.nbytes)
    s = S.PBFSolver(n, PBFConfig(maxNeighbours=8), LambdaCorrParams())
    s.set_particles(recs)
    W, H = 150, 85
    cam = S.default_camera()
    print(f"[render sizes] n={n}", flush=True)
    img = s.render(cam, W, H, point_size=0.0)
    ref = _reference_render(S, cam, pos[vis], col[vis], size[vis], W, H)
    diff = np.abs(img.astype(int) - ref.astype(int))
    assert diff.max() <= 1  # exp, as in the restatement's own tests
    assert (diff.max(axis=2) == 0).mean() >= 0.99
