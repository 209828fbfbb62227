"""Grid Verlet on both sides of the grid size at which its kernel changes form
(1024 tiles of 32x8 on 256 CUs), bit for bit against the FP32 oracle."""
import numpy as np
import pytest

from opencloth_amd import scenes
from tests.helpers import say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w,h", [(1024, 256), (1025, 256), (700, 400), (33, 8001)])
@pytest.mark.parametrize("vbo", [False, True])
def test_bitwise(w, h, vbo):
    from opencloth_amd.cloth import VerletGrid
    from opencloth_amd.hiptime import DeviceBuffer, device_synchronize
    from oracle import Oracle

    say("vgrid", w, h, vbo)
    rng = np.random.default_rng(w + h)
    p = scenes.vgrid_params(w, h)
    sx, sy = p["spacing"]
    ix, iy = np.meshgrid(np.arange(w), np.arange(h))
    X = np.stack([ix.ravel() * sx, rng.uniform(-0.05, 0.05, w * h), iy.ravel() * sy, rng.random(w * h)], 1).astype(np.float32)
    X[:, :3] += (0.2 * min(sx, sy) * rng.standard_normal((w * h, 3))).astype(np.float32)
    XL = X.copy()
    XL[:, :3] -= (0.01 * rng.standard_normal((w * h, 3))).astype(np.float32)
    pin = (rng.random(w * h) < 0.1).astype(np.uint8)
    g = VerletGrid(w, h, X, XL, pin, p)
    buf = DeviceBuffer(16 * w * h) if vbo else None
    g.step(3, buf.ptr if vbo else None)
    Xg, XLg = g.get_state()
    Xr, XLr = Oracle(32).vgrid_rollout(w, h, X, XL, pin, p, 3)
    assert np.array_equal(Xg.view(np.uint32), Xr.view(np.uint32)) and np.array_equal(XLg.view(np.uint32), XLr.view(np.uint32))
    if vbo:
        out = np.empty((w * h, 4), np.float32)
        device_synchronize()
        buf.to_host(out)
        assert np.array_equal(out.view(np.uint32), Xr.view(np.uint32))
    g.close()
