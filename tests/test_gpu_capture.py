"""Steps of a cloth captured into a HIP graph: every replay goes on from where
the cloth is, as the same eager call does, whatever the number of steps (an odd
number of updates inside assemblies would end in the other pair of buffers),
with eager steps in between."""
import ctypes as C

import numpy as np
import pytest

from opencloth_amd import scenes
from tests.helpers import say

pytestmark = pytest.mark.gpu

REL = scenes.StepParams(cg_max_iters=20, cg_tol=1e-4, cg_tol_mode=scenes.TOL_RELATIVE)
FIXED = scenes.StepParams(dt=1.0 / 120.0, cg_max_iters=8, cg_tol=0.0, cg_tol_mode=scenes.TOL_NONE)


@pytest.mark.parametrize("nx,ny,steps,p,entry", [(21, 21, 1, REL, "oc_cloth_step"), (21, 21, 2, REL, "oc_cloth_step"),
                                                 (130, 70, 3, FIXED, "oc_cloth_step"), (130, 70, 4, REL, "oc_cloth_step_noalloc"),
                                                 (640, 512, 2, FIXED, "oc_cloth_step")])
def test_replays_go_on(nx, ny, steps, p, entry):
    from opencloth_amd._lib import check, lib
    from opencloth_amd.cloth import ImplicitCloth
    from opencloth_amd.hiptime import Stream, device_synchronize, hip

    say("capture", nx, ny, steps, entry)
    X = scenes.grid_positions(nx, ny, 4.0, 0.0)
    rng = np.random.default_rng(nx + steps)
    X = (X + 1e-3 / max(nx, ny) * rng.standard_normal(X.shape)).astype(np.float32)
    pins = np.zeros(nx * ny, np.uint8)
    pins[:nx] = 1
    a, b = (ImplicitCloth(nx, ny, X, scenes.grid_springs(nx, ny, X), pins, p) for _ in range(2))
    s = Stream()
    a.set_stream(s.handle)
    a.step(1)
    b.step(1)
    device_synchronize()
    h, g, run = hip(), C.c_void_p(), C.c_void_p()
    assert h.hipStreamBeginCapture(s.s, 2) == 0  # relaxed
    rc = getattr(lib(), entry)(a.h, steps)
    assert h.hipStreamEndCapture(s.s, C.byref(g)) == 0
    check(rc)
    assert h.hipGraphInstantiate(C.byref(run), g, None, None, C.c_size_t(0)) == 0
    for k in range(4):
        assert h.hipGraphLaunch(run, s.s) == 0
        b.step(steps)
        for p0, p1 in zip(a.get_state(), b.get_state()):
            assert np.array_equal(p0.view(np.uint32), p1.view(np.uint32)), k
        assert a.last_status() == b.last_status()
        for n in (3, 2) if k == 1 else ():
            a.step(n)
            b.step(n)
    assert h.hipGraphExecDestroy(run) == 0 and h.hipGraphDestroy(g) == 0
    a.close()
    b.close()
