"""Solves of one and two iterations on cloths of more and of at most 128 tiles: a
single iteration of the larger ones goes by launches (they are counted), the
others are resident; each step bit-exact against the FP32 oracle, also when the
cap changes from step to step."""
import dataclasses

import numpy as np
import pytest

from opencloth_amd import scenes
from tests.helpers import oracle_params, say

pytestmark = pytest.mark.gpu

P = scenes.StepParams(dt=1.0 / 120.0, cg_max_iters=1, cg_tol=0.0, cg_tol_mode=scenes.TOL_NONE)


@pytest.mark.parametrize("nx,ny,large", [(400, 300, True), (512, 512, True), (320, 400, True), (257, 200, False), (256, 250, False)])
def test_short_solves(nx, ny, large):
    from opencloth_amd.cloth import ImplicitCloth
    from oracle import Oracle

    say("short solves", nx, ny)
    X0 = scenes.grid_positions(nx, ny, 4.0, 0.0)
    rng = np.random.default_rng(nx + ny)
    X = (X0 + 1e-3 * rng.standard_normal(X0.shape)).astype(np.float32)
    V = (0.1 * rng.standard_normal(X0.shape)).astype(np.float32)
    pins = np.zeros(nx * ny, np.uint8)
    pins[:nx] = 1
    sp = scenes.grid_springs(nx, ny, X0)
    cl = ImplicitCloth(nx, ny, X, sp, pins, P, V)
    o = Oracle(32)
    s = o.system(nx * ny, sp, pins)
    prev = o.set_threads(8)
    for its in (1, 2, 1):
        p = dataclasses.replace(P, cg_max_iters=its)
        cl.set_params(p)
        cl.set_state(X, V)
        cl.set_dv(None)
        launches = cl.profile_steps(2)
        assert launches["cg_axpy"][1] == (2 * its if large and its == 1 else 0), launches
        Xr, Vr, _, _, it, st = s.rollout(X, V, oracle_params(p, nx, ny), 2)
        X, V = cl.get_state()
        assert cl.last_status()[0] == it[-1] and cl.sticky_status() == st
        assert np.array_equal(X.view(np.uint32), Xr.view(np.uint32)) and np.array_equal(V.view(np.uint32), Vr.view(np.uint32))
    o.set_threads(prev)
    cl.close()
