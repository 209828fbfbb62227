"""The tags of the resident solve's exchanges are 32 bits wide.  A solve of one
iteration, then as many solves that stop at once as would bring the tags round
if each took all that 65536 iterations can use, then a solve that iterates: the
same bits as on a handle without the solves in between."""
import dataclasses

import numpy as np
import pytest

from opencloth_amd import scenes
from tests.helpers import say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("idle", [32767, 1])
def test_idle_solves_use_no_tags(idle):
    from opencloth_amd.cloth import ImplicitCloth

    nx, ny, its = 130, 70, 65536
    X0 = scenes.grid_positions(nx, ny, 4.0, 0.0)
    rng = np.random.default_rng(7)
    X = (X0 + 2e-3 * rng.standard_normal(X0.shape)).astype(np.float32)
    V = (0.1 * rng.standard_normal(X0.shape)).astype(np.float32)
    pins = np.zeros(nx * ny, np.uint8)
    pins[:nx] = 1
    one = scenes.StepParams(cg_max_iters=its, cg_tol=0.99, cg_tol_mode=scenes.TOL_RELATIVE)
    none = dataclasses.replace(one, cg_tol=1e15, cg_tol_mode=scenes.TOL_ABSOLUTE)
    many = dataclasses.replace(one, cg_tol=1e-4)
    got = []
    for n in (idle, 0):
        say("idle solves", n)
        cl = ImplicitCloth(nx, ny, X, scenes.grid_springs(nx, ny, X0), pins, one, V)
        cl.step(1)
        assert cl.last_status()[0] == 1
        cl.set_params(none)
        for left in range(n, 0, -4096):
            cl.step(min(left, 4096))
            assert cl.last_status()[0] == 0
        for k in range(3):
            cl.set_params(many)
            cl.set_state(X, V)
            cl.set_dv(None)
            cl.step(1)
            it, st = cl.last_status()
            got.append((it, *cl.get_state()))
            assert it > 1 and st == 0
            cl.set_params(one)
            cl.set_state(X, V)
            cl.set_dv(None)
            cl.step(1)
        cl.close()
    for a, b in zip(got[:3], got[3:]):
        assert a[0] == b[0]
        assert all(np.array_equal(p.view(np.uint32), q.view(np.uint32)) for p, q in zip(a[1:], b[1:]))
