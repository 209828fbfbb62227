"""States of more than 2 MiB, which several host threads transfer, on a handle
whose stream is hipStreamPerThread (another stream in every thread): read
while steps are still running, and written right before steps."""
import ctypes

import numpy as np
import pytest

from opencloth_amd import scenes
from tests.helpers import say

pytestmark = pytest.mark.gpu

PER_THREAD = 2  # hipStreamPerThread


@pytest.mark.parametrize("kind", ["implicit", "pbd"])
def test_transfers_follow_the_callers_stream(kind):
    from opencloth_amd._lib import check, lib
    from opencloth_amd.cloth import ImplicitCloth, PBDCloth

    n = 448
    say("per-thread stream", kind)
    rng = np.random.default_rng(3)
    X = scenes.grid_positions(n, n, 4.0, 1.0)
    V = (1e-2 * rng.standard_normal(X.shape)).astype(np.float32)
    got = []
    for stream in (None, PER_THREAD):
        if kind == "implicit":
            h = ImplicitCloth(n, n, X, scenes.grid_springs(n, n, X), None,
                              scenes.StepParams(cg_max_iters=20, cg_tol=0.0, cg_tol_mode=scenes.TOL_NONE), V)
        else:
            h = PBDCloth(X, *scenes.pbd_grid_constraints(n, n), None, scenes.PBDParams(), V)
        if stream is not None:
            f = lib().oc_cloth_set_stream if kind == "implicit" else lib().oc_pbd_set_stream
            check(f(h.h, ctypes.c_void_p(stream)))
        out = []
        for k in (60, 40):
            h.step(k)
            out += h.get_state()
            h.set_state(X + np.float32(0.01 * k), V)
            h.step(2)
            out += h.get_state()
        got.append(out)
        h.close()
    for a, b in zip(*got):
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
