"""One array of a state at a time, to the device and back, bit for bit (NaN
payloads too), around the sizes at which its way changes: a copy from 16 KiB
(1365 vertices) on, several slots beyond 87384 vertices."""
import numpy as np
import pytest

from opencloth_amd import scenes
from tests.helpers import say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 1000, 1365, 1366, 1367, 4099, 87383, 87384, 87385, 200003])
def test_one_array(n):
    from opencloth_amd._lib import check, lib, ptr
    from opencloth_amd.cloth import PBDCloth

    rng = np.random.default_rng(n)
    say("one array", n)
    noise = lambda: rng.integers(0, 2**32, (n, 3), np.uint32, endpoint=False).view(np.float32)  # noqa: E731
    cl = PBDCloth(np.zeros((n, 3), np.float32), *scenes.pbd_grid_constraints(1, 1), None, scenes.PBDParams())
    now = [noise(), noise()]
    cl.set_state(*now)
    for k in (0, 1, 1, 0):
        now[k] = noise()
        cl.set_state(**{"XV"[k]: now[k]})
        for j in (0, 1):
            got = np.full((n, 3), 7.0, np.float32)
            args = [None, None]
            args[j] = ptr(got)
            check(lib().oc_pbd_get_state(cl.h, *args))
            assert np.array_equal(got.view(np.uint32), now[j].view(np.uint32)), (k, j)
        both = cl.get_state()
        assert all(np.array_equal(p.view(np.uint32), q.view(np.uint32)) for p, q in zip(both, now))
    cl.close()
