"""Host arrays to the device and back, bit for bit (NaN payloads too), at the
transfer's edges: a slot holds 87384 vertices of xyz or 65538 of xyzw, both
arrays of a state go together up to a slot, and each 2 MiB bring a thread."""
import numpy as np
import pytest

from opencloth_amd import scenes
from tests.helpers import say

pytestmark = pytest.mark.gpu


def noise(rng, n, c):
    return rng.integers(0, 2**32, (n, c), np.uint32, endpoint=False).view(np.float32)


def same(a, b):
    return np.array_equal(a.view(np.uint32), b.view(np.uint32))


@pytest.mark.parametrize("n", [1, 2, 3, 5, 64, 341, 43691, 43692, 43693, 87384, 87385, 262145, 349526, 700001, 1048577])
def test_xyz(n):
    from opencloth_amd.cloth import PBDCloth

    rng = np.random.default_rng(n)
    say("state io xyz", n)
    d, b = scenes.pbd_grid_constraints(1, 1)
    cl = PBDCloth(np.zeros((n, 3), np.float32), d, b, None, scenes.PBDParams())
    X, V = noise(rng, n, 3), noise(rng, n, 3)
    cl.set_state(X, V)
    Xg, Vg = cl.get_state()
    assert same(Xg, X) and same(Vg, V)
    X = noise(rng, n, 3)
    cl.set_state(X=X)
    Xg, Vg = cl.get_state()
    assert same(Xg, X) and same(Vg, V)
    V = noise(rng, n, 3)
    cl.set_state(V=V)
    Xg, Vg = cl.get_state()
    assert same(Xg, X) and same(Vg, V)
    cl.close()


@pytest.mark.parametrize("nx,ny", [(2, 2), (3, 5), (181, 181), (182, 181), (256, 257), (600, 701)])
def test_xyzw(nx, ny):
    from opencloth_amd.cloth import VerletGrid

    rng = np.random.default_rng(nx)
    say("state io xyzw", nx, ny)
    g = VerletGrid(nx, ny, noise(rng, nx * ny, 4))
    X, XL = noise(rng, nx * ny, 4), noise(rng, nx * ny, 4)
    g.set_state(X, XL)
    Xg, Lg = g.get_state()
    assert same(Xg, X) and same(Lg, XL)
    XL = noise(rng, nx * ny, 4)
    g.set_state(None, XL)
    Xg, Lg = g.get_state()
    assert same(Xg, X) and same(Lg, XL)
    g.close()
