"""The PBD step's routes against the FP32 oracle in colour order, bit for bit,
at the edges of their ranges: one workgroup up to 2048 particles (512, 1024
and 2048 are its instances' limits), blocks of up to 1024 owned particles
beyond, closures of more than 64 KB of LDS, and lists that reach too far for
blocks, which run a launch per colour."""
import dataclasses

import numpy as np
import pytest

from opencloth_amd import scenes
from tests.helpers import say

pytestmark = pytest.mark.gpu


def bits(a):
    return np.ascontiguousarray(a, np.float32).view(np.uint32)


def springs(a, b, k):
    d = np.zeros(len(a), scenes.PBD_DISTANCE_DTYPE)
    d["p1"], d["p2"], d["k"] = a, b, k
    return d


CASES = [  # nx, ny, solver iterations, variant
    (1, 1, 2, ""), (2, 1, 1, ""), (16, 16, 2, "k"), (257, 1, 3, ""), (32, 16, 1, "ball"), (27, 19, 2, "k"),
    (32, 32, 2, "ball"), (41, 25, 5, ""), (64, 32, 2, "k"), (64, 32, 2, "none"), (683, 3, 2, "k"),
    (97, 61, 1, "ball"), (97, 61, 2, "ball"), (97, 61, 3, "k"), (130, 127, 2, ""), (50, 50, 2, "none"),
    (150, 140, 2, "reach"), (50, 50, 2, "far"),
]


@pytest.mark.parametrize("nx,ny,ns,variant", CASES)
def test_routes_bitwise(nx, ny, ns, variant):
    from oracle import Oracle, make_pbd_params
    from opencloth_amd.cloth import PBDCloth

    rng = np.random.default_rng(nx * 1000 + ny)
    N = nx * ny
    X = np.stack([np.tile(np.arange(nx), ny) * 0.1 - 1.0, np.full(N, 0.02), np.repeat(np.arange(ny), nx) * 0.1], -1)
    X = (X + 0.01 * rng.standard_normal(X.shape)).astype(np.float32)
    V = (0.3 * rng.standard_normal(X.shape)).astype(np.float32)
    pinned = (rng.random(N) < 0.05).astype(np.uint8)
    V[pinned.astype(bool)] = 0
    dist, bend = scenes.pbd_grid_constraints(nx, ny)
    i = np.arange(N)
    if variant == "none":
        dist, bend = dist[:0], bend[:0]
    elif variant == "reach":  # springs over ten spacings
        r, c = i[i % nx < nx - 10], i[i < N - 10 * nx]
        dist = np.concatenate([dist, springs(r, r + 10, 0.2), springs(c, c + 10 * nx, 0.2)])
    elif variant == "far":
        dist = np.concatenate([dist] + [springs(i[:N // 2], rng.permutation(N // 2) + N // 2, 0.05) for _ in range(4)])
    elif variant == "k":
        dist["k"], bend["k"] = rng.random(len(dist)), rng.random(len(bend))
    prm = scenes.PBDParams(mass=float(np.float32(1.0) / np.float32(N)), solver_iterations=ns, k_damp=0.02)
    prm = dataclasses.replace(prm, ground=variant != "ball")
    ell = scenes.ellipsoid() if variant == "ball" else None
    if ell is not None:
        X[:, 1] += 2.2
    say("pbd route", nx, ny, ns, variant)
    cl = PBDCloth(X, dist, bend, pinned, prm, V)
    s = Oracle(32).pbd(X, pinned, prm.mass, dist, bend, ns)
    for n in (1, 3):
        cl.step(n, ell)
        X, V = s.step(X, V, make_pbd_params(prm), 1, n, ell)
        Xg, Vg = cl.get_state()
        assert np.array_equal(bits(Xg), bits(X)), n
        assert np.array_equal(bits(Vg), bits(V)), n
    assert np.isfinite(X).all()
    cl.close()
