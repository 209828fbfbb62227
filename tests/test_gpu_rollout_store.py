"""The two ways through a rollout's backward pass give the same bits: from
the states kept while running forward, and (once parameters have been set
again) by running each segment forward again from its checkpoint."""
import numpy as np
import pytest

from opencloth_amd import scenes
from tests.helpers import say

pytestmark = pytest.mark.gpu


def same(a, b):
    return all(np.array_equal(x.view(np.uint32), y.view(np.uint32)) for x, y in zip(a, b))


@pytest.mark.parametrize("steps,every", [(1, 1), (1, 5), (5, 1), (5, 2), (6, 3), (7, 7), (4, 9)])
@pytest.mark.parametrize("batch", [False, True])
def test_kept_states_equal_recomputed(steps, every, batch):
    from opencloth_amd.batch import ClothBatch
    from opencloth_amd.cloth import ImplicitCloth

    say("rollout store", steps, every, batch)
    rng = np.random.default_rng(steps * 10 + every)
    if batch:
        sc = scenes.batch_diff_scene(n_cloths=5, sides=(9, 21), seed=1)
        h, kw = ClothBatch.from_scene(sc), {"n_springs": len(sc.springs)}
    else:
        sc, kw = scenes.plain_scene(), {}
        h = ImplicitCloth.from_scene(sc)
    X0 = (sc.X + 1e-3 * rng.standard_normal(sc.X.shape)).astype(np.float32)
    V0 = (0.1 * rng.standard_normal(sc.X.shape)).astype(np.float32)
    h.set_state(X0, V0)
    h.rollout_forward(steps, every)
    end = h.get_state()
    gx = rng.standard_normal(sc.X.shape).astype(np.float32)
    kept = h.rollout_backward(gx, **kw)
    assert same(h.get_state(), end)
    assert same(h.rollout_backward(gx, **kw), kept)  # nothing kept was overwritten
    h.set_params(sc.params)
    again = h.rollout_backward(gx, **kw)
    assert same(again, kept) and same(h.get_state(), end)
    # a longer rollout grows the store, a shorter one fits it
    for n in (steps + 9, steps):
        h.set_state(X0, V0)
        h.rollout_forward(n, every)
        g = h.rollout_backward(gx, **kw)
    assert same(g, kept)
    h.close()
