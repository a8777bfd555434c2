"""Batches padded with all-zero ray records (no direction: such rays hit nothing)."""
import numpy as np
import pytest

from tests.gpu_util import prim_of, random_rays
from trayracer_amd import Renderer, scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scene", [lambda: scenes.soup(n_tris=5000, seed=2), lambda: scenes.instanced(n_instances=8, subdiv=2, seed=2)],
                         ids=["single-level", "two-level"])
@pytest.mark.parametrize("n", [100, 6000], ids=["pinned-exchange", "copies"])
def test_padding_misses_and_leaves_the_others_alone(scene, n):
    sc = scene()
    span = 1.0 if sc["instances"] is None else 100.0
    rays = random_rays(n, seed=5, lo=0.0, hi=1.0)
    rays[:, 0:3] *= span
    padded = np.zeros((2 * n, 8), np.float32)
    padded[::2] = rays
    padded[1::2, 0:3] = rays[:, 0:3]  # half of the padding at the rays' origins, with any length
    padded[1::4, 7] = 1e30
    padded[3::4, 0:3] = 0.0
    r = Renderer(0)
    try:
        r.UpdateScene(sc)
        hits, inst = r.trace_closest(rays)
        occ = r.trace_any(rays)
        ph, pi = r.trace_closest(padded)
        po = r.trace_any(padded)
    finally:
        r.close()
    assert np.array_equal(ph[::2].view(np.uint32), hits.view(np.uint32)) and np.array_equal(pi[::2], inst)
    assert np.array_equal(po[::2], occ)
    assert (prim_of(ph)[1::2] == 0xFFFFFFFF).all() and (po[1::2] == 0).all()
    assert np.array_equal(ph[1::2, 0], padded[1::2, 7])
