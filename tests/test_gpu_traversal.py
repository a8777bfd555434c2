"""GPU traversal: node layouts, leaf edge cases and the adjoint's shadow rays."""
import copy

import numpy as np
import pytest

from tests.gpu_util import prim_of, random_rays
from trayracer_amd import Renderer, scenes

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def rend():
    r = Renderer(0)
    yield r
    r.close()


def _oracle(scene):
    from oracle import Oracle
    return Oracle(scene)


def _check(rend, sc, rays):
    orc = _oracle(sc)
    hg, ig = rend.trace_closest(rays)
    hb, ib = orc.trace_closest(rays, brute=True)
    assert np.array_equal(prim_of(hg), prim_of(hb)) and np.array_equal(ig, ib)
    hit = prim_of(hb) != 0xFFFFFFFF
    assert np.array_equal(hg[hit].view(np.uint32), hb[hit].view(np.uint32))
    assert np.array_equal(rend.trace_any(rays), orc.trace_any(rays, brute=True))
    return hit


def _tiny(n_tris):
    sc = copy.deepcopy(scenes.cornell())
    sc["positions"] = np.asarray(sc["positions"], np.float32)[:n_tris]
    sc["mat_ids"] = np.asarray(sc["mat_ids"])[:n_tris]
    sc["meshes"] = [(0, n_tris)]
    return sc


@pytest.mark.parametrize("n_tris", [1, 2])
def test_rays_that_start_in_the_empty_child(rend, n_tris):
    """A root leaf is stored beside an empty child, a zero box at the origin; a ray that
    starts there with tmin = 0 (as a picked ray of a camera at the origin does) visits the
    empty child's leaf, which holds no triangle and must not keep the ray waiting."""
    sc = _tiny(n_tris)
    rend.UpdateScene(sc, presplit=0.0)
    rays = random_rays(300, seed=n_tris, tmin=0.0, toward=(-1.0, 1.0))
    rays[:200, 0:3] = 0.0
    _check(rend, sc, rays)
