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


def _instanced_view():
    """Twelve instances drawn together, seen whole, under the daylight sky."""
    sc = scenes.instanced(n_instances=12, subdiv=2, seed=4, width=24, height=24, spp=8, max_depth=3)
    sc["instances"][:, 3:12:4] *= 0.05  # translations: the spheres (radius 0.5 to 2) overlap in a 5-unit box
    sc["camera"].update(position=(2.5, 2.5, -8.0), target=(2.5, 2.5, 2.5))
    sc["sky"] = dict(enabled=True, draw_sun=True, dir=(0.3, 0.8, -0.5), angular_diameter=32.0, intensity=1000.0,
                     turbidity=4.0)
    return sc


def test_adjoint_of_an_instanced_scene(rend):
    """The adjoint's shadow rays through two levels: the gradient against the oracle's FP64
    accumulation. Both sides evaluate the same float terms; the device adds at most
    n = 24 x 24 x 8 x 3 of them per parameter in float, whose rounding is below
    n 2^-24 ~ 8e-4 of the terms' magnitudes in the worst case and about sqrt(n) 2^-24 ~ 7e-6
    as it accumulates: 1e-3 of the largest gradient bounds it."""
    sc = _instanced_view()
    rend.UpdateScene(sc)
    theta = scenes.material_params(sc["materials"])
    rend.set_material_params(theta, which=3)
    rend.RenderFrame()
    img = rend.color()[..., :3]
    dldi = (2.0 * (img - 0.5 * img.mean())).astype(np.float32)
    g = rend.backward(dldi)
    orc = _oracle(sc)
    orc.set_material_params(theta, which=3)
    np.testing.assert_array_equal(img, orc.render()["image_f32"])
    ref = orc.backward(dldi)
    assert (np.abs(ref).max(axis=1) > 0).sum() >= 8  # most of the twelve palettes take part
    assert np.abs(g - ref).max() <= 1e-3 * np.abs(ref).max()


def _node_bytes(rend):
    rend.settings.width = rend.settings.height = 16
    rend.settings.spp = 1
    return rend.measure_traversal()["node_bytes"]


@pytest.mark.parametrize("surrounding", [0.0, 3000.0], ids=["compact-nodes", "48-byte-nodes"])
def test_both_node_layouts_match_brute_force(rend, surrounding):
    """A soup, alone (its tree suits the 32-byte nodes) and as a small object far from the
    centre of a large surrounding (its tree is too fine for their grid): hits and occlusion
    equal a brute-force loop over random rays, rays parallel to an axis, unnormalised
    directions and origins far away; and so does a rendered frame, path by path."""
    sc = scenes.soup(n_tris=4000, seed=9, width=48, height=32, spp=4, max_depth=4)
    if surrounding:
        pos = sc["positions"].copy()
        pos[0] = np.tile([-surrounding, -surrounding, -surrounding], 3) + [0, 0, 0, 1, 0, 0, 0, 1, 0]
        pos[1] = np.tile([0.3 * surrounding, 0.2 * surrounding, 0.1 * surrounding], 3) + [0, 0, 0, 1, 0, 0, 0, 1, 0]
        sc["positions"] = pos
    rend.UpdateScene(sc)
    assert _node_bytes(rend) == (48 if surrounding else 32)
    rays = random_rays(6000, seed=3, toward=(0.0, 1.0))
    rng = np.random.default_rng(4)
    for k in range(3):  # parallel to an axis; the other components zero of either sign
        rays[k * 500:(k + 1) * 500, 4:7] = 0.0
        rays[k * 500:(k + 1) * 500, 4 + k] = rng.choice([-1.0, 1.0], 500)
        rays[k * 500:k * 500 + 250, 4 + (k + 1) % 3] = -0.0
    rays[2000:2500, 4:7] *= 1e-6
    rays[2500:3000, 4:7] *= 1e6
    rays[3000:3500, 0:3] = 0.5 - 1e4 * rays[3000:3500, 4:7]
    hit = _check(rend, sc, rays)
    assert hit.sum() > 1000
    rend.SetSettings(rend.settings.from_dict(sc["render"]))
    rend.RenderFrame()
    got = rend.path_radiance()
    want = _oracle(sc).render()["path_rgb"]
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("n", [1, 63, 1024, 1025, 4096, 4097, 70_001])
@pytest.mark.parametrize("levels", ["single", "two-level"])
def test_ray_query_sizes(rend, n, levels):
    """Ray queries at the edges of their paths (one checking block, pinned exchange, copies):
    hits, instances and occlusion equal the oracle's; an invalid last ray is named, and one
    whose only fault is a negative tmin is told apart."""
    from trayracer_amd._lib import TrtError
    sc = _tiny(36) if levels == "single" else _instanced_view()
    rend.UpdateScene(sc)
    rays = random_rays(n, seed=n, lo=-0.2, hi=1.2 if levels == "single" else 5.0, tmin=1e-4)
    orc = _oracle(sc)
    hg, ig = rend.trace_closest(rays)
    hb, ib = orc.trace_closest(rays)
    hit = prim_of(hb) != 0xFFFFFFFF
    assert np.array_equal(prim_of(hg), prim_of(hb)) and np.array_equal(ig, ib)
    assert np.array_equal(hg[hit].view(np.uint32), hb[hit].view(np.uint32))
    assert np.array_equal(rend.trace_any(rays), orc.trace_any(rays))
    for col, val, what in ((6, np.nan, "non-finite"), (3, -1.0, "negative tmin"), (7, np.nan, "NaN bound")):
        bad = rays.copy()
        bad[n - 1, col] = val
        for query in (rend.trace_closest, rend.trace_any):
            with pytest.raises(TrtError, match=f"ray {n - 1} .*{what}"):
                query(bad)
    assert np.array_equal(rend.trace_any(rays), orc.trace_any(rays))  # usable afterwards


@pytest.mark.parametrize("sky", [False, True])
def test_small_frames_after_large_ones(rend, sky):
    """A frame's counters are reset by RayGen's own threads, of which a small frame has few:
    1, 63 and 300 paths after a large frame, with emitter hits or a sky in the emission lists,
    give the oracle's paths, and the counting frame (no accumulation) the same rays."""
    sc = scenes.cornell(width=96, height=64, spp=3, max_depth=5, seed=31)
    if sky:
        sc["sky"] = dict(enabled=True, draw_sun=True, dir=(0.3, 0.8, -0.5), angular_diameter=32.0,
                         intensity=1000.0, turbidity=4.0, sun_nee=True)
    rend.UpdateScene(sc)
    orc = _oracle(sc)
    for size in (dict(width=96, height=64, spp=3), dict(width=1, height=1, spp=1), dict(width=9, height=7, spp=1),
                 dict(width=96, height=64, spp=3), dict(width=10, height=6, spp=5)):
        for k, v in size.items():
            setattr(rend.settings, k, v)
        rend.Reset()
        st = rend.RenderFrame()
        ref = orc.render(render=size)
        assert st["paths"] == st["primary_rays"] == size["width"] * size["height"] * size["spp"]
        assert np.array_equal(rend.path_radiance().view(np.uint32), ref["path_rgb"].view(np.uint32)), size
        assert (st["extend_rays"], st["shadow_rays"]) == tuple(ref["counts"].sum(axis=1)), size
        rend.Reset()  # the same samples again
        m = rend.measure_traversal()
        assert (m["closest_rays"], m["any_rays"]) == (st["extend_rays"], st["shadow_rays"]), size
