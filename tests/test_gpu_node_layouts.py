"""GPU traversal over both node layouts against the oracle, in scenes made for each."""
import numpy as np
import pytest

from tests.gpu_util import prim_of, random_rays
from trayracer_amd import Renderer, scenes

pytestmark = pytest.mark.gpu

SKY = dict(enabled=True, draw_sun=True, dir=(0.3, 0.8, -0.5), angular_diameter=32.0, intensity=1000.0, turbidity=4.0,
           sun_nee=True)


@pytest.fixture(scope="module")
def rend():
    r = Renderer(0)
    yield r
    r.close()


def _node_bytes(rend):
    rend.settings.width = rend.settings.height = 16
    rend.settings.spp = 1
    return rend.measure_traversal()["node_bytes"]


def _oracle(sc):
    from oracle import Oracle
    return Oracle(sc)


def _check_rays(rend, orc, rays):
    hg, ig = rend.trace_closest(rays)
    hb, ib = orc.trace_closest(rays, brute=True)
    assert np.array_equal(prim_of(hg), prim_of(hb)) and np.array_equal(ig, ib)
    hit = prim_of(hb) != 0xFFFFFFFF
    assert hit.mean() > 0.1
    assert np.array_equal(hg[hit].view(np.uint32), hb[hit].view(np.uint32))
    assert np.array_equal(rend.trace_any(rays), orc.trace_any(rays, brute=True))


def _check_frame(rend, sc, orc):
    rend.SetSettings(rend.settings.from_dict(sc["render"]))
    rend.RenderFrame()
    assert np.array_equal(rend.path_radiance().view(np.uint32), orc.render()["path_rgb"].view(np.uint32))


def _plates(axis, heights, half, n=24):
    """Squares of half side `half` at the heights on an axis, n x n cells of two triangles."""
    x = np.linspace(-half, half, n + 1)
    u, v = np.meshgrid(x, x)
    out = []
    for h in heights:
        p = np.empty((n + 1, n + 1, 3))
        p[..., axis], p[..., (axis + 1) % 3], p[..., (axis + 2) % 3] = h, u, v
        a, b, c, d = p[:-1, :-1], p[1:, :-1], p[1:, 1:], p[:-1, 1:]
        for t in ((a, b, c), (a, c, d)):
            out.append(np.concatenate(t, -1).reshape(-1, 9))
    return np.concatenate(out).astype(np.float32)


@pytest.mark.parametrize("axis,levels", [(0, 1), (1, 1), (2, 1), (1, 2)])
@pytest.mark.parametrize("half", [2.0, 50.0])
def test_plates_off_the_grid(rend, axis, levels, half):
    """Finely divided plates whose heights the 32-byte nodes' grid is fitted to: rays from,
    along and grazing the plates as well as random ones equal brute force, and a frame's paths
    the oracle's."""
    heights = (-1.00317, 1.7713)
    sc = scenes.soup(n_tris=1500, seed=6, width=40, height=24, spp=4, max_depth=4)
    plates = _plates(axis, heights, half)
    sc["positions"] = np.concatenate([sc["positions"], plates])
    sc["mat_ids"] = np.concatenate([sc["mat_ids"], np.full(len(plates), 7, np.uint32)])
    sc["meshes"] = [(0, len(sc["positions"]))]
    sc["sky"] = SKY
    if levels == 2:
        sc["instances"] = np.zeros((1, 14), np.float32)
        sc["instances"][0, [0, 5, 10]] = 1.0
    rend.UpdateScene(sc)
    assert _node_bytes(rend) == 32
    orc = _oracle(sc)
    rng = np.random.default_rng(axis)
    rays = random_rays(6000, seed=8, lo=-1.5, hi=2.5, toward=(-1.0, 2.0))
    rays[:3000, 0:3] = rng.uniform(-half, half, (3000, 3))
    rays[:3000, axis] = np.float32(rng.choice(heights, 3000))
    rays[:1500, 4 + axis] *= np.float32(10.0) ** rng.uniform(-9, 0, 1500).astype(np.float32)
    rays[1500:1800, 4 + axis] = 0.0
    _check_rays(rend, orc, rays)
    _check_frame(rend, sc, orc)


def _cluster(n, radius, spread, at, seed):
    """n instances (14 floats) of mesh 0 of the given radius within `spread` of a place."""
    rng = np.random.default_rng(seed)
    inst = np.zeros((n, 14), np.float32)
    for i in range(n):
        m = np.zeros((3, 4))
        m[:, :3] = scenes._random_rotation(rng) * radius * rng.uniform(0.5, 1.0)
        m[:, 3] = np.asarray(at) + rng.uniform(-spread, spread, 3)
        inst[i, :12] = m.reshape(-1)
        inst[i, 12:14] = np.array([0, i % 3], np.uint32).view(np.float32)
    return inst


def _two_level(refusing):
    """A two-level scene that takes 48-byte nodes, by a mesh with a small detailed part in a large
    one, or by a top level with small instances between far ones; seen from nearby."""
    pos, _ = scenes.icosphere(1 if refusing == "top level" else 3)
    if refusing == "top level":
        at = np.array([600.0, 10.0, -300.0])
        inst = np.concatenate([_cluster(150, 0.06, 0.5, at, 5), _cluster(4, 0.3, 2.0, at, 6), _cluster(2, 1.0, 1.0, (-3000, -3000, -3000), 7),
                               _cluster(2, 1.0, 1.0, (3000, 3000, 2000), 8)])
    else:
        at = np.array([0.2, 0.1, 0.1]) * 3000.0 + [0.3, 0.2, 0.1]
        pos = np.concatenate([pos * 0.5 + np.tile(at, 3),
                              np.tile([-3000.0, -3000.0, -3000.0], 3)[None] + np.array([[0, 0, 0, 1, 0, 0, 0, 1, 0]]),
                              np.tile([3000.0, 3000.0, 3000.0], 3)[None] + np.array([[0, 0, 0, 1, 0, 0, 0, 1, 0]])]).astype(np.float32)
        inst = np.zeros((4, 14), np.float32)
        for i in range(4):
            m = np.zeros((3, 4))
            m[:, :3] = np.eye(3)
            m[:, 3] = [0.7 * (i % 2), 0.6 * (i // 2), 0.1 * i]
            inst[i, :12] = m.reshape(-1)
            inst[i, 12:14] = np.array([0, i % 3], np.uint32).view(np.float32)
        at = at + [0.35, 0.3, 0.15]
    mats = np.stack([scenes.material(c, roughness=r, metallic=m) for c, r, m in
                     (((0.8, 0.3, 0.2), 0.4, 0.0), ((0.3, 0.7, 0.4), 0.7, 0.2), ((0.4, 0.4, 0.9), 0.3, 0.8))])
    cam = dict(position=tuple(at + [0.0, 0.4, -3.0]), target=tuple(at), up=(0, 1, 0), fov=0.7, aperture=0.0, focal_dist=1.0,
               distortion=0.0, bokeh_sides=0, bokeh_rotation=0.0)
    return at, dict(positions=pos, normals=None, mat_ids=np.zeros(len(pos), np.uint32), meshes=[(0, len(pos))], materials=mats,
                    instances=inst, camera=cam, sky=SKY,
                    render=dict(width=24, height=24, spp=8, max_depth=3, rr_depth=3, seed=2, ray_epsilon=1e-3, clamp=0.0))


def _check_backward(rend, sc):
    """The gradient against the oracle's FP64 accumulation of the same float terms: the device
    adds at most n = 24 x 24 x 8 x 3 per parameter in float, whose rounding is about
    sqrt(n) 2^-24 ~ 7e-6 of the terms' magnitudes as it accumulates, below n 2^-24 ~ 8e-4 in the
    worst case: 1e-3 of the largest gradient bounds it."""
    theta = scenes.material_params(sc["materials"])
    rend.set_material_params(theta, which=3)
    rend.SetSettings(rend.settings.from_dict(sc["render"]))
    assert rend.RenderFrame()["shadow_rays"] > 500
    img = rend.color()[..., :3]
    dldi = (2.0 * (img - 0.5 * img.mean())).astype(np.float32)
    g = rend.backward(dldi)
    orc = _oracle(sc)
    orc.set_material_params(theta, which=3)
    np.testing.assert_array_equal(img, orc.render()["image_f32"])
    ref = orc.backward(dldi)
    assert (np.abs(ref).max(axis=1) > 0).sum() >= 3
    assert np.abs(g - ref).max() <= 1e-3 * np.abs(ref).max()


@pytest.mark.parametrize("refusing", ["mesh", "top level"])
def test_two_level_scenes_on_48_byte_nodes(rend, refusing):
    """Hits, occlusion, a frame's paths and the gradient of two-level scenes whose trees do not
    suit the 32-byte nodes."""
    at, sc = _two_level(refusing)
    rend.UpdateScene(sc)
    assert _node_bytes(rend) == 48
    orc = _oracle(sc)
    rays = random_rays(3000, seed=11, lo=-2.0, hi=2.0, toward=(-0.6, 0.6))
    rays[:, 0:3] += at.astype(np.float32)
    rays[:300, 4:7] = 0.0
    for k in range(3):  # parallel to an axis
        rays[100 * k:100 * (k + 1), 4 + k] = 1.0
    rays[300:600, 4:7] *= 1e4
    _check_rays(rend, orc, rays)
    _check_frame(rend, sc, orc)
    _check_backward(rend, sc)


def test_gradient_on_48_byte_nodes(rend):
    """The adjoint's shadow rays through a single-level tree of 48-byte nodes."""
    sc = scenes.soup(n_tris=6000, seed=12, width=24, height=24, spp=8, max_depth=3, n_emissive=6)
    far = np.tile(np.array([[-3000.0], [2000.0]]), (1, 9)) + np.array([0, 0, 0, 1, 0, 0, 0, 1, 0])
    sc["positions"] = np.concatenate([sc["positions"], far]).astype(np.float32)
    sc["mat_ids"] = np.concatenate([sc["mat_ids"], np.zeros(2, np.uint32)])
    sc["meshes"] = [(0, len(sc["positions"]))]
    sc["sky"] = SKY
    rend.UpdateScene(sc)
    assert _node_bytes(rend) == 48
    _check_backward(rend, sc)
