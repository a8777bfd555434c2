"""What a user of the renderer has it do, as cases that can be timed and compared.

Five kinds of work, each through the methods of ``trayracer_amd.Renderer``:

``rays``      a batch of ray queries on host arrays (``trace_closest`` / ``trace_any``):
              picking and visibility probes at the small end, baking at the large one
``frames``    a progressive render from a reset: some frames, then the image that the
              program shows (``tonemap``) or keeps (``color``)
``gradient``  one step of inverse rendering: set the material parameters, render, read the
              image, and differentiate a loss of it (``backward``)
``denoise``   the learned denoiser on a rendered frame, and its image
``train``     training steps of that denoiser on rendered pairs

Scenes are the package's own procedural ones (``trayracer_amd.scenes``), at the sizes of
its benchmark configurations and tests or of the same order. Every seed is another input:
another soup, other instances, another camera, other rays, parameters, crops.

Rendered images, what is computed from them (denoised images, trained weights) and the
gradients of a Monte Carlo render follow from the renderer's own random number streams, so
they have no value that could be had without it; the closest hits of free rays do.
"""
import math

import numpy as np

from trayracer_amd import Renderer, scenes
from trayracer_amd.renderer import KernelSettings

SKY = dict(enabled=True, draw_sun=True, dir=(0.3, 0.8, -0.5), angular_diameter=32.0, intensity=1000.0, turbidity=4.0)


def listed():
    return [
        # a probe of a tool or a game loop: a few rays, where the call itself is what counts
        dict(name="rays-pick", kind="rays", scene="cornell", size=36, rays=64, query="closest"),
        # baking or a sensor model: as many rays as a 1000 x 1000 image, incoherent
        dict(name="rays-closest-1m", kind="rays", scene="soup", size=250_000, rays=1_000_003, query="closest"),
        # visibility between points of an instanced scene, a ragged count
        dict(name="rays-any-200k", kind="rays", scene="instanced", size=200, rays=200_003, query="any"),
        # the interactive view while the camera moves: one sample, shown at once
        dict(name="frame-preview", kind="frames", scene="cornell", size=36, width=640, height=360, spp=1, frames=1,
             depth=4, mode="path_tracing", sky=False, lens=False, show=True),
        # the Cornell box of the convergence tests: 256 x 256, 16 spp, depth 4
        dict(name="frame-cornell", kind="frames", scene="cornell", size=36, width=256, height=256, spp=16, frames=1,
             depth=4, mode="path_tracing", sky=False, lens=False, show=False),
        # the benchmark's soup, 1M triangles at 1080p, 8 spp, depth 8: an offline still
        dict(name="frames-soup", kind="frames", scene="soup", size=1_000_000, width=1920, height=1080, spp=8, frames=4,
             depth=8, mode="path_tracing", sky=False, lens=False, show=False),
        # the benchmark's two-level scene, 1000 instances at 4K, 4 spp, depth 6
        dict(name="frames-instanced-4k", kind="frames", scene="instanced", size=1000, width=3840, height=2160, spp=4,
             frames=2, depth=6, mode="path_tracing", sky=False, lens=False, show=True),
        # daylight with the sun as a light, a thin lens and a clamp on a film of odd sides
        dict(name="frame-sky-ragged", kind="frames", scene="soup", size=100_003, width=1279, height=717, spp=3,
             frames=2, depth=5, mode="path_tracing", sky=True, lens=True, show=False),
        # inverse rendering of the differentiable Cornell box: 512 x 512, 64 spp
        dict(name="gradient-cornell", kind="gradient", scene="cornell", size=36, width=512, height=512, spp=64, depth=4),
        # and of a mesh with a material on every triangle, a few samples a step
        dict(name="gradient-mesh", kind="gradient", scene="soup", size=2500, width=256, height=256, spp=4, depth=4),
        # the denoised view at full HD
        dict(name="denoise-1080p", kind="denoise", width=1920, height=1080, spp=2),
        # training: two steps of batches of eight 128 x 128 crops, as the training schedule has them
        dict(name="train-128", kind="train", steps=2, batch=8, crop=128),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _scene_of(rng, soup_hi, inst_hi):
    kind = rng.choice(["cornell", "soup", "instanced"])
    return kind, dict(cornell=36, soup=_log(rng, 500, soup_hi), instanced=_log(rng, 4, inst_hi))[kind]


def draw(rng):
    kind = rng.choice(["rays", "rays", "frames", "frames", "frames", "gradient", "denoise", "train"])
    if kind == "rays":
        scene, size = _scene_of(rng, 250_000, 300)
        return dict(kind=kind, scene=scene, size=size, rays=_log(rng, 16, 1_200_000),
                    query=rng.choice(["closest", "closest", "any"]))
    if kind == "frames":
        scene, size = _scene_of(rng, 250_000, 500)
        w = _log(rng, 64, 1920)
        h = max(33, int(w * rng.uniform(0.4, 1.1)))
        spp = min(_log(rng, 1, 32), max(1, 12_000_000 // (w * h)))
        return dict(kind=kind, scene=scene, size=size, width=w, height=h, spp=spp, frames=rng.randint(1, 3),
                    depth=rng.randint(2, 8),
                    mode=rng.choice(["path_tracing", "path_tracing", "path_tracing", "ambient_occlusion", "shading_normal"]),
                    sky=rng.random() < 0.4, lens=rng.random() < 0.4, show=rng.random() < 0.5)
    if kind == "gradient":
        scene = rng.choice(["cornell", "soup"])
        w, h = _log(rng, 48, 512), _log(rng, 48, 512)
        return dict(kind=kind, scene=scene, size=36 if scene == "cornell" else _log(rng, 100, 3000), width=w, height=h,
                    spp=min(_log(rng, 2, 64), max(1, (8_000_000 if scene == "cornell" else 400_000) // (w * h))),
                    depth=rng.randint(2, 5))
    if kind == "denoise":
        # the network takes widths in multiples of 128 and heights in multiples of 8
        return dict(kind=kind, width=128 * rng.randint(1, 15), height=8 * rng.randint(4, 135), spp=rng.randint(1, 8))
    crop = rng.choice([128, 128, 256])
    return dict(kind=kind, steps=rng.randint(1, 3), batch=rng.randint(1, 8 if crop == 128 else 2), crop=crop)


# ---------------------------------------------------------------------------- preparation
def _make_scene(case, seed):
    if case["scene"] == "soup":
        sc = scenes.soup(n_tris=case["size"], seed=seed, n_emissive=min(64, case["size"] // 4))
    elif case["scene"] == "instanced":
        sc = scenes.instanced(n_instances=case["size"], subdiv=5 if case["size"] >= 1000 else 4, seed=seed)
    else:
        sc = scenes.cornell(seed=seed)
    return sc


def _camera(case, rng, sc):
    """The scene's camera, moved a little by the seed."""
    cam = dict(sc["camera"])
    span = 100.0 if case["scene"] == "instanced" else 1.0
    cam["position"] = tuple(float(p + span * 0.04 * rng.uniform(-1, 1)) for p in cam["position"])
    if case.get("lens"):
        cam["aperture"] = 0.01 * span
        cam["focal_dist"] = 1.5 * span
    return cam


def _bounds(sc):
    if sc["instances"] is not None:
        return np.zeros(3), np.full(3, 100.0)
    v = sc["positions"].reshape(-1, 3)
    return v.min(0).astype(np.float64), v.max(0).astype(np.float64)


def _rays(case, seed):
    """(scene, rays [n, 8]): origins all over the scene's bounds, directions all over the
    sphere, as far as twice the scene's diagonal."""
    sc = _make_scene(case, seed)
    rng = np.random.default_rng(seed + 17)
    lo, hi = _bounds(sc)
    n = case["rays"]
    rays = np.empty((n, 8), np.float32)
    rays[:, 0:3] = lo + (hi - lo) * rng.random((n, 3))
    d = rng.normal(size=(n, 3))
    rays[:, 4:7] = d / np.linalg.norm(d, axis=1, keepdims=True)
    diag = float(np.linalg.norm(hi - lo))
    rays[:, 3] = 1e-5 * diag
    rays[:, 7] = 2.0 * diag
    return sc, rays


def _settings(case, seed):
    eps = {"soup": 1e-5, "instanced": 1e-4, "cornell": 1e-3}[case["scene"]]
    return KernelSettings(width=case["width"], height=case["height"], spp=case["spp"], max_depth=case["depth"],
                          rr_depth=3, seed=seed, ray_epsilon=eps, clamp=10.0 if case.get("sky") else 0.0,
                          mode=_MODES[case.get("mode", "path_tracing")],
                          ao_dist=10.0 if case["scene"] == "instanced" else 0.2)


_MODES = dict(path_tracing=0, ambient_occlusion=1, shading_normal=8)


def _cornell_frames(r, rng, seed, width, height, spp):
    """Renders `spp` samples of the Cornell box from a camera of the seed."""
    r.SetCamera(dict(position=(rng.uniform(0.3, 0.7), rng.uniform(0.3, 0.7), rng.uniform(-1.5, -0.8)),
                     target=(0.5, 0.5, 0.5), up=(0.0, 1.0, 0.0), fov=math.radians(rng.uniform(35.0, 50.0))))
    r.SetSettings(KernelSettings(width=width, height=height, spp=spp, max_depth=4, rr_depth=3, seed=seed))
    r.RenderFrame()


def prepare(case, seed):
    rng = np.random.default_rng(seed)
    r = Renderer(0)
    state = dict(case=case, r=r)
    if case["kind"] == "rays":
        sc, state["rays"] = _rays(case, seed)
        r.UpdateScene(sc)
    elif case["kind"] == "frames":
        sc = _make_scene(case, seed)
        sc["camera"] = _camera(case, rng, sc)
        if case["sky"]:
            sc["sky"] = dict(SKY, sun_nee=True)
        r.UpdateScene(sc)
        r.SetSettings(_settings(case, seed))
        r.SetPhaseTiming(False)
    elif case["kind"] == "gradient":
        if case["scene"] == "cornell":
            sc, target = scenes.cornell_diff(seed=seed)
        else:
            sc = _make_scene(case, seed)
            p = scenes.material_params(sc["materials"])
            target = np.clip(p + rng.normal(0.0, 0.1, p.shape).astype(np.float32), scenes.PARAM_LO, scenes.PARAM_HI)
            sc["sky"] = SKY  # seen from outside, the soup is lit by the sky
        r.UpdateScene(sc)
        r.SetSettings(_settings(case, seed))
        r.SetPhaseTiming(False)
        r.set_material_params(target, which=r.BOTH)
        r.RenderFrame()
        state["target"] = r.color()[..., :3].copy()
        state["params"] = scenes.material_params(sc["materials"])
    elif case["kind"] == "denoise":
        r.UpdateScene(scenes.cornell())
        r.denoiser_init(seed=seed)
        _cornell_frames(r, rng, seed, case["width"], case["height"], case["spp"])
    else:
        width, height, pairs = 512, 384, 4
        r.UpdateScene(scenes.cornell())
        r.denoiser_init(seed=seed)
        r.denoiser_dataset(pairs, width, height)
        for k in range(pairs):
            cam = np.random.default_rng(seed + k)
            _cornell_frames(r, cam, seed + k, width, height, 2 ** k)
            r.denoiser_capture(k, 0)
            cam = np.random.default_rng(seed + k)
            _cornell_frames(r, cam, seed + 100 + k, width, height, 64)
            r.denoiser_capture(k, 1)
        state["seed"] = seed
    return state


# ------------------------------------------------------------------------------ one pass
def run(state):
    case, r = state["case"], state["r"]
    if case["kind"] == "rays":
        if case["query"] == "any":
            return {"occluded": r.trace_any(state["rays"])}
        hits, inst = r.trace_closest(state["rays"])
        return {"t_b1_b2": hits[:, :3], "prim": hits[:, 3].view(np.uint32), "inst": inst}
    if case["kind"] == "frames":
        r.Reset()
        for _ in range(case["frames"]):
            r.RenderFrame()
        return {"image": r.tonemap() if case["show"] else r.color()}
    if case["kind"] == "gradient":
        r.set_material_params(state["params"], which=r.BOTH)
        r.RenderFrame()
        img = r.color()
        grad = r.backward(2.0 * (img[..., :3] - state["target"]))
        return {"image": img, "gradient": grad}
    if case["kind"] == "denoise":
        r.denoise()
        return {"image": r.denoised()}
    losses = r.denoiser_train(case["steps"], batch=case["batch"], crop=case["crop"], lr=1e-3, seed=state["seed"])
    return {"losses": losses, "params": r.denoiser_params()}


# ---------------------------------------------------------------- what it cannot do without
_FLOP_PER_BOX, _FLOP_PER_TRI, _FLOP_PER_VERTEX = 18, 60, 600


def _tris(case):
    return {"cornell": 36, "soup": case["size"], "instanced": 20 * 4 ** (5 if case["size"] >= 1000 else 4)}[case["scene"]]


def _scene_bytes(case):
    """Corners and material of every triangle, 44 B of transform and ids per instance."""
    mats = {"cornell": 5, "soup": case["size"], "instanced": 11 * case["size"]}[case["scene"]]
    return 40 * _tris(case) + 80 * mats + (56 * case["size"] if case["scene"] == "instanced" else 0)


def _ray_flops(case):
    """Two boxes per level of a binary tree down to one triangle."""
    leaves = _tris(case) * (case["size"] if case["scene"] == "instanced" else 1)
    return 2 * _FLOP_PER_BOX * max(1.0, math.log2(leaves)) + _FLOP_PER_TRI


# multiply-adds per full-resolution pixel of the U-Net's fifteen 3 x 3 convolutions: channels
# in, out, and the side's divisor
_CONVS = [(16, 32, 1), (32, 32, 1), (32, 64, 2), (64, 64, 2), (64, 96, 4), (96, 96, 4), (96, 128, 8), (128, 128, 8),
          (224, 96, 4), (96, 96, 4), (160, 64, 2), (64, 64, 2), (96, 32, 1), (32, 32, 1), (32, 3, 1)]
_NET_FLOPS = sum(2 * 9 * ci * co / (dv * dv) for ci, co, dv in _CONVS)
_NET_PARAMS = sum(9 * ci * co + co for ci, co, _ in _CONVS)


def work(case):
    """Inputs once, outputs once; the arithmetic of the algorithm as it stands: for a traced
    ray the boxes of one root-to-leaf walk and a triangle, for a vertex its shading (and in
    a gradient its derivative), for the network its convolutions."""
    if case["kind"] == "rays":
        out = 1 if case["query"] == "any" else 20
        return {"bytes": case["rays"] * (32 + out) + _scene_bytes(case), "flops": case["rays"] * _ray_flops(case)}
    if case["kind"] == "frames":
        pix = case["width"] * case["height"]
        paths = pix * case["spp"] * case["frames"]
        debug = case["mode"] != "path_tracing"
        vertices = 1.0 if debug else 0.4 * case["depth"]
        per = 2 * _ray_flops(case) + (50 if debug else _FLOP_PER_VERTEX)
        return {"bytes": _scene_bytes(case) + pix * (4 if case["show"] else 16), "flops": paths * vertices * per}
    if case["kind"] == "gradient":
        pix = case["width"] * case["height"]
        vertices = pix * case["spp"] * 0.6 * case["depth"]
        return {"bytes": _scene_bytes(case) + pix * (16 + 12) + case["size"] * 20 * 2,
                "flops": vertices * (4 * _ray_flops(case) + 4 * _FLOP_PER_VERTEX)}
    if case["kind"] == "denoise":
        pix = case["width"] * case["height"]
        return {"bytes": pix * (3 * 16 + 16) + 2 * _NET_PARAMS, "flops": pix * _NET_FLOPS}
    pix = case["batch"] * case["crop"] ** 2 * case["steps"]
    return {"bytes": pix * (32 + 12) + case["steps"] * _NET_PARAMS * 4 * 7, "flops": 3 * pix * _NET_FLOPS}


# ------------------------------------------------------------------------- 64-bit answers
def exact(case, seed):
    """Closest hits of free rays by testing every triangle (Moeller-Trumbore, 64 bits), on
    the scene that is small enough for it."""
    if case["kind"] != "rays" or case["query"] != "closest" or case["scene"] != "cornell" or case["rays"] > 400_000:
        return None
    sc, rays = _rays(case, seed)
    tri = sc["positions"].astype(np.float64).reshape(-1, 3, 3)
    rays = rays.astype(np.float64)
    out = np.zeros((len(rays), 3))
    for a in range(0, len(rays), 1 << 16):
        o, tmin, d, tmax = (rays[a:a + (1 << 16), s] for s in (slice(0, 3), 3, slice(4, 7), 7))
        best = tmax.copy()
        bary = np.zeros((len(o), 2))
        for v0, v1, v2 in tri:
            e1, e2 = v1 - v0, v2 - v0
            p = np.cross(d, e2)
            det = p @ e1
            with np.errstate(divide="ignore", invalid="ignore"):
                s = o - v0
                u = (p * s).sum(1) / det
                q = np.cross(s, e1)
                v = (q * d).sum(1) / det
                t = (q @ e2) / det
                hit = (u >= 0) & (v >= 0) & (u + v <= 1) & (t >= tmin) & (t < best)
            best[hit] = t[hit]
            bary[hit, 0], bary[hit, 1] = u[hit], v[hit]
        out[a:a + (1 << 16), 0] = best
        out[a:a + (1 << 16), 1:] = bary
    return {"t_b1_b2": out, "prim": None, "inst": None}
