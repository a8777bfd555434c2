"""Large reads (threads and pinned chunks) against small ones (the runtime's own copy)."""
import numpy as np
import pytest

from trayracer_amd import Renderer, scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("width,height", [(511, 512), (512, 512), (1023, 769), (1920, 1080)])
def test_pixels_round_trip(width, height):
    """An accumulator written and read back whole, at sizes around the first threaded read
    (4 MiB), with a last chunk that is not full, and with every thread reading several
    chunks."""
    rng = np.random.default_rng(width)
    r = Renderer(0)
    try:
        r.UpdateScene(scenes.cornell(width=16, height=16, spp=1))
        acc = rng.random((height, width, 4), np.float32)
        acc[..., 3] = 8.0
        r.write_accum(acc)
        r.settings.width, r.settings.height = width, height
        for _ in range(3):
            assert np.array_equal(r.accum().view(np.uint32), acc.view(np.uint32))
        col = acc * np.float32(1.0 / 8.0)
        col[..., 3] = 1.0
        assert np.array_equal(r.color().view(np.uint32), col.view(np.uint32))
        img = r.tonemap("none", exposure=1.0, gamma=1.0)
        assert img.shape == (height, width, 4) and (img[..., 3] == 255).all()
    finally:
        r.close()


def test_bytes_round_trip():
    """4 MiB + 5 occlusion bytes (a last part whose length is no multiple of 16) against the
    same rays asked in two calls below the threaded reads."""
    from tests.gpu_util import random_rays
    n = (4 << 20) + 5
    rays = random_rays(n, seed=3, lo=0.02, hi=0.98)
    rays[:, 7] = 0.6
    r = Renderer(0)
    try:
        r.UpdateScene(scenes.cornell(width=16, height=16, spp=1))
        whole = r.trace_any(rays)
        parts = np.concatenate([r.trace_any(rays[:n // 2]), r.trace_any(rays[n // 2:])])
    finally:
        r.close()
    assert 0.1 < parts.mean() < 0.9
    assert np.array_equal(whole, parts)
