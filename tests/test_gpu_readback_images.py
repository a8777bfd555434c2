"""Threaded reads of what was queued just before them: whole tonemapped images against the host
transform, other data in every call."""
import numpy as np
import pytest

from trayracer_amd import Renderer, scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("width,height", [(1023, 1027), (1920, 1080)])
def test_tonemapped_images(width, height):
    """4.2 and 8.3 MB of RGBA8 through the pinned chunks, whose source the tonemap kernel has
    just been queued to write; then the float image, and both again with other pixels, so that a
    chunk read too early, left from the last call or misplaced shows."""
    from oracle.oracle_py import tonemap
    rng = np.random.default_rng(width)
    r = Renderer(0)
    try:
        r.UpdateScene(scenes.cornell(width=16, height=16, spp=1))
        r.settings.width, r.settings.height = width, height
        for turn in range(4):
            acc = (rng.random((height, width, 4), np.float32) * np.float32(2 + turn)).astype(np.float32)
            acc[..., 3] = 4.0
            r.write_accum(acc)
            method, gamma = ((0, 2.2), (3, 1.0), (7, 2.0), (0, 1.8))[turn]
            got = r.tonemap(method, 1.0, gamma)
            col = r.color()
            want = acc * np.float32(0.25)
            want[..., 3] = 1.0
            assert np.array_equal(col.view(np.uint32), want.view(np.uint32))
            assert np.array_equal(got, tonemap(want, method, 1.0, gamma))
    finally:
        r.close()
