"""The denoiser network on images whose tensors pass 2^31 bytes."""
import numpy as np
import pytest

from trayracer_amd import Renderer

pytestmark = pytest.mark.gpu


def test_corners_of_a_large_image():
    """8192 x 4104 pixels, empty but for the first and the last corner, against a small image
    with the same corners. The network sees at most 64 pixels far, so the outputs there are the
    same bits, and the parameter gradients of a gradient there have the same terms, which only
    their fp32 sums' order tells apart (at most 2^14 non-zero terms of either sign: sqrt(2^14)
    2^-24 = 7.6e-6 of a sum; 1e-4 in relative norm per parameter block)."""
    from oracle import unet_ref as U
    rng = np.random.default_rng(3)
    ch, cw = 64, 128
    first, last = (rng.normal(0.5, 0.5, (ch, cw, 10)).astype(np.float32) for _ in range(2))
    d_first, d_last = (rng.normal(size=(ch, cw, 3)).astype(np.float32) for _ in range(2))
    res = {}
    rend = Renderer(0)
    try:
        rend.denoiser_set_params(U.init_params(17))
        for H, W in ((256, 512), (4104, 8192)):
            feats = np.zeros((1, H, W, 16), np.float32)
            feats[0, :ch, :cw, :10], feats[0, -ch:, -cw:, :10] = first, last
            out = rend.denoiser_forward(feats)
            corners = out[0, :ch, :cw].copy(), out[0, -ch:, -cw:].copy()
            del feats, out
            dout = np.zeros((1, H, W, 32), np.float32)
            dout[0, :ch, :cw, :3], dout[0, -ch:, -cw:, :3] = d_first, d_last
            res[H] = corners, rend.denoiser_backward(dout).astype(np.float64)
            del dout
    finally:
        rend.close()
    (small, gs), (large, gl) = res[256], res[4104]
    for a, b in zip(small, large):
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
    at = 0
    for ci, co, _ in U.SPEC:
        for n in (co * 9 * ci, co):
            a, b = gl[at:at + n], gs[at:at + n]
            at += n
            assert np.linalg.norm(b) > 0 and np.linalg.norm(a - b) <= 1e-4 * np.linalg.norm(b)
