"""Denoiser training kernels at the edges of their tiles, against the FP64 network."""
import numpy as np
import pytest

from trayracer_amd import Renderer

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,H,W", [(1, 24, 128), (3, 8, 128)], ids=["3-row-coarsest", "1-row-coarsest"])
def test_backward_at_ragged_levels(N, H, W):
    """Weight and bias gradients where the levels' heights leave 8-row tiles part empty and
    chunks of eight tiles cross images (24, 12, 6, 3 rows; 8, 4, 2, 1). The reference applies
    the same bf16 roundings to the device's own activations; what is left is the rounding of
    each layer's incoming gradient to bf16 (2^-9 relative, at most 15 layers deep, partly
    averaging out): sqrt(15) 2^-9 = 7.6e-3, below 1e-2 in relative norm."""
    from oracle import unet_ref as U
    rng = np.random.default_rng(5)
    params = U.init_params(13)
    rend = Renderer(0)
    try:
        rend.denoiser_set_params(params)
        feats = np.zeros((N, H, W, 16), np.float32)
        feats[..., :10] = rng.normal(0.5, 0.5, (N, H, W, 10))
        rend.denoiser_forward(feats)
        levels = [1, 1, 2, 2, 4, 4, 8, 8, 4, 4, 2, 2, 1, 1]
        acts = {i: rend.denoiser_activation(i, (N, H // levels[i], W // levels[i], U.SPEC[i][1])) for i in range(14)}
        dout = rng.normal(size=(N, H, W, 32)).astype(np.float32)
        dout[..., 3:] = 0
        g = rend.denoiser_backward(dout)
        g2 = rend.denoiser_backward(dout)
    finally:
        rend.close()
    assert np.array_equal(g.view(np.uint32), g2.view(np.uint32))
    ref = U.UnetRef(params, round_bf16=True)
    ref.forward(feats)
    ref.use_activations(feats, acts)
    gr = ref.backward(dout.astype(np.float64))
    at = 0
    for ci, co, _ in U.SPEC:
        for n in (co * 9 * ci, co):
            a, b = g[at:at + n], gr[at:at + n]
            at += n
            assert np.linalg.norm(a - b) <= 1e-2 * np.linalg.norm(b)
