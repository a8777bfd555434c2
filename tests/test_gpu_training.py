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


@pytest.mark.parametrize("N,H,W", [(4, 256, 256), (2, 128, 128), (3, 88, 128)],
                         ids=["16-row-tiles", "32-chunks", "33-chunks"])
def test_batch_gradient_is_the_sum_over_its_images(N, H, W):
    """Gradients of a batch against the sum of its images' own, which take other routes: the
    batch of 262144 pixels convolves 16-row tiles in launches of their own and its images
    8-row tiles beside the weight gradient; 32 partial sums are added in registers, 33 in LDS.
    The terms are the same bits (the forward outputs are checked to be), only the order of
    their fp32 additions differs: chains of at most 2^14 additions of terms of either sign
    round by about sqrt(2^14) 2^-24 = 7.6e-6 of a sum; 1e-4 in relative norm per parameter
    block."""
    from oracle import unet_ref as U
    rng = np.random.default_rng(N * H)
    rend = Renderer(0)
    try:
        rend.denoiser_set_params(U.init_params(17))
        feats = np.zeros((N, H, W, 16), np.float32)
        feats[..., :10] = rng.normal(0.5, 0.5, (N, H, W, 10))
        dout = rng.normal(size=(N, H, W, 32)).astype(np.float32)
        dout[..., 3:] = 0
        out = rend.denoiser_forward(feats)
        g = rend.denoiser_backward(dout).astype(np.float64)
        total = np.zeros_like(g)
        for n in range(N):
            one = rend.denoiser_forward(feats[n:n + 1])
            assert np.array_equal(np.asarray(one)[0].view(np.uint32), np.asarray(out)[n].view(np.uint32))
            total += rend.denoiser_backward(dout[n:n + 1])
    finally:
        rend.close()
    at = 0
    for ci, co, _ in U.SPEC:
        for n in (co * 9 * ci, co):
            a, b = g[at:at + n], total[at:at + n]
            at += n
            assert np.linalg.norm(a - b) <= 1e-4 * np.linalg.norm(b)
