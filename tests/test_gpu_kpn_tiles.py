"""GPU tests of the denoiser network's kernels at the edges of their 16x16 tiles and of the tile walk over the XCDs:
single pixels, one tile, one pixel over a tile, fewer tiles than XCDs, and a batch whose tiles do not divide evenly,
against the float32 torch reference of test_gpu_kpn_net with its bf16 rounding points.

Tolerances: the logits differ by FP32 summation order and the bf16 flips that follow from it (2^-9 per layer at most:
1 % of the norm over six layers), gradients also by the bf16 storage of the backward activations (2^-9 relative each,
over up to five layers and with few pixels to average: 5 % of the norm).
"""
import numpy as np
import pytest

from test_gpu_kpn_net import _inputs, _random_params, _reference

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1, 1), (1, 15, 17), (1, 16, 16), (1, 17, 33), (3, 33, 47), (2, 5, 130), (9, 16, 48)]


def _rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


@pytest.mark.parametrize("shape", SHAPES)
def test_tile_edges(vpt, shape):
    print(f"case: kpn tiles {shape}", flush=True)
    import torch

    from cloudrendering_amd import kpn

    n, h, w = shape
    params = _random_params(11)
    net = kpn.KpnDenoiser(parameters=params)
    feats, noisy, target = _inputs(12, n, h, w)
    out = net.denoise(feats, noisy)
    logits = net.logits(n, h, w).permute(0, 3, 1, 2)
    ref_logits, _, ref_loss, ws, bs = _reference(params, feats, noisy, target)
    assert _rel(logits.cpu().numpy(), ref_logits.detach().cpu().numpy()) < 1e-2
    taps = torch.nn.functional.unfold(noisy, 5, padding=2).view(n, 3, 25, h, w)
    pred = (taps * torch.softmax(logits[:, :25], 1).unsqueeze(1)).sum(2)
    np.testing.assert_allclose(out.cpu().numpy(), pred.cpu().numpy(), rtol=1e-5, atol=1e-6)
    loss = net.compute_gradients(feats, noisy, target)
    gw, gb = kpn.KpnDenoiser.split(net.gradients())
    ref_loss.backward()
    assert abs(loss - ref_loss.item()) <= 2e-3 * abs(ref_loss.item())
    for layer in range(6):
        assert _rel(gw[layer], ws[layer].grad.cpu().numpy()) < 5e-2
        assert _rel(gb[layer], bs[layer].grad.cpu().numpy()) < 5e-2
