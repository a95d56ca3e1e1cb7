"""SVGF at image sizes around its 16x16 tiles, over enough frames that the moments filter passes from its short-history
taps to the copy, against the NumPy restatement (oracle/denoise_ref.py) fed with the same feature maps. Tolerance of
test_gpu_denoise: the normal weight max(0, n.n')^128 multiplies the rounding of its input 128-fold (2e-3 relative)."""
import numpy as np
import pytest

from oracle import denoise_ref as D
from test_gpu_denoise import _hwc, _scene

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("h,w", [(1, 1), (3, 5), (16, 16), (17, 33), (40, 15)])
def test_svgf_tile_edges(vpt, oracle, h, w):
    print(f"case: SVGF {h}x{w}, 6 frames", flush=True)
    import torch

    _scene(vpt, oracle)
    vpt.set_denoiser("SVGF")
    s = D.Svgf(h, w)
    t = torch.zeros((4, h, w), dtype=torch.float32, device="cuda")
    try:
        for frame in range(6):
            out = _hwc(vpt.render_frame(t, 1))
            m = {n: _hwc(vpt.get_feature_map_from_string(t, n))
                 for n in ["Result", "Flow", "Normal", "Depth", "Depth (fwidth)"]}
            ref = s.denoise(m["Result"], m["Flow"][..., :2], m["Normal"], m["Depth"][..., 0],
                            m["Depth (fwidth)"][..., 0])
            np.testing.assert_allclose(out[..., :3], ref[..., :3], rtol=2e-3, atol=2e-5, err_msg=f"frame {frame}")
    finally:
        vpt.set_denoiser("None")
