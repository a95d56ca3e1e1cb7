"""The logits of the last forward pass on demand: no memory of their own, a buffer of any float alignment, and a buffer
of more or fewer pixels than the pass had."""
import ctypes

import pytest

from test_gpu_kpn_net import _inputs, _random_params

pytestmark = pytest.mark.gpu


def test_forward_pass_keeps_no_logits(vpt):
    print("case: kpn memory of a forward pass", flush=True)
    import torch

    from cloudrendering_amd import kpn
    from cloudrendering_amd._lib import call

    call("crvpt_kpn_release")
    net = kpn.KpnDenoiser(parameters=_random_params(3))
    small = _inputs(4, 1, 16, 16)
    net.denoise(small[0], small[1])
    net.logits(1, 16, 16)  # loads the kernels
    feats = torch.rand((1, 15, 1024, 1024), device="cuda")
    noisy = torch.rand((1, 3, 1024, 1024), device="cuda")
    out = torch.empty((1, 1024, 1024, 32), device="cuda")
    net.denoise(feats[:, :, :16, :16].contiguous(), noisy[:, :, :16, :16].contiguous())
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    free = torch.cuda.mem_get_info()[0]
    net.denoise(feats, noisy)
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    # six layers' inputs and two gradients of 32 bf16 channels: 512 bytes a pixel
    used = free - torch.cuda.mem_get_info()[0]
    assert used <= 560 << 20, f"{used >> 20} MiB"
    call("crvpt_kpn_get_logits", ctypes.c_void_p(out.data_ptr()), 1, 1024, 1024, None)
    torch.cuda.synchronize()
    assert free - torch.cuda.mem_get_info()[0] <= used
    call("crvpt_kpn_release")


def test_logits_buffers(vpt):
    print("case: kpn logits buffers", flush=True)
    import torch

    from cloudrendering_amd import kpn
    from cloudrendering_amd._lib import call

    call("crvpt_kpn_release")
    net = kpn.KpnDenoiser(parameters=_random_params(5))
    big, small = _inputs(6, 1, 40, 50), _inputs(7, 2, 17, 19)
    net.denoise(big[0], big[1])
    net.denoise(small[0], small[1])
    want = net.logits(2, 17, 19).reshape(-1)
    n = want.numel()
    for pixels in (2 * 17 * 19, 5, 331, 2000):  # the pass', fewer, and as many as an earlier pass
        for offset in (0, 1, 3):
            buf = torch.full((pixels * 32 + 8,), 7.0, device="cuda")
            call("crvpt_kpn_get_logits", ctypes.c_void_p(buf.data_ptr() + 4 * offset), 1, 1, pixels, None)
            torch.cuda.synchronize()
            got = buf[offset:offset + pixels * 32]
            k = min(n, pixels * 32)
            assert torch.equal(got[:k], want[:k])
            assert bool((got[k:] == 0.0).all())
            assert bool((buf[:offset] == 7.0).all()) and bool((buf[offset + pixels * 32:] == 7.0).all())
    with pytest.raises(vpt.CrvptError):
        net.logits(1, 1, 2001)
