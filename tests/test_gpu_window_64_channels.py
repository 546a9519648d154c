"""Convolutions over windows with 33 to 64 output channels: a wave takes all of them from 4096 pieces of 32 pixels x 32 channels on (2048
with exactly 64), pixels and channels that fill no tile, either side of the switches, every epilogue, slices."""
import numpy as np
import pytest
import torch
import torch.nn.functional as F

import dabnn_amd as dab
from dabnn_amd import capi, models

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,h,w,cin,cout,k,stride,pad", [
    (1, 256, 128, 192, 64, 3, 1, 1), (1, 255, 128, 192, 64, 3, 1, 1), (2, 255, 128, 64, 40, 5, 1, 2), (1, 255, 256, 64, 33, 1, 1, 0),
    (3, 157, 139, 320, 56, 3, 1, 1), (1, 256, 256, 128, 64, 5, 2, 2), (33, 45, 47, 128, 64, 1, 1, 0), (1, 256, 256, 192, 65, 3, 1, 1),
    # 150 to 250 words a filter, of which 64 do not fit: the depth split from 4096 pieces on, but 32 channels a wave in chunks of one word or
    # two from 8000 on (with up to 40 channels from 20 000); 108 and 144 words, which fit
    (5, 128, 128, 320, 64, 6, 1, 3), (8, 128, 128, 320, 64, 6, 1, 3), (8, 128, 128, 320, 40, 6, 1, 3), (20, 128, 128, 640, 40, 4, 1, 2),
    (5, 128, 128, 384, 56, 5, 1, 2), (9, 128, 128, 512, 33, 5, 1, 2), (6, 128, 128, 640, 64, 5, 1, 2), (8, 128, 128, 576, 64, 4, 1, 2),
    (4, 128, 128, 768, 48, 3, 1, 1),
])
@pytest.mark.parametrize("epilogue", ["counts", "affine", "sign"])
def test_windows(n, h, w, cin, cout, k, stride, pad, epilogue):
    if epilogue == "sign" and cout % 64 != 0:
        cout = 64
    g = torch.Generator(device="cuda").manual_seed(cin + cout)
    x = torch.randn(n, h, w, cin, device="cuda", generator=g)
    wf = np.random.default_rng(cout).standard_normal((cout, k, k, cin)).astype(np.float32)
    wp = torch.from_numpy(models.pack_weight(wf).view(np.int64)).cuda()
    packed = dab.pack_mat(x)
    cw = cin // 64
    # the input as words 1 .. of pixels of cw + 2, the output as channels 5 .. of cout + 9
    wide = torch.randint(-2**62, 2**62, (n, h, w, cw + 2), dtype=torch.int64, device="cuda", generator=g)
    wide[..., 1:1 + cw] = packed
    oh, ow = (h + 2 * pad - k) // stride + 1, (w + 2 * pad - k) // stride + 1
    out = torch.full((n, oh, ow, cout + 9), -3.0, device="cuda")
    bits = torch.full((n, oh, ow, 3), -1, dtype=torch.int64, device="cuda")
    a, b = torch.randn(cout, device="cuda", generator=g), torch.randn(cout, device="cuda", generator=g) * 50
    with_a, with_bits = epilogue != "counts", epilogue == "sign"
    capi.check(capi.lib.dab_bconv(wide.data_ptr() + 8, cw + 2, n, h, w, cin, wp.data_ptr(), wp.shape[1], k, k, pad, pad, stride, stride, cout,
                                  a.data_ptr() if with_a else None, b.data_ptr() if with_a else None, None, out.data_ptr() + 20, cout + 9,
                                  bits.data_ptr() + 8 if with_bits else None, 3 if with_bits else 0, torch.cuda.current_stream().cuda_stream))
    s = F.pad(torch.where(x > 0, 1.0, -1.0).permute(0, 3, 1, 2), (pad, pad, pad, pad), value=-1.0).cpu()
    few = slice(0, 1)
    want = ((k * k * cin - F.conv2d(s[few], torch.where(torch.from_numpy(wf) > 0, 1.0, -1.0).permute(0, 3, 1, 2), stride=stride)) / 2).permute(0, 2, 3, 1)
    if with_a:
        want = want * a.cpu() + b.cpu()
    got = out[..., 5:5 + cout]
    assert torch.equal(got[few].cpu(), want)
    assert bool((out[..., :5] == -3).all()) and bool((out[..., 5 + cout:] == -3).all())
    if with_bits:
        assert torch.equal(bits[..., 1:1 + cout // 64], dab.pack_mat(got.contiguous()))
        assert bool((bits[..., 0] == -1).all()) and bool((bits[..., 1 + cout // 64:] == -1).all())
    else:
        # the other images as the first would be in their place
        one = torch.full_like(out[:1], -3.0)
        last = wide[-1:].contiguous()
        capi.check(capi.lib.dab_bconv(last.data_ptr() + 8, cw + 2, 1, h, w, cin, wp.data_ptr(), wp.shape[1], k, k, pad, pad, stride, stride, cout,
                                      a.data_ptr() if with_a else None, b.data_ptr() if with_a else None, None, one.data_ptr() + 20, cout + 9, None, 0,
                                      torch.cuda.current_stream().cuda_stream))
        assert torch.equal(one, out[-1:])
