"""BinConv layers from fp32 input: problems that pack and convolve in one launch and those either side of its edges (strip heights,
1 to 8 waves a tile, ragged strips and tiles, channels that fill no group of 64, strides, padding beyond the image, the filters'
padding word, pixels of exactly zero, NaN, outputs of one pixel)."""
import numpy as np
import pytest
import torch
import torch.nn.functional as F

import dabnn_amd as dab
from dabnn_amd import models

pytestmark = pytest.mark.gpu


def reference(x, wf, strides, pads):
    s = torch.where(x > 0, 1.0, -1.0).double().permute(0, 3, 1, 2)  # a NaN is no positive number
    s = F.pad(s, (pads[1], pads[1], pads[0], pads[0]), value=-1.0)
    w = torch.where(torch.from_numpy(wf) > 0, 1.0, -1.0).double().permute(0, 3, 1, 2)
    k = wf[0].size
    return ((k - F.conv2d(s, w, stride=strides)) / 2).permute(0, 2, 3, 1).float()


@pytest.mark.parametrize("n,h,w,cin,cout,k,strides,pads", [
    (1, 3, 3, 64, 8, (3, 3), (1, 1), (0, 0)), (1, 1, 1, 64, 1, (1, 1), (1, 1), (0, 0)), (2, 5, 8, 320, 32, (1, 1), (1, 1), (0, 0)),
    (3, 6, 8, 64, 40, (3, 3), (1, 1), (1, 1)), (16, 56, 56, 64, 64, (3, 3), (1, 1), (1, 1)), (8, 14, 14, 256, 256, (5, 5), (1, 1), (2, 2)),
    (2, 14, 13, 256, 72, (3, 3), (2, 2), (1, 1)), (24, 17, 17, 64, 56, (3, 3), (1, 1), (1, 1)), (1, 33, 31, 128, 65, (5, 5), (2, 2), (2, 2)),
    (2, 9, 11, 192, 136, (3, 3), (1, 1), (1, 1)), (1, 7, 7, 448, 8, (3, 3), (1, 1), (1, 1)), (1, 9, 9, 512, 120, (3, 3), (2, 2), (1, 1)),
    (2, 4, 40, 64, 24, (1, 7), (1, 2), (0, 3)), (2, 40, 4, 128, 24, (7, 2), (3, 1), (3, 1)), (1, 4, 5, 64, 16, (3, 3), (1, 1), (4, 3)),
    (307, 7, 6, 64, 16, (1, 1), (1, 1), (0, 0)), (37, 10, 10, 64, 64, (3, 3), (1, 1), (1, 1)), (1, 60, 130, 64, 16, (3, 3), (1, 1), (1, 1)),
    (1, 12, 12, 1024, 16, (3, 3), (1, 1), (1, 1)), (2, 6, 6, 128, 64, (1, 1), (4, 3), (0, 0)), (1, 3, 70, 64, 64, (3, 3), (1, 1), (0, 0)),
])
def test_counts(n, h, w, cin, cout, k, strides, pads):
    r = np.random.default_rng(n + h + cin + cout)
    wf = r.standard_normal((cout, *k, cin)).astype(np.float32)
    x = r.standard_normal((n, h, w, cin)).astype(np.float32)
    x.reshape(-1)[:: 7] = 0.0
    x.reshape(-1)[3 :: 101] = np.nan
    x = torch.from_numpy(x)
    layer = dab.BinConv(torch.from_numpy(models.pack_weight(wf).view(np.int64)).cuda(), *k, *pads, *strides)
    oh, ow = (h + 2 * pads[0] - k[0]) // strides[0] + 1, (w + 2 * pads[1] - k[1]) // strides[1] + 1
    want = reference(x, wf, strides, pads)
    assert want.shape == (n, oh, ow, cout)
    xd = x.cuda()
    assert torch.equal(layer(xd).cpu(), want)
    # input that starts off the 16-byte grid, the same problem inside a batch that takes the other way
    off = torch.empty(x.numel() + 1, device="cuda")[1:].view(x.shape).copy_(xd)
    assert torch.equal(layer(off).cpu(), want)
    if n * h * w * cin < 300000:
        many = layer(xd.repeat(200, 1, 1, 1))
        assert torch.equal(many[:n].cpu(), want) and torch.equal(many[-n:], many[:n])


@pytest.mark.parametrize("cin,cout,k", [(64, 48, 3), (192, 200, 1), (256, 72, 5)])
def test_nothing_is_stored_past_the_output(cin, cout, k):
    from dabnn_amd import capi
    r = np.random.default_rng(cin)
    n, h, w = 2, 9, 11
    wf = r.standard_normal((cout, k, k, cin)).astype(np.float32)
    weight = torch.from_numpy(models.pack_weight(wf).view(np.int64)).cuda()
    x = torch.from_numpy(r.standard_normal((n, h, w, cin)).astype(np.float32)).cuda()
    guard = 4096
    out = torch.full((n * h * w * cout + 2 * guard,), -7.0, device="cuda")
    need = capi.lib.dab_binconv_workspace_bytes(n, h, w, cin, k, k, k // 2, k // 2, 1, 1)
    ws = torch.empty(need, dtype=torch.uint8, device="cuda")
    wt = dab.weight_transpose(weight)
    capi.check(capi.lib.dab_binconv_forward(x.data_ptr(), n, h, w, cin, weight.data_ptr(), wt.data_ptr(), weight.shape[1], k, k, k // 2, k // 2, 1, 1, cout,
                                            out.data_ptr() + 4 * guard, ws.data_ptr(), need, None, torch.cuda.current_stream().cuda_stream))
    assert bool((out[:guard] == -7).all()) and bool((out[-guard:] == -7).all())
    assert torch.equal(out[guard:-guard].view(n, h, w, cout).cpu(), reference(x.cpu(), wf, (1, 1), (k // 2, k // 2)))


# a layer run in place, and into buffers that begin before its input's end or end behind its start (counted in output elements from x)
@pytest.mark.parametrize("n,h,w,c,k", [(2, 12, 12, 64, 3), (16, 56, 56, 64, 3), (3, 20, 21, 128, 1), (2, 14, 14, 192, 3), (1, 9, 9, 256, 5)])
@pytest.mark.parametrize("where", [0.0, 0.5, -0.75])
def test_output_over_input(n, h, w, c, k, where):
    from dabnn_amd import capi
    r = np.random.default_rng(c + k)
    weight = torch.from_numpy(models.pack_weight(r.standard_normal((c, k, k, c)).astype(np.float32)).view(np.int64)).cuda()
    x = torch.randn((n, h, w, c), device="cuda", generator=torch.Generator(device="cuda").manual_seed(n + c))
    want = dab.BinConv(weight, k, k, k // 2, k // 2, 1, 1)(x)
    size = x.numel()
    buf = torch.empty(3 * size, device="cuda")
    buf[size:2 * size] = x.view(-1)
    at = size + int(where * size) // 4 * 4
    need = capi.lib.dab_binconv_workspace_bytes(n, h, w, c, k, k, k // 2, k // 2, 1, 1)
    ws = torch.empty(need, dtype=torch.uint8, device="cuda")
    wt = dab.weight_transpose(weight)
    capi.check(capi.lib.dab_binconv_forward(buf.data_ptr() + 4 * size, n, h, w, c, weight.data_ptr(), wt.data_ptr(), weight.shape[1], k, k, k // 2, k // 2, 1, 1, c,
                                            buf.data_ptr() + 4 * at, ws.data_ptr(), need, None, torch.cuda.current_stream().cuda_stream))
    assert torch.equal(buf[at:at + size].view_as(want), want)


# windows larger than the padded image, whose output is rounded up to one pixel: those rows and columns are padding
@pytest.mark.parametrize("h,w,c,k,stride", [(9, 3, 64, (3, 5), (1, 3)), (3, 9, 128, (5, 3), (4, 1)), (6, 2, 192, (1, 4), (2, 4)), (2, 2, 64, (3, 3), (3, 2))])
def test_windows_larger_than_the_image(h, w, c, k, stride):
    from dabnn_amd import capi
    r = np.random.default_rng(h)
    cout, n = 40, 3
    wf = r.standard_normal((cout, *k, c)).astype(np.float32)
    weight = torch.from_numpy(models.pack_weight(wf).view(np.int64)).cuda()
    x = torch.from_numpy(r.standard_normal((n, h, w, c)).astype(np.float32)).cuda()
    oh, ow = (int((s - f) / t) + 1 for s, f, t in zip((h, w), k, stride))
    want = reference(F.pad(x, (0, 0, 0, k[1], 0, k[0]), value=-1.0).cpu(), wf, stride, (0, 0))[:, :oh, :ow]
    need = capi.lib.dab_binconv_workspace_bytes(n, h, w, c, *k, 0, 0, *stride)
    ws, wt, out = torch.empty(need, dtype=torch.uint8, device="cuda"), dab.weight_transpose(weight), torch.empty((n, oh, ow, cout), device="cuda")
    # (strides that differ make the 3x3 case the general route's)
    capi.check(capi.lib.dab_binconv_forward(x.data_ptr(), n, h, w, c, weight.data_ptr(), wt.data_ptr(), weight.shape[1], *k, 0, 0, *stride, cout,
                                            out.data_ptr(), ws.data_ptr(), need, None, torch.cuda.current_stream().cuda_stream))
    assert torch.equal(out.cpu(), want)
