"""3x3 float convolutions over three-channel images to up to 64 channels: both sides of the sizes at which they leave the tile kernels, last tiles that are
not full, strides, dilations and pads, channel counts that fill no 32, PRelu with slices and sign bits, infinities and NaNs."""
import ctypes

import pytest
import torch

import dabnn_amd as dab
from dabnn_amd import capi

pytestmark = pytest.mark.gpu


def stream():
    return ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)


def p(t):
    return None if t is None else t.data_ptr()


def reference(x, w, bias, a, b, stride, pad, dil):
    """In 64 bits, and the sum of magnitudes that bounds the rounding errors."""
    conv = lambda u, v: torch.nn.functional.conv2d(u.permute(0, 3, 1, 2).double().cpu(), v.permute(0, 3, 1, 2).double().cpu(), stride=stride, padding=pad,
                                                   dilation=dil).permute(0, 2, 3, 1).cuda()
    v, size = conv(x, w), conv(x.abs(), w.abs())
    if bias is not None:
        v, size = v + bias.double(), size + bias.double().abs()
    if a is not None:
        v, size = v * a.double() + b.double(), size * a.double().abs() + b.double().abs()
    return v, size


@pytest.mark.parametrize("n,h,w,cout,stride,pad,dil,act", [
    (1, 90, 91, 32, 1, 1, 1, "relu"), (1, 91, 91, 32, 1, 1, 1, ""), (1, 100, 99, 64, 1, 1, 1, "prelu"), (1, 100, 100, 64, 1, 1, 1, "prelu"), (1, 100, 101, 64, 1, 1, 1, "relu"),
    (2, 224, 224, 32, 2, 1, 1, "relu"), (7, 61, 83, 1, 1, 0, 1, ""), (3, 120, 75, 33, 1, 2, 2, "relu"), (5, 97, 65, 48, 1, 3, 1, "prelu1"), (9, 130, 64, 17, 2, 1, 3, "relu"),
    (70, 32, 32, 64, 1, 1, 1, "prelu"), (2000, 3, 3, 64, 1, 1, 1, "prelu1"), (30000, 1, 1, 8, 1, 1, 1, "relu"), (80, 112, 112, 32, 1, 1, 1, "relu")])
def test_against_64_bits(n, h, w, cout, stride, pad, dil, act):
    g = torch.Generator(device="cuda").manual_seed(n + h + cout)
    x, wt = torch.randn((n, h, w, 3), device="cuda", generator=g), torch.randn((cout, 3, 3, 3), device="cuda", generator=g) / 5
    bias = torch.randn(cout, device="cuda", generator=g) if cout % 2 else None
    a, b = (torch.randn(cout, device="cuda", generator=g) for _ in range(2)) if cout % 3 else (None, None)
    oh, ow = (h + 2 * pad - 2 * dil - 1) // stride + 1, (w + 2 * pad - 2 * dil - 1) // stride + 1
    want, size = reference(x, wt, bias, a, b, stride, pad, dil)
    ld = cout + 64 if act.startswith("prelu") else cout
    out = torch.full((n, oh, ow, ld), 9.0, device="cuda")
    bits = None
    if act.startswith("prelu"):
        slope = torch.rand(1 if act == "prelu1" else cout, device="cuda", generator=g)
        if cout % 64 == 0:
            bits = torch.zeros((n, oh, ow, cout // 64 + 1), dtype=torch.int64, device="cuda")
        rc = capi.lib.dab_fconv_affine_prelu(p(x), n, h, w, 3, p(wt), p(bias), p(a), p(b), p(slope), slope.numel(), 3, 3, pad, pad, stride, stride, dil, dil, cout, p(out), ld,
                                             p(bits), 0 if bits is None else bits.shape[-1], stream())
        want = torch.where(want < 0, want * slope.double(), want)
    else:
        rc = capi.lib.dab_fconv_affine_relu(p(x), n, h, w, 3, p(wt), p(bias), p(a), p(b), int(act == "relu"), 3, 3, pad, pad, stride, stride, dil, dil, cout, p(out), stream())
        want = torch.where(want < 0, 0 * want, want) if act == "relu" else want
    assert rc == 0, capi.last_error()
    # 27 products in sums of fewer than 27, three operations behind them, a product with the slope
    assert bool(((out[..., :cout].double() - want).abs() <= 32 * 2.0 ** -24 * size + 1e-40).all())
    if ld > cout:
        assert bool((out[..., cout:] == 9.0).all())
    if bits is not None:
        assert torch.equal(bits[..., :-1], dab.pack_mat(out[..., :cout].contiguous())) and not bits[..., -1].any()


@pytest.mark.parametrize("cout", [32, 64])
def test_infinities_and_nans(cout):
    g = torch.Generator(device="cuda").manual_seed(cout)
    x, wt = torch.randn((4, 64, 64, 3), device="cuda", generator=g), torch.randn((cout, 3, 3, 3), device="cuda", generator=g)
    for i, v in enumerate([float("inf"), -float("inf"), float("nan"), 3e38, 1e-40]):
        x[i % 4, 7 * i, 5 * i + 1, i % 3] = v
    wt[3, 1, 1, 2] = float("inf")
    out = torch.empty((4, 64, 64, cout), device="cuda")
    rc = capi.lib.dab_fconv_affine_relu(p(x), 4, 64, 64, 3, p(wt), None, None, None, 0, 3, 3, 1, 1, 1, 1, 1, 1, cout, p(out), stream())
    assert rc == 0
    want = torch.nn.functional.conv2d(x.permute(0, 3, 1, 2).cpu(), wt.permute(0, 3, 1, 2).cpu(), padding=1).permute(0, 2, 3, 1).cuda()
    assert torch.equal(out.isnan(), want.isnan()) and torch.equal(out.isinf(), want.isinf())
    inf = want.isinf()
    assert torch.equal(out[inf], want[inf])


@pytest.mark.parametrize("n,h,w,cout,stride,pad,dil", [
    (1, 90, 92, 32, 1, 1, 1), (1, 100, 100, 64, 1, 1, 1), (1, 128, 128, 64, 1, 1, 1), (6, 112, 112, 32, 2, 1, 1), (1, 181, 181, 64, 1, 1, 1), (1, 181, 182, 33, 1, 1, 1),
    (256, 9, 17, 17, 2, 3, 1), (32, 32, 32, 64, 1, 1, 1), (33, 32, 32, 64, 1, 1, 1), (5, 99, 130, 48, 1, 2, 2), (64, 32, 31, 1, 1, 0, 1), (128, 32, 32, 64, 1, 1, 1),
    (90, 224, 224, 32, 2, 1, 1), (180, 112, 112, 64, 1, 1, 1)])
def test_sums_are_the_tile_kernels_to_the_bit(n, h, w, cout, stride, pad, dil):
    """With the filters of 96 channels (zeros behind the first) the tile kernels run, below 256 tiles of 128 pixels with the depth split over
    waves: the same sums in the same order."""
    g = torch.Generator(device="cuda").manual_seed(n + w)
    x, wt = torch.randn((n, h, w, 3), device="cuda", generator=g), torch.zeros((96, 3, 3, 3), device="cuda")
    wt[:cout] = torch.randn((cout, 3, 3, 3), device="cuda", generator=g)
    oh, ow = (h + 2 * pad - 2 * dil - 1) // stride + 1, (w + 2 * pad - 2 * dil - 1) // stride + 1
    got, want = (torch.full((n, oh, ow, c), 9.0, device="cuda") for c in (cout, 96))
    for c, out in ((cout, got), (96, want)):
        assert capi.lib.dab_fconv_affine_relu(p(x), n, h, w, 3, p(wt), None, None, None, 0, 3, 3, pad, pad, stride, stride, dil, dil, c, p(out), stream()) == 0, capi.last_error()
    differ = (got != want[..., :cout]).float().mean().item()
    assert differ == 0, "%.3g of the values differ" % differ
