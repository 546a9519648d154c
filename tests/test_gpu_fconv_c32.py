"""3x3 convolutions over 32 channels where there are fewer work items than two per wave: blocks of 16 or 32 output
channels, the cross terms of the split operands summed by themselves (dabnn/fconv.h:14-76)."""
import pytest
import torch
import torch.nn.functional as F

import dabnn_amd as dab

pytestmark = pytest.mark.gpu


def reference(x, w, bias, a, b, relu, pad):
    """The layers in 64 bits, and the sum of the products' magnitudes for the bound of the error."""
    wt = w.cpu().double().permute(0, 3, 1, 2)
    xt = x.cpu().double().permute(0, 3, 1, 2)
    y, size = (F.conv2d(v, k, padding=pad).permute(0, 2, 3, 1) for v, k in ((xt, wt), (xt.abs(), wt.abs())))
    if bias is not None:
        y, size = y + bias.cpu().double(), size + bias.cpu().double().abs()
    if a is not None:
        a, b = a.cpu().double(), b.cpu().double()
        y, size = a * y + b, a.abs() * size + b.abs()
    return (y.clamp(min=0) if relu else y), size


def inputs(n, h, w, cout, seed, vectors=True):
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randn(n, h, w, 32, device="cuda", generator=g)
    wt = torch.randn(cout, 3, 3, 32, device="cuda", generator=g) / 17
    vec = [torch.randn(cout, device="cuda", generator=g) for _ in range(3)] if vectors else [None] * 3
    return x, wt, vec


# 36 items (the fewest taken), ragged last row group, paddings 0 to 2, about one item per wave of 256 CUs from either
# side (2016 and 2080 items), about two (4032 and 4116)
CASES = [(1, 48, 48, 1, 32), (1, 48, 48, 1, 64), (3, 49, 48, 1, 64), (2, 50, 34, 0, 32), (2, 31, 62, 2, 64),
         (36, 32, 112, 1, 64), (65, 32, 64, 1, 64), (63, 64, 64, 1, 32), (63, 64, 64, 1, 64), (21, 112, 112, 1, 32)]


@pytest.mark.parametrize("n,h,w,pad,cout", CASES)
def test_against_64_bits(n, h, w, pad, cout):
    x, wt, (bias, a, b) = inputs(n, h, w, cout, 5 * n + h + cout)
    got = dab.fconv_affine_relu(x, wt, bias, a, b, False, 3, 3, pad, pad, 1, 1)
    few = min(n, 4)
    want, size = reference(x[:few], wt, bias, a, b, False, pad)
    err = (got[:few].cpu().double() - want).abs()
    # any order of 288 fp32 additions and four more steps
    assert (err <= 292 * 2.0**-24 * size).all()
    # and typically: about a dozen roundings of half an ulp at the result's size (one sum: 2.4e-7)
    assert err.norm() / want.norm() < (1.5e-7 if n * -(-want.shape[1] // 4) * want.shape[2] // 16 < 4096 else 4e-7)
    # the last images too, in the sums that the first ones had
    again = dab.fconv_affine_relu(torch.cat([x[-few:], x[few:]]), wt, bias, a, b, False, 3, 3, pad, pad, 1, 1)
    assert torch.equal(again[:few], got[-few:])


@pytest.mark.parametrize("n,hw,cout", [(1, 112, 32), (1, 112, 64), (2, 112, 64), (7, 112, 32), (12, 112, 64)])
def test_pooled_equals_two_steps(n, hw, cout):
    x, wt, (bias, a, b) = inputs(n, hw, hw, cout, n + cout)
    pooled, packed = dab.fconv_maxpool(x, wt, bias, a, b, True, 3, 3, 1, 1, 1, 1, want_sign=cout == 64)
    full = dab.fconv_affine_relu(x, wt, bias, a, b, True, 3, 3, 1, 1, 1, 1)
    want = dab.max_pool(full, 3, 3, 1, 1, 2, 2)
    assert torch.equal(pooled, want)
    if cout == 64:
        assert torch.equal(packed, dab.pack_mat(want))


@pytest.mark.parametrize("cout", [32, 64])
@pytest.mark.parametrize("where", ["input", "filter", "none"])
def test_special_values_as_the_general_kernel_gives_them(cout, where):
    """Infinities, NaN, zeros and the largest numbers; a buffer off the 16-byte grid takes the general kernel."""
    x, wt, (bias, a, b) = inputs(2, 48, 48, cout, cout)
    special = torch.tensor([float("inf"), float("-inf"), float("nan"), 3.4028235e38, -3.4028235e38, 0.0, -0.0, 1e-40], device="cuda")
    if where == "input":
        x.view(-1)[1000:1000 + 5000 * 8:5000] = special
    elif where == "filter":
        wt.view(-1)[7:7 + 601 * 8:601] = special
    got = dab.fconv_affine_relu(x, wt, bias, a, b, True, 3, 3, 1, 1, 1, 1)
    off = torch.empty(x.numel() + 1, device="cuda")[1:].view(x.shape).copy_(x)
    want = dab.fconv_affine_relu(off, wt, bias, a, b, True, 3, 3, 1, 1, 1, 1)
    assert torch.equal(got.isnan(), want.isnan())
    assert torch.equal(got.isposinf(), want.isposinf())
    finite = want.isfinite()
    if where == "none":
        assert (got - want)[finite].abs().max() <= 2 * 292 * 2.0**-24 * want[finite].abs().max() * 4
