"""3x3 convolutions over 32 channels with two work items and more per wave, on three bf16 parts: operands kept whole, pixels and filters of
magnitudes far apart, infinities and NaN; with and without the MaxPool; against 64-bit sums."""
import pytest
import torch
import torch.nn.functional as F

import dabnn_amd as dab

pytestmark = pytest.mark.gpu
N = 22  # 112 x 112: 4312 items on 2048 waves


def inputs(cout, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randn(N, 112, 112, 32, device="cuda", generator=g).relu_(), torch.randn(cout, 3, 3, 32, device="cuda", generator=g) / 17


def reference(x, w, pooled):
    wt, xt = w.double().cpu().permute(0, 3, 1, 2), x.double().cpu().permute(0, 3, 1, 2)
    pool = (lambda t: F.max_pool2d(t, 3, 2, 1)) if pooled else (lambda t: t)
    return tuple(pool(F.conv2d(v, k, padding=1)).permute(0, 2, 3, 1) for v, k in ((xt, wt), (xt.abs(), wt.abs())))


def run(x, w, pooled):
    if pooled:
        return dab.fconv_maxpool(x, w, None, None, None, False, 3, 3, 1, 1, 1, 1, want_sign=w.shape[0] == 64)[0]
    return dab.fconv(x, w, None, 3, 3, 1, 1, 1, 1)


def check(x, w, pooled):
    got = run(x, w, pooled)
    few = torch.cat([got[:2], got[-1:]]).double().cpu()
    want, size = reference(torch.cat([x[:2], x[-1:]]), w, pooled)
    # the terms left out: 2^-24 of a product; 54 matrix instructions that round the sum five times each at most, half an ulp a time
    # (and a few to spare); denormal results
    bound = (2.0**-21 + 288 * 2.0**-24) * size + 2.0**-148
    assert bool(((few - want).abs() <= bound).all())
    return float((few - want).norm() / want.norm())


@pytest.mark.parametrize("cout", [32, 64])
@pytest.mark.parametrize("pooled", [False, True])
def test_no_larger_error_than_an_fp32_sum(cout, pooled):
    error = check(*inputs(cout, cout), pooled)
    print("relative 2-norm error %.3g" % error)
    # 288 products in fp32 one after the other: roundings spread evenly over half an ulp (2^-24 / sqrt(3) in the root mean square) of
    # partial sums whose variances 1, 2 .. 288 add up to 288 * 289 / 2
    assert error < 2.0**-24 / 3**0.5 * (289 / 2)**0.5


# every output channel copies one input channel at one tap: no operand loses a bit on its way to the products
@pytest.mark.parametrize("cout", [32, 64])
@pytest.mark.parametrize("pooled", [False, True])
@pytest.mark.parametrize("tap", [(1, 1), (0, 2)])
def test_copied_channels_are_exact(cout, pooled, tap):
    x = torch.randn(N, 112, 112, 32, device="cuda", generator=torch.Generator(device="cuda").manual_seed(cout))
    w = torch.zeros(cout, 3, 3, 32, device="cuda")
    w[torch.arange(cout), tap[0], tap[1], torch.arange(cout) % 32] = 1
    moved = F.pad(x, (0, 0, 1, 1, 1, 1))[:, tap[0]:tap[0] + 112, tap[1]:tap[1] + 112, torch.arange(cout) % 32].contiguous()
    assert torch.equal(run(x, w, pooled), dab.max_pool(moved, 3, 3, 1, 1, 2, 2) if pooled else moved)


@pytest.mark.parametrize("cout,pooled", [(32, False), (64, False), (64, True)])
@pytest.mark.parametrize("case", ["scales", "large", "tiny", "far pixels", "far filters"])
def test_magnitudes(cout, pooled, case):
    x, w = inputs(cout, 3)
    if case == "scales":
        x *= 2.0 ** (torch.arange(N, device="cuda") % 9 * 20.0 - 80).view(-1, 1, 1, 1)
        x[:, ::16] *= 2.0**-11
        w *= 2.0 ** (torch.arange(cout, device="cuda") % 16 * 2.0 - 16).view(-1, 1, 1, 1)
    elif case == "large":
        x *= 2.0**120
        w *= 2.0**-10
    elif case == "tiny":
        x *= 2.0**-100
        w *= 2.0**60
    elif case == "far pixels":
        x[:, 40:60, 32:80] *= 2.0**-40  # inside items, and items of nothing else
        x[0, :8, :40] = 0
    else:
        w[5::9, :, :, 3:] *= 2.0**-33
        x[..., :3] = 0
    check(x, w, pooled)


# finite operands whose sums are below every float: max_pool starts at the lowest float, which a cell of nothing but such sums holds
@pytest.mark.parametrize("cout", [32, 64])
def test_pool_of_sums_that_overflow(cout):
    x = torch.full((N, 112, 112, 32), 3e38, device="cuda")
    x[0] = 1.0
    w = torch.zeros(cout, 3, 3, 32, device="cuda")
    w[::2, 1, 1] = -1.0
    w[1::2, 1, 1, 0] = 0.5
    full = run(x, w, False)
    assert bool(full[1:, :, :, ::2].isneginf().all()) and bool(full[:, :, :, 1::2].isfinite().all())
    got = run(x, w, True)
    assert torch.equal(got, dab.max_pool(full, 3, 3, 1, 1, 2, 2))
    assert bool((got[1:, :, :, ::2] == torch.finfo(torch.float32).min).all())


@pytest.mark.parametrize("cout", [32, 64])
@pytest.mark.parametrize("where", ["pixels", "filters"])
def test_infinities_and_nan(cout, where):
    x, w = inputs(cout, 4)
    values = torch.tensor([float("inf"), float("-inf"), float("nan")], device="cuda")
    if where == "pixels":
        x.view(-1)[7000:7000 + 40001 * 3:40001] = values
    else:
        w.view(-1)[100:100 + 401 * 3:401] = values
    w.view(-1)[5::7] = 0
    got = run(x, w, False)[:2].cpu().double()
    want, _ = reference(x[:2], w, False)
    assert torch.equal(got.isnan(), want.isnan())
    assert torch.equal(got[got.isinf()], want[want.isinf()])
    ok = want.isfinite()
    assert torch.allclose(got[ok], want[ok], rtol=1e-4, atol=1e-4)
