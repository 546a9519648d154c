"""The one-pass 7x7 stem on three bf16 parts: operands kept whole, rows and filters of magnitudes far apart, infinities, NaN, several
channel tiles; against 64-bit sums."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


def reference(x, wgt):
    """Convolution and pool in 64 bits, and the pooled sums of magnitudes."""
    def conv(a, b):
        return F.max_pool2d(F.conv2d(a.permute(0, 3, 1, 2), b.permute(0, 3, 1, 2), stride=2, padding=3), 3, 2, 1).permute(0, 2, 3, 1)
    x, wgt = x.double().cpu(), wgt.double().cpu()
    return conv(x, wgt), conv(x.abs(), wgt.abs())


def operands(n, h, w, cout, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randn((n, h, w, 3), device="cuda", generator=gen), torch.randn((cout, 7, 7, 3), device="cuda", generator=gen) * 0.1


# The terms left out are below 2^-24 of a product; 30 matrix instructions round the sum five times each at most, half an ulp a time:
# 2^-21 + 160 * 2^-24 of the sum of magnitudes is above all of it.
BOUND = 2.0**-21 + 160 * 2.0**-24


@pytest.mark.parametrize("n,h,w,cout,scale_x,scale_w", [
    (1, 8, 224, 64, 0, 0), (2, 15, 223, 64, 100, -60), (3, 40, 224, 68, -70, -20), (2, 16, 224, 128, -20, 110), (2, 16, 224, 64, 60, 45),
    (260, 8, 224, 64, 0, 0),
])
def test_scales(n, h, w, cout, scale_x, scale_w):
    import dabnn_amd as dab
    x, wgt = operands(n, h, w, cout, h + cout)
    x, wgt = x * 2.0**scale_x, wgt * 2.0**scale_w
    x[0, : h // 2] *= 2.0**-9  # bands of one image with scales of their own
    wgt *= (2.0 ** (torch.arange(cout, device="cuda") % 16 - 8)).view(-1, 1, 1, 1)  # and filters
    got, bits = dab.fconv_maxpool(x, wgt, None, None, None, False, 7, 7, 3, 3, 2, 2, want_sign=cout % 64 == 0)
    want, size = reference(x, wgt)
    assert bool(((got.double().cpu() - want).abs() <= BOUND * size).all())
    if bits is not None:
        assert torch.equal(bits, dab.pack_mat(got))


@pytest.mark.parametrize("where", ["rows", "filters", "both"])
def test_values_far_below_the_largest(where):
    import dabnn_amd as dab
    x, wgt = operands(2, 16, 224, 64, 5)
    # the first columns and the first filters meet nothing but small values: their sums show what was kept of those
    if where != "filters":
        x[1, :, :100] *= 2.0**-45
    if where != "rows":
        wgt[:8, :, :, :2] = 0
        wgt[:8, :, :, 2] *= 2.0**-40
        wgt[:8, 3, 3, 1] = 2.0**10
        x[0, :, :, 1] = 0
    got, _ = dab.fconv_maxpool(x, wgt, None, None, None, False, 7, 7, 3, 3, 2, 2)
    want, size = reference(x, wgt)
    assert bool(((got.double().cpu() - want).abs() <= BOUND * size).all())


@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan")])
@pytest.mark.parametrize("where", ["rows", "filters"])
def test_infinities_and_nan(value, where):
    import dabnn_amd as dab
    x, wgt = operands(2, 16, 224, 64, 6)
    if where == "rows":
        x[1, 9, 77, 2] = value
    else:
        wgt[11, 2, 4, 1] = value
    wgt[3, 2, 4, 1] = 0
    a = torch.ones(64, device="cuda")
    # values without an order among them (the pool passes over NaN as the reference's loop does): the convolution by itself
    pooled, _ = dab.fconv_maxpool(x, wgt, None, a, torch.zeros_like(a), False, 7, 7, 3, 3, 2, 2)
    conv = dab.fconv(x, wgt, None, 7, 7, 3, 3, 2, 2)
    want = dab.max_pool(conv, 3, 3, 1, 1, 2, 2)
    # max(x, 0) aside, equal where neither is finite, and close elsewhere
    assert torch.equal(torch.isnan(pooled), torch.isnan(want))
    assert torch.equal(torch.isinf(pooled), torch.isinf(want)) and torch.equal(pooled[torch.isinf(pooled)], want[torch.isinf(want)])
    ok = torch.isfinite(want)
    assert torch.allclose(pooled[ok], want[ok], rtol=1e-5, atol=1e-5)


# every output channel copies one input channel at one tap: no operand loses a bit on its way to the products
@pytest.mark.parametrize("n,h,w,cout", [(2, 16, 224, 64), (3, 40, 223, 128)])
def test_copied_channels_are_exact(n, h, w, cout):
    import dabnn_amd as dab
    x, wgt = operands(n, h, w, cout, 8)
    wgt = torch.zeros_like(wgt)
    padded, oh, ow = F.pad(x, (0, 0, 3, 3, 3, 3)), (h - 1) // 2 + 1, (w - 1) // 2 + 1
    copies = []
    for co in range(cout):
        ky, kx, c = co % 7, co // 7 % 7, co % 3
        wgt[co, ky, kx, c] = 1
        copies.append(padded[:, ky:ky + 2 * oh - 1:2, kx:kx + 2 * ow - 1:2, c])
    got, _ = dab.fconv_maxpool(x, wgt, None, None, None, False, 7, 7, 3, 3, 2, 2)
    assert torch.equal(got, dab.max_pool(torch.stack(copies, -1).contiguous(), 3, 3, 1, 1, 2, 2))


def test_no_larger_error_than_an_fp32_sum():
    import dabnn_amd as dab
    x, wgt = operands(8, 112, 224, 64, 7)
    got, _ = dab.fconv_maxpool(x, wgt, None, None, None, False, 7, 7, 3, 3, 2, 2)
    want, _ = reference(x, wgt)
    error = float((got.double().cpu() - want).norm() / want.norm())
    print("relative 2-norm error %.3g" % error)
    # 147 products in fp32 one after the other: roundings spread evenly over half an ulp (2^-24 / sqrt(3) in the root mean square) of
    # partial sums whose variances 1, 2 .. 147 add up to 147 * 148 / 2
    assert error < 2.0**-24 / 3**0.5 * (148 / 2)**0.5
