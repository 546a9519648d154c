"""1x1 float convolutions with 64 to 256 input channels, large problems: errors against 64-bit sums, operands kept whole, pixels that fill
no tile, channels that fill no column, channel slices with sign bits, averages of odd images, infinities and values far apart."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def problem(m, c, cout, seed=1):
    gen = torch.Generator(device="cuda").manual_seed(seed + c + cout)
    x = torch.randn((1, m, 1, c), device="cuda", generator=gen)
    wgt = torch.randn((cout, 1, 1, c), device="cuda", generator=gen)
    return (x, wgt) + tuple(torch.randn(cout, device="cuda", generator=gen) for _ in range(3))


def sums(x, wgt, bias):
    rows, wt = x.reshape(-1, x.shape[-1]).double(), wgt.reshape(wgt.shape[0], -1).double()
    # a sum of c products and a bias, each step rounded once at most: (c + 1) half ulps of the sum of magnitudes
    bound = (x.shape[-1] + 1) * 2.0**-24 * (rows.abs() @ wt.abs().t() + bias.abs())
    return rows @ wt.t() + bias, bound


# pixels * channels = 4 M, with the outputs 2^29, from 192 channels on 5 * 2^26, and one pixel fewer; pixels that fill no tile
@pytest.mark.parametrize("m,c,cout", [
    (65536, 64, 64), (65535, 64, 64), (70001, 64, 320), (32768, 128, 96), (33001, 128, 416), (131071, 128, 128), (2048, 128, 2048), (2047, 128, 2048),
    (21846, 192, 160), (22001, 192, 128), (16384, 256, 64), (16399, 256, 256), (8192, 256, 512), (16401, 256, 288),
    (2560, 256, 512), (2559, 256, 512), (1024, 256, 1280), (24576, 192, 256), (24577, 192, 256), (8193, 64, 1024),
])
def test_against_64_bit_sums(m, c, cout):
    import dabnn_amd as dab
    x, wgt, bias, a, b = problem(m, c, cout)
    got = dab.fconv(x, wgt, bias, 1, 1, 0, 0, 1, 1)
    want, bound = sums(x, wgt, bias)
    err = (got.reshape(-1, cout).double() - want).abs()
    assert bool((err <= bound).all())
    # no worse than c products and a bias in fp32 one after the other: c + 1 roundings, each spread evenly over half an ulp of at most 2^-23
    # of its partial sum (2^-24 / sqrt(3) of it in the root mean square), of sums whose variances 1, 2 .. c + 1 make (c + 1) * (c + 2) / 2
    assert float((err**2).mean().sqrt() / (want**2).mean().sqrt()) < 2.0**-24 / 3**0.5 * ((c + 2) / 2)**0.5
    sep = got.clone()
    dab.affine_inplace(sep, a, b)
    assert torch.equal(dab.fconv_affine_relu(x, wgt, bias, a, b, False, 1, 1, 0, 0, 1, 1), sep)
    assert torch.equal(dab.fconv_affine_relu(x, wgt, bias, a, b, True, 1, 1, 0, 0, 1, 1), sep.clamp_min(0))
    # a pixel's result does not depend on its place
    if m > 100000:
        assert torch.equal(dab.fconv(x[:, 5:].contiguous(), wgt, bias, 1, 1, 0, 0, 1, 1), got[:, 5:])


@pytest.mark.parametrize("m,c,cout,extra,first", [(32777, 128, 192, 72, 8), (16411, 256, 128, 3, 1), (8200, 256, 256, 128, 64), (65539, 64, 64, 65, 64)])
def test_prelu_into_a_slice(m, c, cout, extra, first):
    import dabnn_amd as dab
    from dabnn_amd import capi
    x, wgt, bias, a, b = problem(m, c, cout)
    want = dab.fconv_affine_relu(x, wgt, bias, a, b, False, 1, 1, 0, 0, 1, 1)
    want = torch.where(want < 0, want * b, want)
    wide = torch.full((1, m, 1, cout + extra), 7.0, device="cuda")
    bits = torch.full((1, m, 1, cout // 64 + 2), 5, dtype=torch.int64, device="cuda")
    capi.check(capi.lib.dab_fconv_affine_prelu(
        x.data_ptr(), 1, m, 1, c, wgt.data_ptr(), bias.data_ptr(), a.data_ptr(), b.data_ptr(), b.data_ptr(), cout, 1, 1, 0, 0, 1, 1, 1, 1, cout,
        wide.data_ptr() + 4 * first, cout + extra, bits.data_ptr() + 8, cout // 64 + 2, None))
    torch.cuda.synchronize()
    assert torch.equal(wide[..., first:first + cout], want)
    assert (wide[..., :first] == 7).all() and (wide[..., first + cout:] == 7).all()
    assert torch.equal(bits[..., 1:-1], dab.pack_mat(want.contiguous()).reshape(1, m, 1, -1))
    assert (bits[..., 0] == 5).all() and (bits[..., -1] == 5).all()


@pytest.mark.parametrize("n,h,w,c,cout", [
    (11, 113, 121, 128, 128), (17, 65, 67, 256, 320), (9, 65, 67, 256, 512), (2, 150, 130, 128, 1024), (21, 113, 121, 64, 128), (9, 150, 130, 64, 192),
    (8, 113, 121, 192, 96), (8, 113, 121, 192, 192), (17, 65, 67, 256, 96), (5, 65, 67, 256, 320), (40, 29, 28, 128, 512)])
@pytest.mark.parametrize("want_pooled", [True, False])
def test_averages_are_those_of_the_pool(n, h, w, c, cout, want_pooled):
    import dabnn_amd as dab
    gen = torch.Generator(device="cuda").manual_seed(h)
    x = torch.randn((n, h, w, c), device="cuda", generator=gen)
    _, wgt, bias, a, b = problem(1, c, cout)
    pooled, out = dab.ave_pool2_fconv1x1(x, wgt, bias, a, b, True, want_pooled)
    sep = dab.ave_pool(x, 2, 2, 0, 0, 2, 2)
    if want_pooled:
        assert torch.equal(pooled, sep)
    assert torch.equal(out, dab.fconv_affine_relu(sep, wgt, bias, a, b, True, 1, 1, 0, 0, 1, 1))


@pytest.mark.parametrize("c", [128, 192, 256])
def test_special_values(c):
    import dabnn_amd as dab
    x, wgt, bias, _, _ = problem(32776, c, 160)
    x[0, 7, 0, 3], x[0, 90, 0, 60], x[0, 32775, 0, 1] = float("inf"), float("-inf"), float("nan")
    x[0, 1000, 0, ::2] *= 2.0**-60
    x[0, 2000] *= 2.0**100
    x[0, 3000] *= 2.0**-110
    x[0, 4000] = 0
    wgt[33, 0, 0, ::2] *= 2.0**-50
    got = dab.fconv(x, wgt, bias, 1, 1, 0, 0, 1, 1).reshape(-1, 160).double()
    want, bound = sums(x, wgt, bias)
    finite = want.isfinite()
    assert torch.equal(finite, got.isfinite())
    assert bool((got.isnan() == want.isnan()).all())
    assert bool(((got - want).abs() <= bound)[finite].all())
    assert torch.equal(got[~finite & ~want.isnan()], want[~finite & ~want.isnan()])


# every output channel copies one input channel: no operand loses a bit on its way to the products, so the values come back exactly
@pytest.mark.parametrize("pool", ["none", "average", "maxima"])
@pytest.mark.parametrize("hw,c,cout", [(128, 256, 512), (128, 192, 256), (182, 128, 416), (256, 64, 128)])
def test_copied_channels_are_exact(pool, hw, c, cout):
    import dabnn_amd as dab
    from dabnn_amd import capi
    gen = torch.Generator(device="cuda").manual_seed(c)
    n = 1 if pool == "none" else 4
    x = torch.randn((n, hw, hw, c), device="cuda", generator=gen)
    wgt = torch.zeros((cout, 1, 1, c), device="cuda")
    wgt[torch.arange(cout), 0, 0, torch.arange(cout) % c] = 1
    if pool == "none":
        want, got = x, dab.fconv(x, wgt, None, 1, 1, 0, 0, 1, 1)
    elif pool == "average":
        want, got = dab.ave_pool(x, 2, 2, 0, 0, 2, 2), dab.ave_pool2_fconv1x1(x, wgt, None, None, None, False, False)[1]
    else:
        want, got = dab.max_pool(x, 2, 2, 0, 0, 2, 2), torch.empty((n, hw // 2, hw // 2, cout), device="cuda")
        capi.check(capi.lib.dab_max_pool2_fconv1x1(x.data_ptr(), n, hw, hw, c, wgt.data_ptr(), None, None, None, 0, None, 0, cout,
                                                   got.data_ptr(), cout, None, 0, None))
        torch.cuda.synchronize()
    assert torch.equal(got, want[..., torch.arange(cout) % c])
