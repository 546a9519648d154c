"""1x1 float convolutions on the 64 x 64 tile: pixels and channels that fill no tile, depths that fill no 32-deep slice, both
sides of the switches (three quarters of the CUs; deep problems of four 128 x 128 tiles a CU), strides, biases, Affine."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,h,w,c,cout,stride", [
    (1, 95, 64, 4, 65, 1), (1, 96, 64, 36, 72, 1), (3, 57, 37, 100, 100, 1), (9, 31, 33, 192, 130, 1), (4, 61, 63, 8, 128, 2),
    (16, 28, 27, 516, 256, 1), (1, 47, 64, 64, 256, 1), (1, 49, 63, 64, 256, 1), (1, 230, 285, 1024, 256, 1), (1, 230, 284, 516, 256, 1),
])
def test_1x1_against_64_bit_sums(n, h, w, c, cout, stride):
    import dabnn_amd as dab
    gen = torch.Generator(device="cuda").manual_seed(c + cout)
    x = torch.randn((n, h, w, c), device="cuda", generator=gen)
    wgt = torch.randn((cout, 1, 1, c), device="cuda", generator=gen)
    bias, a, b = (torch.randn(cout, device="cuda", generator=gen) for _ in range(3))
    got = dab.fconv(x, wgt, bias, 1, 1, 0, 0, stride, stride)
    rows, wt = x[:, ::stride, ::stride].reshape(-1, c).double(), wgt.reshape(cout, c).double()
    want = rows @ wt.t() + bias
    # a sum of c products and a bias, each step rounded once at most: (c + 1) half ulps of the sum of magnitudes
    bound = (c + 1) * 2.0**-24 * (rows.abs() @ wt.abs().t() + bias.abs())
    assert bool(((got.reshape(-1, cout).double() - want).abs() <= bound).all())
    sep = got.clone()
    dab.affine_inplace(sep, a, b)
    assert torch.equal(dab.fconv_affine_relu(x, wgt, bias, a, b, False, 1, 1, 0, 0, stride, stride), sep)
