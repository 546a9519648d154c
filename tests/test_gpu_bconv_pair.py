"""dab_bconv3x3_pair: two residual layers in one pass, bit for bit two calls of dab_bconv3x3_affine_add_sign; strips of every height (one image to many),
ragged last strips, widths either side of a tile, images of one row, zeros and NaN in the shortcut."""
import pytest
import torch

import dabnn_amd as dab
from dabnn_amd import capi

pytestmark = pytest.mark.gpu


def operands(n, h, w, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    v0 = torch.randn(n, h, w, 64, device="cuda", generator=g)
    ws = [torch.randint(-2**62, 2**62, (64, 9), dtype=torch.int64, device="cuda", generator=g) * 2 + 1 for _ in range(2)]
    ab = [(0.05 * torch.randn(64, device="cuda", generator=g), torch.randn(64, device="cuda", generator=g)) for _ in range(2)]
    return v0, ws, ab


def pair(v0, ws, ab, want_bits=True, guard=0):
    n, h, w, _ = v0.shape
    out = torch.full((v0.numel() + 2 * guard,), -5.0, device="cuda")
    bits = torch.full((n * h * w + 2 * guard,), -5, dtype=torch.int64, device="cuda")
    x = dab.pack_mat(v0)
    rc = capi.lib.dab_bconv3x3_pair(x.data_ptr(), v0.data_ptr(), n, h, w, ws[0].data_ptr(), ab[0][0].data_ptr(), ab[0][1].data_ptr(), ws[1].data_ptr(),
                                    ab[1][0].data_ptr(), ab[1][1].data_ptr(), out.data_ptr() + 4 * guard, bits.data_ptr() + 8 * guard if want_bits else None,
                                    torch.cuda.current_stream().cuda_stream)
    return rc, out, bits


def same(a, b):
    """Bit for bit, but for the bits of a NaN."""
    nan = b.isnan()
    return torch.equal(a.isnan(), nan) and torch.equal(a[~nan].view(torch.int32), b[~nan].view(torch.int32))


@pytest.mark.parametrize("n,h,w", [
    (1, 56, 56), (2, 56, 56), (37, 56, 56), (300, 56, 56), (1, 1, 16), (1, 2, 31), (3, 3, 32), (2, 5, 33), (3, 17, 17), (40, 28, 28), (5, 14, 18),
    (2, 57, 55), (1, 61, 64), (3, 23, 65), (2, 9, 100), (2, 7, 160), (70, 15, 57), (1, 200, 40), (260, 16, 16),
])
def test_equals_two_layers(n, h, w):
    v0, ws, ab = operands(n, h, w, n + h + w)
    v0.view(-1)[::37] = 0.0
    v0.view(-1)[5::5003] = float("nan")
    v1, x1 = dab.bconv_3x3_affine_add_sign(dab.pack_mat(v0), ws[0], *ab[0], v0, 1, 1)
    v2, x2 = dab.bconv_3x3_affine_add_sign(x1, ws[1], *ab[1], v1, 1, 1)
    guard = 1024
    rc, out, bits = pair(v0, ws, ab, guard=guard)
    assert rc == capi.DAB_OK
    assert same(out[guard:-guard], v2.view(-1))
    assert torch.equal(bits[guard:-guard], x2.view(-1))
    assert bool((out[:guard] == -5).all()) and bool((out[-guard:] == -5).all()) and bool((bits[:guard] == -5).all()) and bool((bits[-guard:] == -5).all())
    rc, alone, untouched = pair(v0, ws, ab, want_bits=False)
    assert rc == capi.DAB_OK and bool((untouched == -5).all())
    assert same(alone, v2.view(-1))


@pytest.mark.parametrize("h,w", [(8, 15), (8, 300), (8, 129)])
def test_widths_that_do_not_fit_are_refused(h, w):
    v0, ws, ab = operands(1, h, w, 1)
    rc, out, _ = pair(v0, ws, ab)
    assert rc == capi.DAB_EUNSUPPORTED and bool((out == -5).all())
