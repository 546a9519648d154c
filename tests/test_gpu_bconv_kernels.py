"""The direct 3x3 binary convolution at the sizes where its kernels and the rule that picks one of them can go wrong:
tiles that are not full in pixels or channels, both sides of every switch, windows that fit no kernel but the last one,
and operands whose bits are all equal (the largest and the smallest count).  Counts are whole numbers: bit for bit."""
import ctypes

import numpy as np
import pytest
import torch

import oracle as orc

pytestmark = pytest.mark.gpu


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a).view(np.int64) if a.dtype == np.uint64 else np.ascontiguousarray(a)).cuda()


def pieces(n, h, w, cout, stride, pad):
    o = n * ((h + 2 * pad - 3) // stride + 1) * ((w + 2 * pad - 3) // stride + 1)
    return -(-o // 32) * -(-cout // 32)


@pytest.mark.parametrize("n,h,w,cin,cout,stride,pad", [
    # one pixel, one group of eight channels; a row of pixels; channel counts that fill no 16- or 32-channel tile
    (1, 1, 1, 64, 8, 1, 1), (1, 1, 1, 512, 8, 1, 1), (1, 1, 17, 128, 24, 1, 1), (1, 5, 7, 256, 40, 1, 1), (3, 3, 3, 512, 72, 3, 0),
    # 64 input channels: 222 / 224 / 228 pieces (16- and 32-pixel tiles), 760 / 768 (walking kernel), with 64 output
    # channels or fewer, more, and from 6000 pieces
    (1, 37, 96, 64, 64, 1, 1), (1, 56, 64, 64, 64, 1, 1), (1, 57, 64, 64, 40, 1, 1), (17, 19, 19, 64, 128, 1, 1), (9, 30, 45, 64, 64, 1, 1),
    (13, 57, 33, 64, 56, 1, 1), (11, 33, 29, 64, 88, 1, 1), (67, 41, 35, 64, 72, 1, 1),
    # deeper: 160 / 165 pieces, 1280 / 1296, 2032 / 2048
    (5, 16, 16, 128, 128, 1, 1), (6, 17, 17, 256, 96, 1, 1), (1, 28, 41, 512, 1128, 1, 1), (20, 16, 16, 512, 256, 1, 1),
    (7, 20, 58, 128, 256, 1, 1), (16, 16, 32, 256, 256, 1, 1), (25, 21, 31, 512, 136, 1, 1),
    # walking kernel over ragged tiles at stride 2 and 3 and without padding
    (30, 27, 31, 128, 328, 2, 1), (90, 27, 31, 256, 72, 3, 1), (40, 19, 23, 512, 200, 2, 0),
    # windows too wide for LDS, and outputs that reach past the image on both sides
    (2, 70, 250, 512, 128, 1, 1), (60, 12, 12, 256, 128, 1, 2), (400, 4, 4, 128, 256, 1, 2), (300, 2, 9, 128, 256, 2, 2),
])
@pytest.mark.parametrize("bits", ["random", "equal", "opposite"])
def test_bconv_at_the_edges_of_its_kernels(n, h, w, cin, cout, stride, pad, bits):
    import dabnn_amd as dab
    if bits != "random" and pieces(n, h, w, cout, stride, pad) > 1300:
        pytest.skip("the extremes need no large problem")
    r = np.random.default_rng(n * 1000 + h * 10 + cin)
    cw = cin // 64
    shape, wshape = (n, h, w, cw), (cout, 9 * cw)
    if bits == "random":
        x, wgt = r.integers(0, 2**64, size=shape, dtype=np.uint64), r.integers(0, 2**64, size=wshape, dtype=np.uint64)
    else:
        ones = np.uint64(0xffffffffffffffff)
        x, wgt = np.full(shape, ones), np.full(wshape, ones if bits == "equal" else np.uint64(0))
    sample = sorted({0, n // 2, n - 1})
    want = np.stack([orc.baseline_bconv(x[i], wgt, 3, 3, pad, pad, stride, stride) for i in sample])
    got = dab.bconv_3x3(dev(x), dev(wgt), stride, pad)
    np.testing.assert_array_equal(got[sample].cpu().numpy(), want)
    a, b = (r.standard_normal(cout) / 50).astype(np.float32), r.standard_normal(cout).astype(np.float32)
    a[::5], b[::10] = 0.0, 0.0
    shortcut = r.standard_normal(got.shape).astype(np.float32)
    shortcut[..., ::10] = 0.0
    # the separate layers over the counts: each of their steps is rounded by itself in the fused pass too
    sep = got.clone()
    dab.affine_inplace(sep, dev(a), dev(b))
    assert torch.equal(dab.bconv_3x3_affine_add(dev(x), dev(wgt), dev(a), dev(b), None, stride, pad), sep)
    dab.add_inplace(sep, dev(shortcut))
    assert torch.equal(dab.bconv_3x3_affine_add(dev(x), dev(wgt), dev(a), dev(b), dev(shortcut), stride, pad), sep)
    if cout % 64 == 0:
        fused, packed = dab.bconv_3x3_affine_add_sign(dev(x), dev(wgt), dev(a), dev(b), dev(shortcut), stride, pad)
        assert torch.equal(fused, sep) and torch.equal(packed, dab.pack_mat(sep))


# The last tile of a walking kernel is ragged: its rows past the tensor, and channels past the last, are stored nowhere.
@pytest.mark.parametrize("n,h,w,cin,cout", [(13, 57, 33, 64, 56), (67, 41, 35, 64, 72), (30, 27, 31, 128, 328), (25, 21, 31, 512, 136),
                                            (11, 27, 29, 256, 320), (1, 1, 1, 64, 8)])
def test_bconv_stores_nothing_past_its_output(n, h, w, cin, cout):
    import dabnn_amd as dab
    from dabnn_amd import capi
    r = np.random.default_rng(cin + cout)
    x = dev(r.integers(0, 2**64, size=(n, h, w, cin // 64), dtype=np.uint64))
    wgt = dev(r.integers(0, 2**64, size=(cout, 9 * cin // 64), dtype=np.uint64))
    a, b = dev(r.standard_normal(cout).astype(np.float32)), dev(r.standard_normal(cout).astype(np.float32))
    size, guard = n * h * w * cout, 64 * cout  # a tile reaches 64 pixels at most
    ptr = lambda t, at=0: ctypes.c_void_p(t.data_ptr() + at)
    for fused in (False, True):
        buf = torch.full((guard + size + guard,), -7.0, device="cuda")
        if fused:
            want = dab.bconv_3x3_affine_add(x, wgt, a, b, None, 1, 1)
            capi.check(capi.lib.dab_bconv3x3_affine_add(ptr(x), n, h, w, cin, ptr(wgt), cout, 1, 1, ptr(a), ptr(b), None, ptr(buf, 4 * guard), None))
        else:
            want = dab.bconv_3x3(x, wgt, 1, 1)
            capi.check(capi.lib.dab_bconv3x3(ptr(x), n, h, w, cin, ptr(wgt), cout, 1, 1, ptr(buf, 4 * guard), None))
        torch.cuda.synchronize()
        assert torch.equal(buf[guard:guard + size], want.reshape(-1))
        assert bool((buf[:guard] == -7).all()) and bool((buf[guard + size:] == -7).all())
