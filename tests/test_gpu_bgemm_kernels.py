"""The binary GEMM and the convolution over any window at the sizes where their two kernels and the rule between them can
go wrong: depths that end inside a unit, tiles that are not full, both sides of each switch, the deepest sum that fp32
holds, filters with a padding word, channel slices of wider tensors.  Counts are whole numbers: bit for bit."""
import ctypes

import numpy as np
import pytest
import torch

import oracle as orc

pytestmark = pytest.mark.gpu


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a).view(np.int64) if a.dtype == np.uint64 else np.ascontiguousarray(a)).cuda()


def words(r, *shape):
    return r.integers(0, 2**64, size=shape, dtype=np.uint64)


@pytest.mark.parametrize("m,n,k", [
    # depths of one to three units (walking kernel at any size), an odd and an even number of words in the last one
    (5, 3, 1), (40, 33, 2), (33, 31, 3), (64, 32, 11), (31, 65, 12),
    # four units and more: split over a block's waves; 1023 / 1024 pieces (32 and 64 channels a block)
    (1, 1, 13), (96, 320, 17), (992, 1056, 14), (1024, 1024, 14),
    # 2046 / 2048 pieces; with filters that fit LDS, and that do not
    (352, 5952, 20), (512, 4096, 20), (512, 4096, 19), (24, 65600, 37), (64, 33000, 150),
])
def test_bgemm_at_the_edges_of_its_kernels(m, n, k):
    import dabnn_amd as dab
    r = np.random.default_rng(m + n + k)
    lda, ldb, ldc = m + 3, k + (n % 3), m + 1
    a, b = words(r, k, lda), words(r, n, ldb)
    c0 = r.integers(0, 1000, size=(n, ldc)).astype(np.float32)
    got, over = dev(c0), dev(c0)
    dab.bgemm(m, n, k, dev(a), lda, dev(b), ldb, got, ldc)
    dab.bgemm_overwrite(m, n, k, dev(a), lda, dev(b), ldb, over, ldc)
    rows = sorted(set([0, n // 2, n - 1]) | set(r.integers(0, n, 20).tolist()))
    cnt = np.stack([np.bitwise_count(a[:, :m] ^ b[j, :k, None]).sum(axis=0) for j in rows]).astype(np.float32)
    want = c0[rows]
    want[:, :m] += cnt
    np.testing.assert_array_equal(got[rows].cpu().numpy(), want)
    want[:, :m] = cnt
    np.testing.assert_array_equal(over[rows].cpu().numpy(), want)


@pytest.mark.parametrize("value,count", [(0xffffffffffffffff, 0), (0, 64)])
@pytest.mark.parametrize("m,n,k", [(40, 33, 131071), (24, 70000, 11)])
def test_bgemm_of_equal_and_opposite_bits(m, n, k, value, count):
    """The largest magnitudes of the accumulators: every bit equal, every bit different (k = 131071 words is the limit)."""
    import dabnn_amd as dab
    a, b = torch.full((k, m), -1, dtype=torch.int64, device="cuda"), dev(np.full((n, k), value, np.uint64))
    c = torch.empty((n, m), device="cuda")
    dab.bgemm_overwrite(m, n, k, a, m, b, k, c, m)
    assert torch.equal(c, torch.full_like(c, float(count * k)))


@pytest.mark.parametrize("n,h,w,c,cout,kh,kw,pad_h,pad_w,stride_h,stride_w", [
    # words per pixel: 1 to 9 and 12 (units of 1, 2, 3 and 4 dwords per half wave); windows that are not square
    (2, 7, 9, 64, 12, 5, 5, 2, 2, 1, 1), (1, 6, 5, 128, 5, 1, 1, 0, 0, 1, 1), (3, 9, 8, 192, 33, 3, 3, 1, 1, 1, 1),
    (2, 8, 8, 256, 64, 2, 3, 0, 1, 2, 1), (1, 11, 7, 320, 40, 3, 3, 1, 1, 2, 2), (2, 5, 5, 384, 64, 3, 1, 1, 0, 1, 2),
    (1, 9, 9, 448, 24, 5, 5, 2, 2, 2, 2), (2, 7, 7, 512, 72, 4, 4, 3, 3, 3, 3), (1, 6, 6, 576, 8, 3, 3, 1, 1, 1, 1), (1, 5, 7, 768, 64, 3, 3, 2, 2, 1, 1),
    # 1023 / 1024 pieces of few units, 2047 / 2048: the walking kernel; a depth whose filters do not fit LDS
    (31, 32, 33, 64, 40, 3, 3, 1, 1, 1, 1), (32, 32, 32, 192, 64, 3, 3, 1, 1, 1, 1), (23, 89, 16, 128, 64, 1, 1, 0, 0, 1, 1), (32, 32, 32, 512, 64, 5, 5, 2, 2, 1, 1),
    (20, 41, 40, 192, 72, 3, 3, 1, 1, 1, 1),
])
def test_bconv_over_any_window(n, h, w, c, cout, kh, kw, pad_h, pad_w, stride_h, stride_w):
    import dabnn_amd as dab
    from dabnn_amd import capi
    r = np.random.default_rng(h * w + c)
    cw, k = c // 64, kh * kw * c // 64
    wide = words(r, n, h, w, cw + 3)  # the input is words 2 .. of a wider tensor
    x = np.ascontiguousarray(wide[..., 2:2 + cw])
    wgt = words(r, cout, k)
    padded = np.concatenate([wgt, words(r, cout, 1)], axis=1) if k % 2 else wgt  # the padding word meets zeros
    extra = np.bitwise_count(padded[:, k:]).sum(axis=1).astype(np.float32)
    sample = sorted({0, n // 2, n - 1})
    want = np.stack([orc.baseline_bconv(x[i], wgt, kh, kw, pad_h, pad_w, stride_h, stride_w) for i in sample])
    got = dab.bconv(dev(x), dev(wgt), kh, kw, pad_h, pad_w, stride_h, stride_w)
    np.testing.assert_array_equal(got[sample].cpu().numpy(), want)
    counts = dab.bconv(dev(x), dev(padded), kh, kw, pad_h, pad_w, stride_h, stride_w)
    np.testing.assert_array_equal(counts[sample].cpu().numpy(), want + extra)
    a, b = dev((r.standard_normal(cout) / 50).astype(np.float32)), dev(r.standard_normal(cout).astype(np.float32))
    shortcut = dev(r.standard_normal(tuple(got.shape)).astype(np.float32))
    sep = got.clone()
    dab.affine_inplace(sep, a, b)
    assert torch.equal(dab.bconv(dev(x), dev(wgt), kh, kw, pad_h, pad_w, stride_h, stride_w, a, b), sep)
    dab.add_inplace(sep, shortcut)
    assert torch.equal(dab.bconv(dev(x), dev(wgt), kh, kw, pad_h, pad_w, stride_h, stride_w, a, b, shortcut), sep)
    # strided on both sides: a channel slice in, a channel slice out, the rest of the output untouched
    out = torch.full(tuple(got.shape[:-1]) + (cout + 5,), -7.0, device="cuda")
    xd, wd = dev(wide), dev(wgt)
    capi.check(capi.lib.dab_bconv(ctypes.c_void_p(xd.data_ptr() + 16), cw + 3, n, h, w, c, ctypes.c_void_p(wd.data_ptr()), k, kh, kw, pad_h, pad_w,
                                  stride_h, stride_w, cout, None, None, None, ctypes.c_void_p(out.data_ptr() + 8), cout + 5, None, 0, None))
    torch.cuda.synchronize()
    assert torch.equal(out[..., 2:2 + cout], got) and bool((out[..., :2] == -7).all()) and bool((out[..., 2 + cout:] == -7).all())
    if cout % 64 == 0:
        res, packed = dab.bconv(dev(x), dev(wgt), kh, kw, pad_h, pad_w, stride_h, stride_w, a, b, shortcut, want_sign=True)
        assert torch.equal(res, sep) and torch.equal(packed, dab.pack_mat(sep))
