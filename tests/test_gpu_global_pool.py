"""The average over a whole image at the sizes where its kernel can go wrong: windows around the numbers of taps it keeps
under way, channel counts that fill no wave, one image and many.  The taps are added in the reference's order
(dabnn/layers/AvePool.cpp:84-123), so the result is the oracle's bit for bit."""
import numpy as np
import pytest
import torch

import oracle as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,h,w,c", [
    (1, 1, 17, 1), (3, 4, 4, 64), (9, 4, 5, 3), (2, 31, 1, 64), (5, 4, 8, 66), (17, 3, 11, 5), (9, 7, 7, 512), (300, 7, 7, 20),
    (4, 5, 10, 63), (2, 7, 9, 65), (11, 8, 8, 256), (3, 5, 13, 7), (2, 9, 11, 100), (33, 16, 16, 256), (1, 56, 56, 64), (1, 1, 129, 4),
])
def test_average_over_the_whole_image(n, h, w, c):
    import dabnn_amd as dab
    x = np.random.default_rng(h * 100 + w).standard_normal((n, h, w, c)).astype(np.float32)
    x[-1, 0, 0, 0] = np.inf
    got = dab.ave_pool(torch.from_numpy(x).cuda(), h, w, 0, 0, 3, 2).cpu().numpy()
    sample = sorted({0, n // 2, n - 1})
    np.testing.assert_array_equal(got[sample], np.stack([orc.ave_pool(x[i], h, w, 0, 0, 3, 2) for i in sample]))


@pytest.mark.parametrize("m,cout", [(1, 70), (8, 64), (9, 33), (40, 1000), (256, 1000), (300, 31), (70000, 8)])
def test_a_second_copy_of_the_result(m, cout):
    """dab_fconv_affine_relu_copy: the result and what pinned memory holds are the plain call's, whichever kernel runs; nothing is written past them."""
    import ctypes
    import torch
    from dabnn_amd import capi
    g = torch.Generator(device="cuda").manual_seed(m)
    x, w = torch.randn((m, 1, 1, 64), device="cuda", generator=g), torch.randn((cout, 64), device="cuda", generator=g)
    s = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    args = (x.data_ptr(), m, 1, 1, 64, w.data_ptr(), None, None, None, 1, 1, 1, 0, 0, 1, 1, 1, 1, cout)
    want, out = torch.empty((m, cout), device="cuda"), torch.empty((m, cout), device="cuda")
    host = torch.full((m * cout + 8,), -3.0).pin_memory()
    assert capi.lib.dab_fconv_affine_relu(*args, want.data_ptr(), s) == 0
    assert capi.lib.dab_fconv_affine_relu_copy(*args, out.data_ptr(), host.data_ptr(), s) == 0
    torch.cuda.synchronize()
    assert torch.equal(out, want) and torch.equal(host[:-8].view(m, cout), want.cpu()) and bool((host[-8:] == -3).all())
    if m <= 8:
        y = torch.randn((m, 7, 7, 64), device="cuda", generator=g)
        pooled = torch.empty((m, 64), device="cuda")
        gap = (y.data_ptr(), m, 7, 7, 64, w.data_ptr(), None, None, None, 0, cout, pooled.data_ptr())
        assert capi.lib.dab_global_ave_pool_fconv1x1(*gap, want.data_ptr(), s) == 0
        assert capi.lib.dab_global_ave_pool_fconv1x1_copy(*gap, out.data_ptr(), host.data_ptr(), s) == 0
        torch.cuda.synchronize()
        assert torch.equal(out, want) and torch.equal(host[:-8].view(m, cout), want.cpu())


@pytest.mark.parametrize("n,h,c,cout,k,pad", [(3, 5, 64, 40, 3, 1), (2, 9, 20, 33, 1, 0), (5, 6, 3, 70, 5, 2), (4, 7, 65, 31, 3, 0), (1, 12, 7, 100, 2, 1), (9, 40, 64, 64, 3, 1)])
def test_a_second_copy_of_windows(n, h, c, cout, k, pad):
    """The copying forms of the kernel that splits the depth: padded and not, four channels a load and one; and a larger problem, copied by a launch."""
    import ctypes
    from dabnn_amd import capi
    g = torch.Generator(device="cuda").manual_seed(n + c)
    x, w, b = (torch.randn(s, device="cuda", generator=g) for s in ((n, h, h, c), (cout, k, k, c), (cout,)))
    s, o = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream), h + 2 * pad - k + 1
    args = (x.data_ptr(), n, h, h, c, w.data_ptr(), b.data_ptr(), None, None, 0, k, k, pad, pad, 1, 1, 1, 1, cout)
    want, out = torch.empty((n, o, o, cout), device="cuda"), torch.empty((n, o, o, cout), device="cuda")
    host = torch.full((want.numel() + 8,), -3.0).pin_memory()
    assert capi.lib.dab_fconv_affine_relu(*args, want.data_ptr(), s) == 0
    assert capi.lib.dab_fconv_affine_relu_copy(*args, out.data_ptr(), host.data_ptr(), s) == 0
    torch.cuda.synchronize()
    assert torch.equal(out, want) and torch.equal(host[:-8].view_as(want), want.cpu()) and bool((host[-8:] == -3).all())
