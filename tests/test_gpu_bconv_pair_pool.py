"""dab_bconv3x3_pair_pool: two residual layers in one pass whose result is written pooled 2x2 and as sign bits, bit for bit dab_bconv3x3_pair (or,
where that does not take the shape, two layers), the AvePool's order of additions and pack_mat; and the nets that use it."""
import ctypes

import numpy as np
import pytest
import torch

import dabnn_amd as dab
from dabnn_amd import capi

pytestmark = pytest.mark.gpu


def same(a, b):
    nan = b.isnan()
    return torch.equal(a.isnan(), nan) and torch.equal(a[~nan].view(torch.int32), b[~nan].view(torch.int32))


# strips of every even height, a last strip of two rows, tiles that end inside a row pair, the widest and narrowest images
@pytest.mark.parametrize("n,h,w", [(1, 56, 56), (300, 56, 56), (37, 56, 56), (1, 2, 2), (5, 2, 64), (3, 4, 2), (2, 6, 34), (3, 18, 18), (40, 28, 28), (9, 14, 18),
                                   (600, 10, 64), (700, 26, 50), (2, 130, 4), (1, 62, 64), (300, 22, 46)])
@pytest.mark.parametrize("special", [False, True])
def test_bit_for_bit(n, h, w, special):
    g = torch.Generator(device="cuda").manual_seed(n + h + w)
    v0 = torch.randn(n, h, w, 64, device="cuda", generator=g)
    if special:
        for value in (float("nan"), float("inf"), -float("inf"), -0.0):
            v0.view(-1)[torch.randint(0, v0.numel(), (20,), device="cuda", generator=g)] = value
    ws = [torch.randint(-2**62, 2**62, (64, 9), dtype=torch.int64, device="cuda", generator=g) * 2 + 1 for _ in range(2)]
    ab = [(0.05 * torch.randn(64, device="cuda", generator=g), torch.randn(64, device="cuda", generator=g)) for _ in range(2)]
    x, guard = dab.pack_mat(v0), 64
    pooled = torch.full((v0.numel() // 4 + 2 * guard,), -5.0, device="cuda")
    bits = torch.full((n * h * w + 2 * guard,), -5, dtype=torch.int64, device="cuda")
    rc = capi.lib.dab_bconv3x3_pair_pool(x.data_ptr(), v0.data_ptr(), n, h, w, ws[0].data_ptr(), ab[0][0].data_ptr(), ab[0][1].data_ptr(), ws[1].data_ptr(),
                                         ab[1][0].data_ptr(), ab[1][1].data_ptr(), pooled.data_ptr() + 4 * guard, bits.data_ptr() + 8 * guard,
                                         ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert rc == 0, capi.last_error()
    v = v0
    for wt, (a, b) in zip(ws, ab):
        v = (a * dab.bconv_3x3(dab.pack_mat(v), wt, 1, 1) + b) + v
    s = (0.0 + v[:, 0::2, 0::2]) + v[:, 0::2, 1::2]
    s = ((s + v[:, 1::2, 0::2]) + v[:, 1::2, 1::2]) * 0.25
    assert same(pooled[guard:-guard].view_as(s), s)
    assert torch.equal(bits[guard:-guard].view(n, h, w, 1), dab.pack_mat(v))
    assert bool((pooled[:guard] == -5).all()) and bool((pooled[-guard:] == -5).all()) and bool((bits[:guard] == -5).all()) and bool((bits[-guard:] == -5).all())


def test_bireal18_reads_the_pooled_blob():
    """At 20 images the first stage's second pass writes its result pooled; the result, the branch and the blob inside the pass are made for who
    asks, at any time, and stay what the layers say."""
    from dabnn_amd import dab_format, models, net
    from oracle import net as orc_net
    layers, inits, inputs = models.bireal18(4)
    n = net.Net(batch=20).read_buf(dab_format.write_model(layers, inits, inputs))
    assert sum("written pooled 2x2" in d for d in n.layers()) == 1
    gone = {"conv1_out", "conv1_out_bn"} | {"s%db0_sc_pool_out" % s for s in (2, 3, 4)}
    r = np.random.default_rng(6)
    for run in range(5):
        n.run(r.standard_normal((20, 224, 224, 3)).astype(np.float32))
        if run == 3:
            n.get_blob("s1b3_out")
    i = 13
    for name, first_type, want in orc_net.run_segments(layers, inits, lambda b: n.get_blob(b)[i], gone):
        got = n.get_blob(name)[i]
        if first_type == "BinConv2D":
            np.testing.assert_array_equal(got, want, err_msg=name)
        else:
            np.testing.assert_allclose(got, want, rtol=1e-4, atol=1e-4 * np.abs(want).max(), err_msg=name)
    n.close()
