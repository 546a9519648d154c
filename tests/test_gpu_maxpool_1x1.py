"""MaxPool 2x2 inside the 1x1 convolution behind it: the kernel against the two calls, bit for bit, infinities and NaNs included; nets
that use it, with the pooled blob asked for before, between and after runs."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,h,w,c,cout,slopes,relu,extra,first,special", [
    (64, 32, 32, 256, 128, 1, False, 128, 64, False), (70, 33, 31, 256, 192, 192, False, 5, 3, False), (60, 45, 52, 128, 128, 0, True, 0, 0, True),
    (17, 90, 91, 128, 256, 0, False, 0, 0, False), (30, 61, 59, 192, 64, 64, False, 64, 64, True), (9, 100, 100, 192, 320, 0, True, 0, 0, False),
    (33, 91, 92, 64, 96, 0, True, 0, 0, False), (70, 64, 62, 64, 320, 1, False, 64, 0, True), (8, 64, 64, 256, 512, 0, False, 0, 0, True), (20, 32, 32, 256, 256, 256, False, 64, 64, True),
])
def test_against_the_two_calls(n, h, w, c, cout, slopes, relu, extra, first, special):
    import dabnn_amd as dab
    from dabnn_amd import capi
    gen = torch.Generator(device="cuda").manual_seed(n + h)

    def normal(*shape):
        return torch.randn(shape, device="cuda", generator=gen)

    assert capi.lib.dab_max_pool2_fconv1x1_takes(n, h, w, c, cout) == 1
    x, wgt, bias, a, b = normal(n, h, w, c), normal(cout, 1, 1, c), normal(cout), normal(cout), normal(cout)
    if special:
        x[0, 2, 3, 5], x[1, 4:6, 6:8, 7], x[2, 0, 0, 1], x[3] = float("inf"), float("-inf"), float("nan"), x[3] * 2.0**-120
        x[4, :, :, ::2] *= 2.0**-60
    want = dab.fconv_affine_relu(dab.max_pool(x, 2, 2, 0, 0, 2, 2), wgt, bias, a, b, relu, 1, 1, 0, 0, 1, 1)
    slope = normal(slopes) if slopes else None
    if slopes:
        want = torch.where(want < 0, want * slope, want)
    oh, ow = want.shape[1:3]
    wide = torch.full((n, oh, ow, cout + extra), 7.0, device="cuda")
    sign = cout % 64 == 0
    bits = torch.full((n, oh, ow, cout // 64 + 2), 5, dtype=torch.int64, device="cuda")
    capi.check(capi.lib.dab_max_pool2_fconv1x1(
        x.data_ptr(), n, h, w, c, wgt.data_ptr(), bias.data_ptr(), a.data_ptr(), b.data_ptr(), int(relu), slope.data_ptr() if slopes else None, slopes, cout,
        wide.data_ptr() + 4 * first, cout + extra, bits.data_ptr() + 8 if sign else None, cout // 64 + 2 if sign else 0, None))
    torch.cuda.synchronize()
    assert torch.equal(wide[..., first:first + cout].view(torch.int32), want.view(torch.int32))
    assert (wide[..., :first] == 7).all() and (wide[..., first + cout:] == 7).all()
    if sign:
        assert torch.equal(bits[..., 1:-1], dab.pack_mat(want.contiguous()).reshape(n, oh, ow, -1))
        assert (bits[..., 0] == 5).all() and (bits[..., -1] == 5).all()


def test_what_it_refuses():
    import dabnn_amd as dab
    from dabnn_amd import capi
    for shape in [(39, 32, 32, 256, 128), (64, 32, 32, 320, 128), (64, 32, 32, 256, 32), (64, 32, 32, 256, 136), (64, 1, 64, 256, 128)]:
        assert capi.lib.dab_max_pool2_fconv1x1_takes(*shape) == 0
    x, wgt, out = (torch.zeros(s, device="cuda") for s in [(64, 32, 32, 256), (128, 256), (64, 16, 16, 128)])

    def call(x_at, n, slopes, ld):
        return capi.lib.dab_max_pool2_fconv1x1(x_at, n, 32, 32, 256, wgt.data_ptr(), None, None, None, 0, wgt.data_ptr() if slopes else None, slopes, 128,
                                               out.data_ptr(), ld, None, 0, None)

    assert call(x.data_ptr(), 39, 0, 128) == capi.DAB_EUNSUPPORTED
    assert call(x.data_ptr() + 4, 63, 0, 128) == capi.DAB_EUNSUPPORTED
    assert call(x.data_ptr(), 64, 3, 128) == capi.DAB_EINVAL
    assert call(x.data_ptr(), 64, 0, 127) == capi.DAB_EINVAL


@pytest.mark.parametrize("batch,hw,inside", [(40, 32, True), (39, 32, False)])
@pytest.mark.parametrize("asked", [0, 1, 4])
def test_net(batch, hw, inside, asked):
    from dabnn_amd import dab_format, models, net
    model = models.dense_bnn(3, hw=hw)
    buf = dab_format.write_model(*model)
    n, plain = net.Net(batch=batch).read_buf(buf), net.Net(batch=batch, optimize=False).read_buf(buf)
    assert any("MaxPool 2x2 of" in d for d in n.layers()) == inside
    source = next(l["input"] for l in model[0] if l["name"] == "t1_pool")
    r = np.random.default_rng(batch + asked)
    for run in range(6):
        if run == asked:
            n.get_blob("t1_pool_out")
        x = r.standard_normal((batch, hw, hw, 3)).astype(np.float32)
        n.run(x)
        plain.run(x)
        got, want = n.get_blob("logits"), plain.get_blob("logits")
        np.testing.assert_allclose(got, want, rtol=1e-4, atol=1e-4 * np.abs(want).max())
        if run >= asked:
            whole = n.get_blob(source).reshape(batch, hw // 2, 2, hw // 2, 2, -1)
            np.testing.assert_array_equal(n.get_blob("t1_pool_out"), whole.max(axis=(2, 4)))
    n.close()
    plain.close()
