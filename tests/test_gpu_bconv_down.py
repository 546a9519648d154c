"""dab_bconv3x3_down: the first layer of a down-sampling block with its shortcut branch in one launch.  Given the branch's values, counts,
Affine, Add and sign bits are bit for bit the separate calls'; the branch's fp32 sums are compared with 64-bit ones and, bit for bit, with
dab_ave_pool2_fconv1x1's."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    import torch
    import dabnn_amd as dab
    from dabnn_amd import capi
    return torch, dab, capi


def ptr(t):
    return ctypes.c_void_p(0 if t is None else t.data_ptr())


def down(gpu, x, packed, w, coef, sw, bias, branch, cout, sign=True, want_branch=True, pooled=None):
    torch, dab, capi = gpu
    n, h, wd, cin = x.shape
    out = torch.full((n, h // 2, wd // 2, cout), 7.0, device="cuda")
    sc = torch.full_like(out, 7.0) if want_branch else None
    bits = torch.zeros((n, h // 2, wd // 2, cout // 64), dtype=torch.int64, device="cuda") if sign else None
    rc = capi.lib.dab_bconv3x3_down(ptr(packed), ptr(x if pooled is None else pooled), pooled is not None, n, h, wd, cin, ptr(w), ptr(coef[0]), ptr(coef[1]), cout, ptr(sw), ptr(bias), ptr(branch[0]),
                                    ptr(branch[1]), ptr(sc), ptr(out), ptr(bits), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert rc == 0, capi.lib.dab_last_error()
    return out, sc, bits


def problem(gpu, n, h, w, cin, cout, seed, scale=None):
    torch, dab, _ = gpu
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randn((n, h, w, cin), device="cuda", generator=g)
    wt = torch.randint(-2**63, 2**63 - 1, (cout, 9 * cin // 64), dtype=torch.int64, device="cuda", generator=g)
    v = [torch.randn(cout, device="cuda", generator=g) * 0.1 for _ in range(5)]
    sw = torch.randn((cout, cin), device="cuda", generator=g) / cin ** 0.5
    return x, wt, v, sw


def check(gpu, x, wt, v, sw, cout, with_bias, with_affine, special=False):
    torch, dab, capi = gpu
    packed = dab.pack_mat(x)
    bias, branch = (v[4] if with_bias else None), ((v[2], v[3]) if with_affine else (None, None))
    out, sc, bits = down(gpu, x, packed, wt, v, sw, bias, branch, cout)
    # the branch: pooled in fp32 as the layer does, summed in 64 bits, rounded like the layers behind the sum
    s = x[:, 0::2, 0::2] + x[:, 0::2, 1::2]
    s = (s + x[:, 1::2, 0::2] + x[:, 1::2, 1::2]) * 0.25
    pooled = s.reshape(-1, x.shape[3]).double()
    exact = pooled @ sw.double().T
    size = pooled.abs() @ sw.double().abs().T
    if with_bias:
        exact, size = exact + v[4].double(), size + v[4].double().abs()
    if with_affine:
        exact, size = exact * v[2].double() + v[3].double(), size * v[2].double().abs() + v[3].double().abs()
    got = sc.reshape(exact.shape).double()
    if special:
        finite = torch.isfinite(exact)
        assert torch.equal(torch.isnan(got), torch.isnan(exact)) and torch.equal(got[~finite & ~torch.isnan(exact)], exact[~finite & ~torch.isnan(exact)])
        got, exact, size = got[finite], exact[finite], size[finite]
    # an fp32 sum of K products in any order: at most K roundings of partial sums of no more than `size`, and four behind it
    assert bool(((got - exact).abs() <= (x.shape[3] + 8) * 2.0 ** -24 * size + 1e-42).all())
    # everything else to the bit
    cnt = dab.bconv_3x3(packed, wt, 2, 1)
    want = (v[0] * cnt + v[1]) + sc
    assert torch.equal(out.nan_to_num(nan=5e37), want.nan_to_num(nan=5e37))
    assert torch.equal(bits, dab.pack_mat(out))
    # without the outputs that may be left out: the same result
    again, _, _ = down(gpu, x, packed, wt, v, sw, bias, branch, cout, sign=False, want_branch=False)
    assert torch.equal(again.nan_to_num(nan=5e37), out.nan_to_num(nan=5e37))
    # from the pooled tensor: its values, and the same bounds (the kernel for few pieces does not take it)
    out, sc, bits = down(gpu, x, packed, wt, v, sw, bias, branch, cout, pooled=s)
    pgot = sc.reshape(-1, cout).double()
    pgot = pgot[finite] if special else pgot
    assert bool(((pgot - exact).abs() <= (x.shape[3] + 8) * 2.0 ** -24 * size + 1e-42).all())
    assert torch.equal(out.nan_to_num(nan=5e37), ((v[0] * cnt + v[1]) + sc).nan_to_num(nan=5e37)) and torch.equal(bits, dab.pack_mat(out))
    rel = ((got - exact).norm() / exact.norm()).item()
    return rel


# (images, h, w, cin, cout): 16 x 16 and 32 x 32 tiles, 128-channel tiles, walking blocks; last tiles of 1 to 31 pixels, channel
# blocks that the output does not fill, both sides of every switch, a single pixel
SHAPES = [(1, 2, 2, 64, 64), (1, 2, 2, 256, 64), (3, 6, 10, 64, 128), (1, 28, 28, 128, 256), (2, 14, 14, 256, 512), (1, 30, 34, 128, 320), (5, 14, 18, 128, 64),
          (7, 14, 14, 256, 192), (4, 26, 30, 64, 192), (6, 56, 56, 64, 128), (9, 28, 28, 128, 256), (11, 26, 22, 256, 320), (9, 56, 56, 64, 128),
          (11, 30, 34, 64, 448), (17, 28, 30, 128, 192), (16, 14, 14, 256, 512), (33, 14, 18, 256, 192), (40, 56, 56, 64, 128), (29, 50, 46, 64, 192),
          (60, 28, 28, 128, 256), (67, 30, 26, 128, 320), (61, 28, 30, 128, 512)]


@pytest.mark.parametrize("n,h,w,cin,cout", SHAPES)
def test_given_the_branch_the_rest_is_exact(gpu, n, h, w, cin, cout):
    x, wt, v, sw = problem(gpu, n, h, w, cin, cout, n * h + cin)
    flags = n % 4
    check(gpu, x, wt, v, sw, cout, flags & 1, flags < 2)
    check(gpu, x, wt, v, sw, cout, not flags & 1, flags >= 2)


@pytest.mark.parametrize("n,h,w,cin,cout", [(2, 14, 14, 128, 128), (16, 28, 28, 128, 256), (60, 28, 28, 128, 256), (40, 56, 56, 64, 128), (16, 14, 14, 256, 512)])
@pytest.mark.parametrize("what", ["inf", "nan", "tiny", "inf filter", "tiny filter", "zero"])
def test_infinities_nans_and_tiny_values(gpu, n, h, w, cin, cout, what):
    torch, _, _ = gpu
    x, wt, v, sw = problem(gpu, n, h, w, cin, cout, 3)
    r = np.random.default_rng(n)
    where = [(int(r.integers(n)), int(r.integers(h)), int(r.integers(w)), int(r.integers(cin))) for _ in range(40)]
    if what == "inf":
        for i, at in enumerate(where):
            x[at] = float("inf") if i % 2 else -float("inf")
    elif what == "nan":
        for at in where:
            x[at] = float("nan")
    elif what == "tiny":
        x[n // 2] *= 2.0 ** -118
    elif what == "inf filter":
        sw[5, 7] = float("inf")
        sw[cout - 1, 0] = -float("inf")
    elif what == "tiny filter":
        sw[3:37] *= 2.0 ** -115
        x[0] *= 2.0 ** 60
    else:
        x[:, :, :, ::3] = 0.0
        sw[:, 1::2] = 0.0
    check(gpu, x, wt, v, sw, cout, False, what.startswith("tiny"), special=True)


@pytest.mark.parametrize("n,h,cin,cout", [(40, 56, 64, 128), (100, 56, 64, 128), (100, 28, 128, 256), (16, 28, 128, 256), (6, 14, 256, 512), (1, 56, 64, 128)])
def test_no_further_from_64_bits_than_the_separate_launch(gpu, n, h, cin, cout):
    """Normally distributed operands: relative error (2-norm) of the branch, and that of dab_ave_pool2_fconv1x1."""
    torch, dab, capi = gpu
    x, wt, v, sw = problem(gpu, n, h, h, cin, cout, 11)
    rel = check(gpu, x, wt, v, sw, cout, False, False)
    out = torch.empty((n, h // 2, h // 2, cout), device="cuda")
    rc = capi.lib.dab_ave_pool2_fconv1x1(ptr(x), n, h, h, cin, ptr(sw), None, None, None, 0, cout, None, ptr(out), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert rc == 0
    s = x[:, 0::2, 0::2] + x[:, 0::2, 1::2]
    s = (s + x[:, 1::2, 0::2] + x[:, 1::2, 1::2]) * 0.25
    exact = s.reshape(-1, cin).double() @ sw.double().T
    before = ((out.reshape(exact.shape).double() - exact).norm() / exact.norm()).item()
    print("relative error %.3g, separate launch %.3g" % (rel, before))
    assert rel <= 1.02 * before


# more than eight pooled pixels (fewer go to a matrix-vector kernel in the separate launch), and the sizes around which that launch
# splits the depth over its waves and those at which this one changes its tiles
BRANCH_SHAPES = [s for s in SHAPES if s[0] * s[1] * s[2] > 32] + [
    (3, 2, 6, 64, 64), (11, 28, 28, 128, 256), (15, 28, 28, 128, 256), (21, 14, 14, 256, 512), (30, 14, 14, 256, 512), (7, 56, 56, 64, 128), (10, 48, 48, 64, 128),
    (1, 128, 190, 64, 128), (1, 156, 156, 64, 128), (1, 128, 254, 64, 64), (1, 144, 226, 64, 64), (1, 126, 128, 128, 192), (1, 128, 128, 128, 192),
    (1, 8, 8, 64, 12288), (1, 8, 8, 256, 12224), (256, 14, 14, 256, 512)]
# blocks that walk over pixel tiles, from 780 tiles on: either side of that, last tiles of 1 to 31 pixels, channel blocks that are not full
WALK_SHAPES = [(1, 312, 320, 64, 64), (1, 310, 320, 64, 64), (45, 50, 46, 64, 192), (33, 56, 56, 64, 320), (1, 2, 50562, 64, 128), (1, 320, 312, 128, 64),
               (131, 30, 26, 128, 320), (128, 28, 28, 128, 256), (515, 14, 14, 128, 448)]
BRANCH_SHAPES += WALK_SHAPES


@pytest.mark.parametrize("n,h,w,cin,cout", WALK_SHAPES)
@pytest.mark.parametrize("with_bias,with_affine", [(False, True), (True, True), (False, False)])
def test_walking_blocks(gpu, n, h, w, cin, cout, with_bias, with_affine):
    x, wt, v, sw = problem(gpu, n, h, w, cin, cout, n + cout)
    r = np.random.default_rng(n)
    for value in (float("inf"), -float("inf"), float("nan")):
        x[int(r.integers(n)), int(r.integers(h)), int(r.integers(w)), int(r.integers(cin))] = value
    check(gpu, x, wt, v, sw, cout, with_bias, with_affine, special=True)


@pytest.mark.parametrize("n,h,w,cin,cout", BRANCH_SHAPES)
def test_branch_is_the_separate_launchs_to_the_bit(gpu, n, h, w, cin, cout):
    """The sums of dab_ave_pool2_fconv1x1, in its order, from the whole and from the pooled tensor."""
    torch, dab, capi = gpu
    x, wt, v, sw = problem(gpu, n, h, w, cin, cout, n + h + cin)
    packed = dab.pack_mat(x)
    pooled, want = torch.empty((n, h // 2, w // 2, cin), device="cuda"), torch.empty((n, h // 2, w // 2, cout), device="cuda")
    for bias, branch in ((v[4], (v[2], v[3])), (None, (None, None))):
        rc = capi.lib.dab_ave_pool2_fconv1x1(ptr(x), n, h, w, cin, ptr(sw), ptr(bias), ptr(branch[0]), ptr(branch[1]), 0, cout, ptr(pooled), ptr(want),
                                             ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
        assert rc == 0, capi.lib.dab_last_error()
        for given in (None, pooled):
            _, got, _ = down(gpu, x, packed, wt, v, sw, bias, branch, cout, pooled=given)
            differ = (got.view(torch.int32) != want.view(torch.int32)).float().mean().item()
            assert differ == 0, "%.3g of the values differ, %s" % (differ, "pooled" if given is not None else "whole")


def block_net(models, n_in, cout, hw, seed=0, relu=False, second_reader=False):
    """1x1 convolution to n_in channels -> down-sampling block -> binary convolution -> classifier."""
    r = np.random.default_rng(seed)
    layers, inits = [], []

    def tensor(name, data, shape=None, align=False):
        inits.append({"name": name, "shape": list(data.shape if shape is None else shape), "data": data, "align_hwc_to_128": align})
        return name

    def fconv(name, src, dst, cin, co, k):
        layers.append({"type": "FpConv2D", "name": name, "input": src, "weight": tensor(name + "_w", (r.standard_normal((co, k, k, cin)) / np.sqrt(k * k * cin)).astype(np.float32)),
                       "output": dst, "pads": [k // 2] * 4, "strides": [1, 1], "dilations": [1, 1]})

    def bconv(name, src, cin, co, stride):
        wf = r.standard_normal((co, 3, 3, cin)).astype(np.float32)
        layers.append({"type": "BinConv2D", "name": name, "input": src, "weight": tensor(name + "_w", models.pack_weight(wf).ravel(), shape=[co, 3, 3, cin], align=cin != 64),
                       "output": name + "_cnt", "pads": [1] * 4, "strides": [stride, stride], "dilations": [1, 1]})
        a, b = models.fold_bn(np.full(co, 0.5, np.float32), (0.1 * r.standard_normal(co)).astype(np.float32), np.zeros(co, np.float32),
                              np.full(co, 9.0 * cin, np.float32), 1e-5, 9 * cin)
        layers.append({"type": "Affine", "name": name + "_affine", "input": name + "_cnt", "a": tensor(name + "_a", a), "b": tensor(name + "_b", b), "output": name + "_bn"})

    fconv("stem", "data", "s", 3, n_in, 3)
    bconv("b0", "s", n_in, cout, 2)
    layers.append({"type": "AvePool", "name": "sc_pool", "input": "s", "output": "sc_pool_out", "kernel_shape": [2, 2], "pads": [0] * 4, "strides": [2, 2]})
    fconv("sc", "sc_pool_out", "sc_out", n_in, cout, 1)
    layers.append({"type": "Affine", "name": "sc_affine", "input": "sc_out", "a": tensor("sc_a", (1 + 0.1 * r.standard_normal(cout)).astype(np.float32)),
                   "b": tensor("sc_b", (0.1 * r.standard_normal(cout)).astype(np.float32)), "output": "sc_bn"})
    layers.append({"type": "Add", "name": "add", "input1": "b0_bn", "input2": "sc_bn", "output": "b0_out"})
    cur = "b0_out"
    if relu:  # rewrites what the pass writes
        layers.append({"type": "Relu", "name": "relu", "input": cur, "output": "b0_relu"})
        cur = "b0_relu"
    if second_reader:
        layers.append({"type": "MaxPool", "name": "peek", "input": "sc_bn", "output": "peek_out", "kernel_shape": [2, 2], "pads": [0] * 4, "strides": [2, 2]})
    bconv("b1", cur, cout, 64, 1)
    layers.append({"type": "AvePool", "name": "gap", "input": "b1_bn", "output": "gap_out", "kernel_shape": [hw // 2, hw // 2], "pads": [0] * 4, "strides": [1, 1]})
    fconv("fc", "gap_out", "logits", 64, 10, 1)
    return layers, inits, [("data", [1, hw, hw, 3])]


@pytest.mark.parametrize("cin,cout,hw,batch,inside", [(64, 128, 16, 1, True), (128, 256, 12, 3, True), (64, 128, 56, 20, True), (256, 192, 14, 33, True),
                                                      (128, 128, 28, 60, True), (256, 512, 14, 190, True), (64, 64, 4, 1, False)])
def test_net_every_blob_on_every_run(cin, cout, hw, batch, inside):
    from dabnn_amd import dab_format, models, net
    from oracle import net as orc_net
    layers, inits, inputs = block_net(models, cin, cout, hw)
    n = net.Net(batch=batch).read_buf(dab_format.write_model(layers, inits, inputs))
    assert any("its shortcut convolution in the same pass" in d for d in n.layers()) == inside, n.layers()
    gone = {"sc_pool_out"} if (hw // 2) ** 2 * batch > 8 else set()
    r = np.random.default_rng(batch)
    for run in range(6):
        n.run(r.standard_normal((batch, hw, hw, 3)).astype(np.float32))
        if run < 2:
            continue  # asked for from the captured run on
        i = (run * 7) % batch
        for name, first_type, want in orc_net.run_segments(layers, inits, lambda b: n.get_blob(b)[i], gone):
            got = n.get_blob(name)[i]
            if first_type == "BinConv2D":
                np.testing.assert_array_equal(got, want, err_msg=name)
            else:
                np.testing.assert_allclose(got, want, rtol=1e-4, atol=1e-4 * np.abs(want).max(), err_msg=name)
    n.close()


@pytest.mark.parametrize("kind", [{"relu": True}, {"second_reader": True}])
def test_net_keeps_the_branch_where_its_blobs_have_other_users(kind):
    from dabnn_amd import dab_format, models, net
    layers, inits, inputs = block_net(models, 64, 128, 16, **kind)
    n = net.Net(batch=2).read_buf(dab_format.write_model(layers, inits, inputs))
    assert not any("its shortcut convolution in the same pass" in d for d in n.layers())
    n.close()
