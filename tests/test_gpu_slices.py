"""Float convolutions with PRelu, sign bits and a result that is a slice of a wider tensor, and nets whose Concats copy
nothing: against the separate layers, bit for bit (the sums are the same tiles', and every step rounds alike)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,h,w,c,cout,k,stride,pad,bias,affine,slopes", [
    (33, 32, 32, 3, 64, 3, 1, 1, False, True, 64),       # 128 x 64 tiles, element loader, the last tile not full
    (128, 16, 17, 256, 128, 1, 1, 0, False, True, 1),    # 128 x 128 tiles
    (4, 112, 113, 3, 64, 7, 2, 3, True, True, 64),       # three-channel loader
    (130, 16, 16, 12, 40, 3, 1, 1, True, False, 40),     # 64 channels a tile for 40, no sign bits
    (8, 40, 40, 16, 32, 3, 1, 1, False, False, 1),       # (c32 shapes aside) 32 channels
    (24, 16, 16, 128, 128, 1, 1, 0, False, True, 128),   # 64 x 128 tiles and smaller
    (9, 16, 16, 64, 192, 1, 1, 0, True, True, 192),
    (2, 9, 7, 64, 128, 1, 1, 0, False, True, 1),         # 32 x 32 tiles, the depth split over the waves
    (1, 12, 11, 5, 64, 3, 1, 1, True, True, 64),
    (1, 3, 3, 64, 64, 1, 1, 0, False, False, 64),
    (5, 20, 20, 32, 64, 3, 1, 1, False, True, 64),
])
def test_fconv_prelu_into_a_slice(n, h, w, c, cout, k, stride, pad, bias, affine, slopes):
    import dabnn_amd as dab
    from dabnn_amd import capi
    gen = torch.Generator(device="cuda").manual_seed(n + h + cout)

    def normal(*shape):
        return torch.randn(shape, device="cuda", generator=gen)

    x, wgt, slope = normal(n, h, w, c), normal(cout, k, k, c), normal(slopes)
    bs, a, b = normal(cout) if bias else None, normal(cout) if affine else None, normal(cout) if affine else None
    want = dab.fconv_affine_relu(x, wgt, bs, a, b, False, k, k, pad, pad, stride, stride)
    want = torch.where(want < 0, want * slope, want)
    oh, ow = want.shape[1:3]
    ld, first = cout + 72, 8
    wide = torch.full((n, oh, ow, ld), 7.0, device="cuda")
    sign = cout % 64 == 0
    bits_ld = cout // 64 + 2
    bits = torch.full((n, oh, ow, bits_ld), 5, dtype=torch.int64, device="cuda")

    def ptr(t):
        return None if t is None else t.data_ptr()

    capi.check(capi.lib.dab_fconv_affine_prelu(
        ptr(x), n, h, w, c, ptr(wgt), ptr(bs), ptr(a), ptr(b), ptr(slope), slopes, k, k, pad, pad, stride, stride, 1, 1, cout,
        wide.data_ptr() + 4 * first, ld, bits.data_ptr() + 8 if sign else None, bits_ld if sign else 0, None))
    torch.cuda.synchronize()
    assert torch.equal(wide[..., first:first + cout], want)
    assert (wide[..., :first] == 7).all() and (wide[..., first + cout:] == 7).all()
    if sign:
        assert torch.equal(bits[..., 1:1 + cout // 64], dab.pack_mat(want.contiguous()).reshape(n, oh, ow, -1))
        assert (bits[..., 0] == 5).all() and (bits[..., -1] == 5).all()


def random_net(seed):
    """A graph of binary and float convolutions, Concats of any two blobs of a size, Adds, pools and in-place layers: the
    Concats that can be stored in place and all the ways in which one cannot."""
    from dabnn_amd import models
    r = np.random.default_rng(seed)
    hw = int(r.integers(5, 12))
    layers, inits = [], []

    def tensor(data, shape=None, align=False):
        inits.append({"name": "t%d" % len(inits), "shape": list(data.shape if shape is None else shape), "data": data, "align_hwc_to_128": align})
        return inits[-1]["name"]

    blobs = {"data": 64}  # name of the newest in-place version -> channels
    names = ["data"]

    def new(name, c):
        blobs[name] = c
        names.append(name)
        return name

    def in_place(kind, old, **more):
        layers.append(dict({"type": kind, "name": "%s%d" % (kind, len(layers)), "input": old, "output": "%s_%d" % (old, len(layers))}, **more))
        blobs[layers[-1]["output"]] = blobs.pop(old)
        return layers[-1]["output"]

    def affine_prelu(name, c):
        name = in_place("Affine", name, a=tensor(r.uniform(-0.2, 0.2, c).astype(np.float32)), b=tensor(r.standard_normal(c).astype(np.float32)))
        if r.random() < 0.4:
            name = in_place("PRelu", name, slope=tensor(r.uniform(0.1, 0.4, c if r.random() < 0.5 else 1).astype(np.float32)))
        return name

    for step in range(12):
        pick = list(blobs)
        src = pick[int(r.integers(max(0, len(pick) - 3), len(pick)))] if r.random() < 0.8 else pick[int(r.integers(0, len(pick)))]
        c = blobs[src]
        kind = r.choice(["bin", "float", "concat", "grow", "add", "relu", "pool"], p=[.15, .15, .15, .4, .05, .05, .05]) if step else "float"
        if kind == "grow":  # what a dense block does: 64 new channels behind the ones they were made from
            src, kind = pick[-1], "bin"
            c, grow = blobs[src], True
        else:
            grow = False
        if kind == "bin" and c % 64 == 0:
            cout, k = int(r.choice([64] if grow else [64, 64, 128, 32, 24])), int(r.choice([1, 3, 3]))
            wf = r.standard_normal((cout, k, k, c)).astype(np.float32)
            layers.append({"type": "BinConv2D", "name": "bin%d" % step, "input": src, "weight": tensor(models.pack_weight(wf).ravel(), [cout, k, k, c], c != 64),
                           "output": new("bin%d_out" % step, cout), "pads": [k // 2] * 4, "strides": [1, 1], "dilations": [1, 1]})
            out = "bin%d_out" % step
            if grow or r.random() < 0.9:
                out = affine_prelu(out, cout) if r.random() < 0.2 else in_place(
                    "Affine", out, a=tensor(np.full(cout, -0.1, np.float32)), b=tensor((0.05 * 9 * c + r.standard_normal(cout)).astype(np.float32)))
            if grow and blobs[src] + cout <= 512:
                layers.append({"type": "Concat", "name": "concat%d" % step, "inputs": [src, out] if r.random() < 0.8 else [out, src], "axis": 3,
                               "output": new("concat%d_out" % step, c + cout)})
        elif kind == "float":
            cout, k = int(r.choice([64, 64, 128, 32])), int(r.choice([1, 3]))
            layers.append({"type": "FpConv2D", "name": "float%d" % step, "input": src, "weight": tensor((r.standard_normal((cout, k, k, c)) / np.sqrt(k * k * c)).astype(np.float32)),
                           "output": new("float%d_out" % step, cout), "pads": [k // 2] * 4, "strides": [1, 1], "dilations": [1, 1]})
            affine_prelu("float%d_out" % step, cout)
        elif kind == "concat":
            other = pick[int(r.integers(0, len(pick)))] if r.random() < 0.3 else pick[-1]
            if blobs[src] + blobs[other] <= 512:
                layers.append({"type": "Concat", "name": "concat%d" % step, "inputs": [src, other], "axis": 3,
                               "output": new("concat%d_out" % step, c + blobs[other])})
        elif kind == "add":
            other = [b for b in pick if blobs[b] == c and b != src]
            if other and src != "data":
                layers.append({"type": "Add", "name": "add%d" % step, "input1": src, "input2": other[-1], "output": "add%d_out" % step})
                blobs["add%d_out" % step] = blobs.pop(src)
        elif kind == "relu" and src != "data":
            in_place("Relu", src)
        elif kind == "pool":
            layers.append({"type": "MaxPool", "name": "pool%d" % step, "input": src, "output": new("pool%d_out" % step, c), "kernel_shape": [3, 3],
                           "pads": [1] * 4, "strides": [1, 1]})
    return layers, inits, [("data", [1, hw, hw, 64])], [b for b in blobs if b != "data"]


@pytest.mark.parametrize("seed", range(40))
def test_concats_in_place_leave_every_blob_as_it_was(seed):
    from dabnn_amd import dab_format, net
    layers, inits, inputs, blobs = random_net(seed)
    buf = dab_format.write_model(layers, inits, inputs)
    batch = 1 + seed % 3
    shape = [batch] + inputs[0][1][1:]
    x = np.random.default_rng(seed).standard_normal(shape).astype(np.float32)
    plain = net.Net(batch=batch, optimize=False).read_buf(buf)
    plain.run(x)
    fused = net.Net(batch=batch).read_buf(buf)
    for run in range(4):  # the last two from the HIP graph
        fused.run(x if run != 2 else -x)
        if run == 2:
            continue
        for b in blobs:
            np.testing.assert_array_equal(fused.get_blob(b), plain.get_blob(b), err_msg="seed %d %s run %d" % (seed, b, run))
    for layer in layers:
        if layer["type"] == "BinConv2D" and any("DIRECT" in d for d in fused.layers()):
            fused.get_blob("binaized_for_%s_cal" % layer["output"])
    plain.close()
    fused.close()


def test_most_dense_forms_are_stored_in_place():
    """The graphs above hold both kinds; a dense block holds only the kind that copies nothing."""
    from dabnn_amd import dab_format, models, net
    n = net.Net(batch=2).read_buf(dab_format.write_model(*models.dense_bnn(1, hw=12)))
    descs = [d for d in n.layers() if d.startswith("Concat")]
    assert len(descs) == 5 and all("in place" in d for d in descs), descs
    n.close()
    counts = {True: 0, False: 0}
    for seed in range(40):
        layers, inits, inputs, _ = random_net(seed)
        n = net.Net().read_buf(dab_format.write_model(layers, inits, inputs))
        for d in n.layers():
            if d.startswith("Concat"):
                counts["in place" in d] += 1
        n.close()
    assert counts[True] > 10 and counts[False] > 10, counts
