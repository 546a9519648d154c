"""The work whose speed this framework is judged by: whole networks through ``dabnn_amd.net.Net`` and the reference's
operators through ``dabnn_amd.ops``, each as a user's program calls them.

``listed()`` names the cases, ``draw(rng)`` gives another one of the same ranges, ``prepare(case, seed)`` makes what the
program holds before the call, ``run(state)`` is one pass, ``work(case)`` the bytes and operations no implementation
can do without and ``tolerance(case)`` how far two correct implementations may be apart.

Kinds of case
  net      Bi-Real-18 at 224 x 224 (``models.bireal18``), input on the host or on the device, logits to the host
  dense    a BiDenseNet-style net (``models.dense_bnn``): Concat, PRelu, 192-channel layers through im2col + bgemm
  stages   the seven 3x3 binary convolutions of the ResNet-18 stages on packed input, raw counts
  block    one binary convolution with Affine (+ Add) and the next layer's packed input
  layer    a BinConv layer from fp32 input
  bgemm    the xor/popcount GEMM alone, adding to C or overwriting it
  pack     sign packing of an fp32 tensor
"""
import math

import numpy as np
import torch

import dabnn_amd as dab
from dabnn_amd import dab_format, models, net

# (height = width, input channels, output channels, stride)
STAGES = [(56, 64, 64, 1), (28, 128, 128, 1), (14, 256, 256, 1), (7, 512, 512, 1),
          (56, 64, 128, 2), (28, 128, 256, 2), (14, 256, 512, 2)]


def listed():
    return [
        # one photograph in host memory, logits back: how the reference is called on a phone, and the latency of a server
        {"name": "net_b1_host", "kind": "net", "batch": 1, "stem": False, "host": True},
        # a handful of images already on the GPU, three-convolution stem: a server that batches what has arrived
        {"name": "net_stem_b6", "kind": "net", "batch": 6, "stem": True, "host": False},
        # a mid-sized batch as an image loader hands it over, in host memory
        {"name": "net_b40_host", "kind": "net", "batch": 40, "stem": False, "host": True},
        # the stem variant at an odd, large batch
        {"name": "net_stem_b100", "kind": "net", "batch": 100, "stem": True, "host": False},
        # offline throughput: the largest batch that the framework's benchmark quotes
        {"name": "net_b256", "kind": "net", "batch": 256, "stem": False, "host": False},
        # the other graph family, on 32 x 32 images
        {"name": "dense_b128", "kind": "dense", "batch": 128, "hw": 32},
        # the benchmark's headline step: binary convolutions alone at batch 64
        {"name": "stages_b64", "kind": "stages", "batch": 64},
        # a residual block at a ragged size (81 x 27 x 29 pixels are no multiple of any tile)
        {"name": "block_ragged", "kind": "block", "n": 81, "h": 27, "w": 29, "cin": 128, "cout": 192, "stride": 1, "pad": 1,
         "shortcut": True, "sign": True},
        # a layer used on its own from fp32 activations, first stage, 3x3
        {"name": "layer_56x56x64_b16", "kind": "layer", "n": 16, "h": 56, "w": 56, "cin": 64, "cout": 64, "k": 3, "stride": 1, "pad": 1},
        # 5x5 filters, which only im2col + bgemm takes (a row of the reference's benchmark, over a batch)
        {"name": "layer_5x5_b8", "kind": "layer", "n": 8, "h": 14, "w": 14, "cin": 256, "cout": 256, "k": 5, "stride": 1, "pad": 2},
        # the reference's GEMM by itself
        {"name": "bgemm_512x3136", "kind": "bgemm", "m": 512, "n": 3136, "k": 72, "add": True},
        # the smallest call: one image's activations packed
        {"name": "pack_1x56x56x64", "kind": "pack", "n": 1, "h": 56, "w": 56, "c": 64},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["net", "net", "dense", "stages", "block", "layer", "layer", "bgemm", "pack"])
    if kind == "net":
        host = rng.random() < 0.5
        stem = rng.random() < 0.5
        return {"kind": kind, "batch": _log(rng, 1, 40 if host else 128 if stem else 256), "stem": stem, "host": host}
    if kind == "dense":
        return {"kind": kind, "batch": _log(rng, 1, 256), "hw": 2 * rng.randint(4, 16)}
    if kind == "stages":
        return {"kind": kind, "batch": 2 * _log(rng, 1, 128) - 1}
    if kind == "bgemm":
        return {"kind": kind, "m": _log(rng, 8, 1024), "n": _log(rng, 16, 20000), "k": _log(rng, 4, 160), "add": rng.random() < 0.5}
    h = _log(rng, 5, 60)
    w = max(4, h + rng.choice([0, 0, 0, -1, 2, 3]))
    if kind == "pack":
        c = 64 * rng.choice([1, 2, 3, 4, 8])
        return {"kind": kind, "n": _log(rng, 1, max(2, 100_000_000 // (h * w * c))), "h": h, "w": w, "c": c}
    cin = rng.choice([64, 128, 256, 512])
    stride = rng.choice([1, 1, 2])
    most = max(2, 40_000_000 // (h * w * 256))
    if kind == "block":
        return {"kind": kind, "n": _log(rng, 1, most), "h": h, "w": w, "cin": cin, "cout": 64 * rng.randint(1, 8), "stride": stride,
                "pad": 1, "shortcut": rng.random() < 0.7, "sign": rng.random() < 0.7}
    k = rng.choice([3, 3, 3, 1, 5])
    return {"kind": kind, "n": _log(rng, 1, most), "h": h, "w": w, "cin": rng.choice([cin, 64 * rng.randint(1, 8)]),
            "cout": 8 * _log(rng, 1, 64), "k": k, "stride": stride, "pad": k // 2}


def _out(size, k, stride, pad):
    return (size + 2 * pad - k) // stride + 1


def _words(gen, *shape):
    """Sign bits of activations and weights: both signs equally often."""
    return torch.randint(-2**63, 2**63 - 1, shape, dtype=torch.int64, device="cuda", generator=gen)


def _normal(gen, *shape):
    return torch.randn(shape, device="cuda", generator=gen)


def _affine(seed, cout, cin):
    """Coefficients as the converter folds them behind a binary convolution of 9 * cin bits."""
    r = np.random.default_rng(seed)
    a, b = models.fold_bn((0.5 + 0.05 * r.standard_normal(cout)).astype(np.float32), (0.1 * r.standard_normal(cout)).astype(np.float32),
                          np.zeros(cout, np.float32), np.full(cout, 9.0 * cin, np.float32), 1e-5, 9 * cin)
    return torch.from_numpy(a).cuda(), torch.from_numpy(b).cuda()


def prepare(case, seed):
    kind = case["kind"]
    gen = torch.Generator(device="cuda").manual_seed(seed)
    if kind in ("net", "dense"):
        if kind == "net":
            model = models.bireal18(seed, stem=case["stem"])
            shape = (case["batch"], 224, 224, 3)
        else:
            model = models.dense_bnn(seed, hw=case["hw"])
            shape = (case["batch"], case["hw"], case["hw"], 3)
        handle = net.Net(batch=case["batch"]).read_buf(dab_format.write_model(*model))
        x = _normal(gen, *shape)
        return kind, handle, x.cpu().numpy() if case.get("host") else x
    if kind == "stages":
        n = case["batch"]
        return kind, [(_words(gen, n, hw, hw, cin // 64), _words(gen, cout, 9 * cin // 64), stride) for hw, cin, cout, stride in STAGES]
    if kind == "bgemm":
        m, n, k = case["m"], case["n"], case["k"]
        c = torch.randint(0, 1000, (n, m), device="cuda", generator=gen).float()
        return kind, (dab.bgemm if case["add"] else dab.bgemm_overwrite), (m, n, k, _words(gen, k, m), m, _words(gen, n, k), k, c, m)
    if kind == "pack":
        return kind, _normal(gen, case["n"], case["h"], case["w"], case["c"])
    n, h, w, cin, cout, stride, pad = (case[key] for key in ("n", "h", "w", "cin", "cout", "stride", "pad"))
    if kind == "block":
        a, b = _affine(seed, cout, cin)
        shortcut = _normal(gen, n, _out(h, 3, stride, pad), _out(w, 3, stride, pad), cout) if case["shortcut"] else None
        fn = dab.bconv_3x3_affine_add_sign if case["sign"] else dab.bconv_3x3_affine_add
        return kind, fn, (_words(gen, n, h, w, cin // 64), _words(gen, cout, 9 * cin // 64), a, b, shortcut, stride, pad)
    k = case["k"]
    packed = models.pack_weight(np.random.default_rng(seed).standard_normal((cout, k, k, cin)).astype(np.float32))
    layer = dab.BinConv(torch.from_numpy(packed.view(np.int64)).cuda(), k, k, pad, pad, stride, stride)
    return kind, layer, _normal(gen, n, h, w, cin)


def run(state):
    kind = state[0]
    if kind in ("net", "dense"):
        _, handle, x = state
        handle.run(x)
        return handle.get_blob("logits")
    if kind == "stages":
        return [dab.bconv_3x3(x, w, stride, 1) for x, w, stride in state[1]]
    if kind == "pack":
        return dab.pack_mat(state[1])
    if kind == "layer":
        return state[1](state[2])
    return state[1](*state[2])  # block, bgemm


def _conv_work(n, h, w, cin, cout, k, stride, pad, in_bytes, out_bytes):
    """Bytes in and out and operations of a convolution, filters of one bit per weight."""
    pixels = n * _out(h, k, stride, pad) * _out(w, k, stride, pad)
    return (n * h * w * cin * in_bytes + cout * k * k * cin / 8 + pixels * cout * out_bytes, 2.0 * pixels * cout * k * k * cin)


def work(case):
    """Binary operations count as the 2 per weight and output that the same float convolution would have."""
    kind = case["kind"]
    if kind == "net":
        n = case["batch"]
        binary = sum(2.0 * _out(hw, 3, s, 1) ** 2 * cout * 9 * cin for hw, cin, cout, s in STAGES)
        binary += sum(2 * 2.0 * hw * hw * c * 9 * c for hw, c in ((56, 64), (28, 128), (14, 256), (7, 512)))
        binary += 2.0 * 56 * 56 * 64 * 9 * 64  # the first stage has a fourth block at stride 1
        stem = 2.0 * 112 * 112 * (32 * 27 + 32 * 288 + 64 * 288) if case["stem"] else 2.0 * 112 * 112 * 64 * 147
        shortcuts = 2.0 * (28 * 28 * 128 * 64 + 14 * 14 * 256 * 128 + 7 * 7 * 512 * 256)
        return {"bytes": n * (224 * 224 * 3 + 1000) * 4.0 + 4.2e6, "flops": n * (binary + stem + shortcuts + 2.0 * 512 * 1000)}
    if kind == "dense":
        n, hw, half = case["batch"], case["hw"], case["hw"] // 2
        macs = hw * hw * (64 * 27 + 9 * 64 * (64 + 128 + 192)) + half * half * (256 * 128 + 9 * 64 * (128 + 192)) + 256 * 10
        return {"bytes": n * (hw * hw * 3 + 10) * 4.0 + 2.5e5, "flops": 2.0 * n * macs}
    if kind == "stages":
        each = [_conv_work(case["batch"], hw, hw, cin, cout, 3, stride, 1, 1 / 8, 4) for hw, cin, cout, stride in STAGES]
        return {"bytes": sum(b for b, _ in each), "flops": sum(f for _, f in each)}
    if kind == "bgemm":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": 8.0 * k * (m + n) + (8.0 if case["add"] else 4.0) * m * n, "flops": 2.0 * m * n * 64 * k}
    if kind == "pack":
        return {"bytes": case["n"] * case["h"] * case["w"] * case["c"] * 4.125, "flops": 0.0}
    out_bytes = 4.0
    if kind == "block":
        out_bytes += (4.0 if case["shortcut"] else 0.0) + (0.125 if case["sign"] else 0.0)
    b, f = _conv_work(case["n"], case["h"], case["w"], case["cin"], case["cout"], case.get("k", 3), case["stride"], case["pad"],
                      4 if kind == "layer" else 1 / 8, out_bytes)
    return {"bytes": b, "flops": f}


def tolerance(case):
    if case["kind"] not in ("net", "dense"):
        return "exact"  # counts are whole numbers, and each step behind them is rounded as the reference's layers round it
    # An fp32 sum of the float layers in another order changes its last bits, and where such a value lies at zero the
    # sign it passes on flips, which changes whole counts downstream.  Seen when the inputs' last bits move or the stem
    # sums in another order: per image nothing or 0.01 to 0.03, over 40 images and more 0.003 (three-convolution stem
    # 0.009), single logits by 0.11 of their root mean square; the dense net 0.005 on single images.
    if case["kind"] == "dense":
        return {"rel": 0.02, "max": 0.2}
    return {"rel": 0.03 if case["stem"] or case["batch"] < 32 else 0.01, "max": 0.4}
