"""Large host inputs: the first layers run on the images that have arrived.  Logits and blobs are bit for bit those of a run from device memory,
from pageable and pinned memory, on every run, below and above the two shares (of 8 MB; an image is 0.6) where that begins, at batches that
end inside a share, and for who looks at blobs in between."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def model():
    from dabnn_amd import dab_format, models
    return dab_format.write_model(*models.bireal18(21))


def open_net(model, batch):
    from dabnn_amd import net
    return net.Net(batch=batch).read_buf(model)


@pytest.mark.parametrize("batch", [27, 28, 29, 40, 57, 100])
def test_same_bits_as_from_the_device(model, batch):
    r = np.random.default_rng(batch)
    a, b = open_net(model, batch), open_net(model, batch)
    for run in range(5):
        x = r.standard_normal((batch, 224, 224, 3)).astype(np.float32)
        host = torch.from_numpy(x).pin_memory().numpy() if run % 3 == 2 else x
        a.run(host)
        b.run(torch.from_numpy(x).cuda())
        assert np.array_equal(a.get_blob("logits"), b.get_blob("logits")), run
        for name in ("pool1_out", "s1b1_out", "s1b3_out", "s2b0_out", "s2b0_sc_conv_out") if run in (1, 4) else ():
            assert np.array_equal(a.get_blob(name), b.get_blob(name)), (run, name)
    # a device input in between, and back
    x = r.standard_normal((batch, 224, 224, 3)).astype(np.float32)
    a.run(torch.from_numpy(x).cuda())
    first = a.get_blob("logits")
    a.run(x)
    assert np.array_equal(a.get_blob("logits"), first)
    a.set_use_graph(False)
    a.run(x)
    assert np.array_equal(a.get_blob("logits"), first)
    a.set_profile(True)
    a.run(x)
    assert np.array_equal(a.get_blob("logits"), first) and "Float Conv" in a.time_report()
    a.close()
    b.close()


def test_two_nets_on_threads(model):
    import threading
    r = np.random.default_rng(3)
    xs = [r.standard_normal((32, 224, 224, 3)).astype(np.float32) for _ in range(2)]
    nets = [open_net(model, 32) for _ in xs]
    want = [open_net(model, 32).run(torch.from_numpy(x).cuda()).get_blob("logits") for x in xs]
    got = [[] for _ in xs]

    def work(i):
        for _ in range(8):
            nets[i].run(xs[i])
            got[i].append(nets[i].get_blob("logits"))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for g, w in zip(got, want):
        assert len(g) == 8 and all(np.array_equal(v, w) for v in g)


def headed_net(blocks, hw, seed=0, width=64, classifier=True):
    """7x7 stem and MaxPool -> binary layers, each (output channels, stride, residual, Affine) -> classifier; and the names of all blobs."""
    from dabnn_amd import models
    r = np.random.default_rng(seed)
    layers, inits, names = [], [], []

    def tensor(name, data, shape=None, align=False):
        inits.append({"name": name, "shape": list(data.shape if shape is None else shape), "data": data, "align_hwc_to_128": align})
        return name

    def add(kind, name, out, **fields):
        layers.append({"type": kind, "name": name, "output": out, **fields})
        names.append(out)
        return out

    cur, cin = add("FpConv2D", "stem", "stem_out", input="data", weight=tensor("stem_w", (r.standard_normal((width, 7, 7, 3)) / 12).astype(np.float32)), pads=[3] * 4, strides=[2, 2],
                   dilations=[1, 1]), width
    a, b = (1 + 0.1 * r.standard_normal(width)).astype(np.float32), (0.1 * r.standard_normal(width)).astype(np.float32)
    cur = add("Affine", "stem_affine", "stem_bn", input=cur, a=tensor("stem_a", a), b=tensor("stem_b", b))
    cur = add("MaxPool", "pool", "pool_out", input=cur, kernel_shape=[3, 3], pads=[1] * 4, strides=[2, 2])
    size = (hw + 1) // 2
    size = (size + 1) // 2
    for i, (cout, stride, residual, affine) in enumerate(blocks):
        p = "b%d" % i
        wf = r.standard_normal((cout, 3, 3, cin)).astype(np.float32)
        out = add("BinConv2D", p, p + "_cnt", input=cur, weight=tensor(p + "_w", models.pack_weight(wf).ravel(), shape=[cout, 3, 3, cin], align=cin != 64), pads=[1] * 4,
                  strides=[stride, stride], dilations=[1, 1])
        if affine:
            a, b = models.fold_bn(np.full(cout, 0.5, np.float32), (0.1 * r.standard_normal(cout)).astype(np.float32), np.zeros(cout, np.float32),
                                  np.full(cout, 9.0 * cin, np.float32), 1e-5, 9 * cin)
            out = add("Affine", p + "_affine", p + "_bn", input=out, a=tensor(p + "_a", a), b=tensor(p + "_b", b))
        if residual:
            out = add("Add", p + "_add", p + "_out", input1=out, input2=cur)
        cur, cin, size = out, cout, (size - 1) // stride + 1
    if not classifier:
        return (layers, inits, [("data", [1, hw, hw, 3])]), names
    cur = add("AvePool", "gap", "gap_out", input=cur, kernel_shape=[size, size], pads=[0] * 4, strides=[1, 1])
    add("FpConv2D", "fc", "logits", input=cur, weight=tensor("fc_w", (r.standard_normal((10, 1, 1, cin)) / 8).astype(np.float32)), pads=[0] * 4, strides=[1, 1], dilations=[1, 1])
    return (layers, inits, [("data", [1, hw, hw, 3])]), names


# An odd number of residual layers over 64 channels, and layers over 128 without and with a shortcut; layers without Affine and without sign
# bits for a next one; a stride without a branch; images of the packed blobs that are no multiple of 16 bytes, behind which the head ends; a
# wider stem.
HEADS = {
    "odd": ([(64, 1, True, True)] * 3 + [(128, 1, False, True), (128, 1, True, True), (64, 1, False, True)], 224, 37, 64),
    "single": ([(64, 1, True, True)], 224, 30, 64),
    "no shortcut": ([(64, 1, False, True), (64, 1, True, True), (256, 1, False, True), (256, 1, True, True)], 224, 29, 64),
    "no affine": ([(64, 1, False, True), (64, 1, False, False), (64, 1, True, True)], 224, 33, 64),
    "strided": ([(64, 1, True, True), (128, 2, False, True), (128, 1, True, True), (256, 2, False, True)], 224, 41, 64),
    "unaligned": ([(64, 2, False, True)] * 3 + [(128, 1, False, True), (64, 1, False, True)], 224, 35, 64),
    "wide stem": ([(128, 1, True, True), (128, 1, True, True)], 224, 31, 128),
}


@pytest.mark.parametrize("kind", sorted(HEADS))
def test_heads_of_other_nets(kind):
    """Every blob that can be asked for, from pageable and pinned memory, against a run from the device."""
    from dabnn_amd import dab_format, net
    blocks, hw, batch, width = HEADS[kind]
    model, names = headed_net(blocks, hw, width=width)
    data = dab_format.write_model(*model)
    a, b = (net.Net(batch=batch).read_buf(data) for _ in range(2))
    assert batch * hw * hw * 12 >= 16 << 20
    r = np.random.default_rng(7)

    def blobs(n):
        out = {}
        for name in names:
            try:
                out[name] = n.get_blob(name)
            except Exception as e:
                assert "is not produced" in str(e), e
        return out

    for run in range(6):
        x = r.standard_normal((batch, hw, hw, 3)).astype(np.float32)
        a.run(torch.from_numpy(x).pin_memory().numpy() if run % 2 else x)
        b.run(torch.from_numpy(x).cuda())
        assert np.array_equal(a.get_blob("logits"), b.get_blob("logits")), run
        if run < 3:
            continue  # the blobs inside passes are asked for behind captured runs, and kept up to date by those after
        got, want = blobs(a), blobs(b)
        assert got.keys() == want.keys() and len(got) > len(blocks)
        for name in got:
            assert np.array_equal(got[name], want[name]), (run, name)
    a.close()
    b.close()


@pytest.mark.parametrize("blocks", [[(64, 1, True, True)], [(64, 1, True, True)] * 2, [(64, 1, False, True), (64, 1, True, True), (128, 2, False, True)]])
def test_nets_that_end_with_their_head(blocks):
    """No layer is left behind it; results too large to be copied for who asks, and (64 x 7 x 7) small enough."""
    from dabnn_amd import dab_format, net
    for blocks in (blocks, blocks + [(64, 2, False, True)] * 2):
        model, names = headed_net(blocks, 224, classifier=False)
        data = dab_format.write_model(*model)
        a, b = (net.Net(batch=30).read_buf(data) for _ in range(2))
        r = np.random.default_rng(len(blocks))
        for run in range(6):
            x = r.standard_normal((30, 224, 224, 3)).astype(np.float32)
            a.run(torch.from_numpy(x).pin_memory().numpy() if run % 2 else x)
            b.run(torch.from_numpy(x).cuda())
            assert np.array_equal(a.get_blob(names[-1]), b.get_blob(names[-1])), run
        a.close()
        b.close()
