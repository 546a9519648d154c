"""Nets whose residual layers over 64 channels run two in a pass: every blob a user can ask for, the ones inside the passes included, on
several runs (eager, captured, replayed), first asked for at different times; which layers run that way."""
import numpy as np
import pytest

from oracle import net as orc_net
import oracle as orc

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def mods():
    from dabnn_amd import dab_format, models, net
    return dab_format, models, net


def residual_net(models, blocks, hw, seed=0, extra_reader=False):
    """stem 3x3 -> `blocks` residual layers over 64 channels -> 1x1 classifier over the whole image."""
    r = np.random.default_rng(seed)
    layers, inits = [], []

    def tensor(name, data, shape=None, align=False):
        inits.append({"name": name, "shape": list(data.shape if shape is None else shape), "data": data, "align_hwc_to_128": align})
        return name

    layers.append({"type": "FpConv2D", "name": "stem", "input": "data", "weight": tensor("stem_w", (r.standard_normal((64, 3, 3, 3)) / 5).astype(np.float32)),
                   "output": "s", "pads": [1] * 4, "strides": [1, 1], "dilations": [1, 1]})
    cur = "s"
    for i in range(blocks):
        p = "b%d" % i
        wf = r.standard_normal((64, 3, 3, 64)).astype(np.float32)
        layers.append({"type": "BinConv2D", "name": p, "input": cur, "weight": tensor(p + "_w", models.pack_weight(wf).ravel(), shape=[64, 3, 3, 64]),
                       "output": p + "_cnt", "pads": [1] * 4, "strides": [1, 1], "dilations": [1, 1]})
        a, b = models.fold_bn(np.full(64, 0.5, np.float32), (0.1 * r.standard_normal(64)).astype(np.float32), np.zeros(64, np.float32),
                              np.full(64, 9.0 * 64, np.float32), 1e-5, 9 * 64)
        layers.append({"type": "Affine", "name": p + "_affine", "input": p + "_cnt", "a": tensor(p + "_a", a), "b": tensor(p + "_b", b), "output": p + "_bn"})
        layers.append({"type": "Add", "name": p + "_add", "input1": p + "_bn", "input2": cur, "output": p + "_out"})
        cur = p + "_out"
    if extra_reader:  # of the first pass's inner blob
        layers.append({"type": "MaxPool", "name": "peek", "input": "b0_out", "output": "peek_out", "kernel_shape": [2, 2], "pads": [0] * 4, "strides": [2, 2]})
    layers.append({"type": "AvePool", "name": "gap", "input": cur, "output": "gap_out", "kernel_shape": [hw, hw], "pads": [0] * 4, "strides": [1, 1]})
    layers.append({"type": "FpConv2D", "name": "fc", "input": "gap_out", "weight": tensor("fc_w", (r.standard_normal((10, 1, 1, 64)) / 8).astype(np.float32)),
                   "output": "logits", "pads": [0] * 4, "strides": [1, 1], "dilations": [1, 1]})
    return layers, inits, [("data", [1, hw, hw, 3])]


def passes(n):
    return sum("in one pass with the next layer" in d for d in n.layers())


def check_image(n, layers, inits, i):
    checked = 0
    for name, first_type, want in orc_net.run_segments(layers, inits, lambda b: n.get_blob(b)[i]):
        got = n.get_blob(name)[i]
        if first_type == "BinConv2D":
            np.testing.assert_array_equal(got, want, err_msg=name)
        else:
            np.testing.assert_allclose(got, want, rtol=1e-4, atol=1e-4 * np.abs(want).max(), err_msg=name)
        checked += 1
    return checked


@pytest.mark.parametrize("blocks,hw,batch,pairs", [(2, 28, 62, 1), (3, 32, 47, 1), (5, 56, 16, 2), (4, 64, 12, 2), (4, 28, 61, 0), (4, 65, 12, 0), (2, 16, 188, 1)])
def test_every_blob_on_every_run(mods, blocks, hw, batch, pairs):
    df, models, net = mods
    layers, inits, inputs = residual_net(models, blocks, hw)
    n = net.Net(batch=batch).read_buf(df.write_model(layers, inits, inputs))
    assert passes(n) == pairs
    r = np.random.default_rng(batch)
    for run in range(6):
        n.run(r.standard_normal((batch, hw, hw, 3)).astype(np.float32))
        if run == 1:  # a packed copy from inside a pass, before the blob it is the copy of
            np.testing.assert_array_equal(n.get_blob("binaized_for_b1_cnt_cal")[3], orc.pack_mat(n.get_blob("b0_out")[3]))
        if run >= 2:
            assert check_image(n, layers, inits, (run * 7) % batch) == blocks + 3
    i = batch - 1
    packed, col = n.get_blob("binaized_for_b1_cnt_cal"), n.get_blob("col_for_b1_cnt_cal")
    np.testing.assert_array_equal(packed[i], orc.pack_mat(n.get_blob("b0_out")[i]))
    bits = np.unpackbits(np.ascontiguousarray(packed[i]).view(np.uint8), axis=-1, bitorder="little").reshape(hw, hw, 64)
    want = orc.fused_binarize_im2col(np.where(bits, 1, -1).astype(np.float32), 3, 3, 1, 1, 1, 1)
    np.testing.assert_array_equal(col.reshape(batch, -1)[i], want.ravel())
    n.close()


def test_first_asked_for_from_a_replay_and_column_matrix_first(mods):
    df, models, net = mods
    layers, inits, inputs = residual_net(models, 4, 28, seed=3)
    n = net.Net(batch=64).read_buf(df.write_model(layers, inits, inputs))
    r = np.random.default_rng(5)
    for run in range(5):
        n.run(r.standard_normal((64, 28, 28, 3)).astype(np.float32))
    col = n.get_blob("col_for_b3_cnt_cal").copy()
    packed = n.get_blob("binaized_for_b3_cnt_cal")
    np.testing.assert_array_equal(packed[9], orc.pack_mat(n.get_blob("b2_out")[9]))
    assert check_image(n, layers, inits, 9) == 7
    n.run(r.standard_normal((64, 28, 28, 3)).astype(np.float32))
    assert not np.array_equal(n.get_blob("col_for_b3_cnt_cal"), col)
    assert check_image(n, layers, inits, 63) == 7
    n.close()


def test_a_blob_with_another_reader_is_kept(mods):
    df, models, net = mods
    layers, inits, inputs = residual_net(models, 4, 28, extra_reader=True)
    n = net.Net(batch=64).read_buf(df.write_model(layers, inits, inputs))
    assert passes(n) == 1  # b0 and b1 stay apart, b1 and b2 go together
    n.run(np.random.default_rng(1).standard_normal((64, 28, 28, 3)).astype(np.float32))
    assert check_image(n, layers, inits, 5) == 8
    n.close()


def test_bireal18_stage_one(mods):
    df, models, net = mods
    layers, inits, inputs = models.bireal18(4)
    n = net.Net(batch=24).read_buf(df.write_model(layers, inits, inputs))
    assert passes(n) == 2 and sum("+ Affine + Add" in d for d in n.layers()) == 16
    r = np.random.default_rng(6)
    x = r.standard_normal((24, 224, 224, 3)).astype(np.float32)
    for _ in range(4):
        n.run(x)
    first = n.get_blob("logits")
    pool = n.get_blob("s1b0_out")  # inside the first pass
    n.run(x)
    assert np.array_equal(n.get_blob("logits"), first) and np.array_equal(n.get_blob("s1b0_out"), pool)
    n.close()
