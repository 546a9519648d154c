"""Inputs from host memory and blobs back to it: small inputs through the layers' first kernel, large ones in blocks whose places are
used again, pinned callers, both kinds of input in turn, outputs that every run leaves in pinned memory."""
import threading

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def make(batch, hw, stem=False):
    from dabnn_amd import dab_format, models, net
    model = models.bireal18(7, stem=stem) if hw == 224 else models.dense_bnn(7, hw=hw)
    return net.Net(batch=batch).read_buf(dab_format.write_model(*model))


# input bytes: 12 KB, 1 044 480 and 1 056 768 (either side of a megabyte, where the layers' first kernel stops taking it), 8.4 MB (several
# transfers), 24 MB, 36 MB (more than the pinned memory: blocks that go round)
@pytest.mark.parametrize("batch,hw", [(1, 32), (85, 32), (86, 32), (14, 224), (40, 224), (60, 224)])
def test_host_and_device_inputs_give_the_same(batch, hw):
    n = make(batch, hw)
    r = np.random.default_rng(batch)
    held = torch.empty((batch, hw, hw, 3), device="cuda")
    for i in range(6):  # two eager runs, a capture, replays
        x = r.standard_normal((batch, hw, hw, 3)).astype(np.float32)
        n.run(x)
        from_host = n.get_blob("logits")
        if i % 2 == 0:
            assert np.array_equal(n.get_blob(n.input_name), x)
        assert np.array_equal(n.get_blob("logits"), from_host)
        held.copy_(torch.from_numpy(x))
        n.run(held)
        assert np.array_equal(n.get_blob("logits"), from_host)
    pinned = torch.from_numpy(x).pin_memory()
    n.run(pinned.numpy())
    assert np.array_equal(n.get_blob("logits"), from_host)
    n.close()


def test_blobs_of_every_size_come_back_whole():
    """Downloads in pieces of 512 KB, and what the library keeps of a wrong size."""
    n = make(3, 224)
    x = np.random.default_rng(0).standard_normal((3, 224, 224, 3)).astype(np.float32)
    n.run(x)
    assert np.array_equal(n.get_blob(n.input_name), x)
    assert np.array_equal(n.get_blob(n.input_name), x)
    with pytest.raises(ValueError):
        n.run(x[:2])


def test_several_nets_and_threads():
    nets = [make(12, 224) for _ in range(3)]
    r = np.random.default_rng(1)
    xs = [r.standard_normal((12, 224, 224, 3)).astype(np.float32) for _ in nets]
    want = []
    for n, x in zip(nets, xs):
        n.run(x)
        want.append(n.get_blob("logits"))
    got = [None] * len(nets)

    def work(i):
        for _ in range(6):
            nets[i].run(xs[i])
            got[i] = nets[i].get_blob("logits")

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(nets))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for a, b in zip(got, want):
        assert np.array_equal(a, b)


def copies_in_a_run(n, x):
    """Launches of the copy kernel in one run of a net without a graph."""
    from torch.profiler import ProfilerActivity, profile
    with profile(activities=[ProfilerActivity.CUDA]) as p:
        n.run(x)
        torch.cuda.synchronize()
    names = [e.name for e in p.events()]
    assert any("fconv" in s for s in names), names  # the trace shows the layers
    return sum("copy_f32" in s for s in names)


def test_outputs_are_copied_for_who_asks():
    n = make(2, 32)
    n.set_use_graph(False)
    x = torch.randn(2, 32, 32, 3, device="cuda")
    for _ in range(3):
        n.run(x)
    assert copies_in_a_run(n, x) == 0
    want = n.get_blob("logits")
    assert np.array_equal(n.get_blob("logits"), want)
    assert copies_in_a_run(n, x) == 1
    assert np.array_equal(n.get_blob("logits"), want)


# the copies begin before the graph is captured, in the graph's place, and behind either kind of input
@pytest.mark.parametrize("first_look", [1, 2, 3, 5])
def test_blobs_asked_for_late(first_look):
    n = make(2, 32)
    r = np.random.default_rng(first_look)
    for i in range(1, 12):
        x = r.standard_normal((2, 32, 32, 3)).astype(np.float32)
        n.run(x if i % 3 else torch.from_numpy(x).cuda())
        if i >= first_look:
            got = n.get_blob("logits")
            other = make(2, 32).run(x)
            assert np.array_equal(got, other.get_blob("logits")), i
            other.close()
