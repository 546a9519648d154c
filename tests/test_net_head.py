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
