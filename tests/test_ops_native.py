"""The native module behind the operators: it leaves every call that is not the plain case to the Python function (whose
checks and errors are the documented ones), and the plain case gives what the C ABI gives."""
import pytest
import torch


def test_host_tensors_and_wrong_arguments_are_left_to_python():
    from dabnn_amd.ops import _native
    x, w = torch.zeros((1, 4, 4, 1), dtype=torch.int64), torch.zeros((8, 9), dtype=torch.int64)
    assert _native.pack_mat(torch.zeros((1, 2, 2, 64))) is None
    assert _native.pack_mat("no tensor") is None and _native.pack_mat() is None
    assert _native.bconv_3x3(x, w, 1, 1) is None and _native.bconv_3x3(x, w, "1", 1) is None
    assert _native.bconv_3x3_affine_add(x, w, x, x, None, 1, 1) is None
    assert _native.bgemm(1, 1, 1, x, 1, x, 1, x, 1) is None and _native.bgemm(1, 2**40, 1, x, 1, x, 1, x, 1) is None
    assert _native.binconv(torch.zeros((1, 4, 4, 64)), w, w, None, 3, 3, 1, 1, 1, 1) is None


@pytest.mark.gpu
def test_plain_calls_and_their_errors():
    import dabnn_amd as dab
    from dabnn_amd import capi
    from dabnn_amd.ops import _native
    g = torch.Generator(device="cuda").manual_seed(1)
    x = torch.randn((3, 7, 5, 128), device="cuda", generator=g)
    packed = _native.pack_mat(x)
    assert torch.equal(packed, dab.pack_mat(x)) and tuple(packed.shape) == (3, 7, 5, 2)
    w = torch.randint(-2**63, 2**63 - 1, (64, 18), dtype=torch.int64, device="cuda", generator=g)
    counts = dab.bconv_3x3(packed, w, stride=2)
    layer = dab.BinConv(w, 3, 3, 1, 1, 2, 2)
    assert torch.equal(layer(x), counts) and layer.method == layer.DIRECT_CONV
    first = layer._ws
    assert torch.equal(layer(x[:2].contiguous()), counts[:2]) and layer._ws.data_ptr() == first.data_ptr()  # kept while it fits
    # on a stream of its own, the result is ready there
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        there = dab.bconv_3x3(packed, w, 2, 1)
    side.synchronize()
    assert torch.equal(there, counts)
    # not the plain case: Python's checks answer
    with pytest.raises(capi.DabError, match="contiguous"):
        dab.bconv_3x3(packed.transpose(1, 2), w)
    with pytest.raises(capi.DabError, match="expected 1152"):
        dab.bconv_3x3(packed, w[:, :17].contiguous())
    with pytest.raises(capi.DabError, match="multiple of 64"):
        dab.pack_mat(torch.zeros((2, 3), device="cuda"))
    # refused by the C ABI: its code and message
    with pytest.raises(capi.DabUnsupported, match="not covered by the direct kernel"):
        dab.bconv_3x3(packed, w[:63].contiguous())
