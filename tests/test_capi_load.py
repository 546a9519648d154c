"""Host-side checks of the C ABI that need no GPU: the library loads, exports
every symbol the header declares, and rejects bad arguments before touching
the device."""
import ctypes
import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def declared_symbols(headers=("dabnn_hip.h", "dabnn_hip_tuning.h")):
    text = "".join(open(os.path.join(ROOT, "include", h)).read() for h in headers)
    return sorted(set(re.findall(r"^DAB_API [^;(]*?\b(dab_\w+)\(", text, flags=re.M)))


def test_dispatch_probes_live_in_the_tuning_header():
    """dabnn_hip.h is the reference's surface plus the documented extensions; the probes that only say which kernel
    would run are declared in dabnn_hip_tuning.h."""
    probes = declared_symbols(("dabnn_hip_tuning.h",))
    assert probes == sorted(["dab_bconv3x3_build", "dab_bconv3x3_counts_build", "dab_bconv3x3_epilogue_build", "dab_bconv3x3_splits_depth", "dab_bconv3x3_fused_shares_tiles", "dab_bconv3x3_kernel",
                             "dab_global_ave_pool_fconv1x1_takes", "dab_fconv_maxpool_pays"])
    assert not set(probes) & set(declared_symbols(("dabnn_hip.h",)))


def test_which_kernel_a_direct_convolution_takes():
    """The rule the launches follow, at its edges; -1 for what the entry points refuse.  (No GPU is asked.)"""
    from dabnn_amd import capi
    split_16, split_32x32, split_32x64, stream_32x32, stream_32x64, stream_64x64, window = range(7)
    kernel = capi.lib.dab_bconv3x3_kernel
    # pixels in a row, so that pieces of 32 x 32 outputs are easy to count
    for cin, cout, mode, edges in [
            (64, 32, 0, [(224, split_16), (225, split_32x32), (767, split_32x32), (768, stream_32x32), (9000, stream_32x32)]),
            (64, 96, 0, [(74, split_16), (75, split_32x32), (255, split_32x32), (256, stream_32x64), (9000, stream_32x64)]),
            (64, 64, 1, [(112, split_16), (113, split_32x32), (384, stream_32x64), (2999, stream_32x64), (3000, stream_64x64)]),
            (128, 128, 2, [(40, split_16), (41, split_32x32), (319, split_32x32), (320, split_32x64), (511, split_32x64), (512, window)]),
            (256, 32, 1, [(160, split_16), (161, split_32x32), (1279, split_32x32), (1280, split_32x64), (2047, split_32x64), (2048, window)]),
            (512, 32, 0, [(160, split_16), (161, split_32x32), (1279, split_32x32), (1280, split_32x64), (2047, split_32x64), (2048, window)]),
            (1024, 32, 0, [(1, split_32x32), (5000, split_32x32)])]:
        for tiles, want in edges:
            assert kernel(tiles * 4, 2, 4, cin, cout, 1, 1, mode) == want, (cin, cout, mode, tiles)
    assert kernel(2, 70, 250, 512, 128, 1, 1, 0) == split_32x64  # the window of a tile does not fit LDS
    assert kernel(400, 4, 4, 128, 256, 1, 2, 0) == split_32x64  # the windows are no run of pixels
    assert kernel(1, 3, 3, 64, 2**22, 1, 1, 0) == split_32x64 and kernel(1, 3, 3, 1024, 2**22, 1, 1, 0) == split_32x32
    for bad in [(1, 4, 4, 192, 64, 1, 1, 0), (1, 4, 4, 64, 12, 1, 1, 0), (1, 4, 4, 1024, 64, 1, 1, 1), (1, 4, 4, 64, 72, 1, 1, 2), (1, 2, 2, 64, 8, 1, 0, 0),
                (0, 4, 4, 64, 8, 1, 1, 0), (1, 4, 4, 64, 8, 0, 1, 0), (1, 4, 4, 64, 8, 1, -1, 0), (1, 4, 4, 64, 8, 1, 1, 3), (2**20, 64, 64, 64, 8, 1, 1, 0)]:
        assert kernel(*bad) == -1, bad


def test_header_declares_the_expected_entry_points():
    names = declared_symbols()
    for must in ["dab_bitpack_nhwc", "dab_bitpack_nchw", "dab_fused_binarize_im2col", "dab_bgemm", "dab_bconv3x3",
                 "dab_binconv_forward", "dab_last_error", "dab_fconv", "dab_affine_inplace", "dab_add_inplace",
                 "dab_ave_pool", "dab_max_pool", "dab_pad_bit", "dab_weight_transpose"]:
        assert must in names


def test_library_exports_every_declared_symbol():
    from dabnn_amd import capi
    for name in declared_symbols():
        assert hasattr(capi.lib, name), name
        assert name in capi.SIGNATURES, "no ctypes signature for " + name
    assert capi.lib.dab_version() >= 1


def test_missing_library_fails_loudly(monkeypatch, tmp_path):
    import importlib
    from dabnn_amd import capi
    monkeypatch.setattr(capi, "LIB_PATH", str(tmp_path / "nope.so"))
    with pytest.raises(ImportError, match="no CPU fallback"):
        capi._load()
    importlib.reload(capi)


def test_argument_validation_without_device():
    from dabnn_amd import capi
    lib = capi.lib
    null = ctypes.c_void_p(None)
    one = ctypes.c_void_p(16)  # never dereferenced: validation fails first
    assert lib.dab_bitpack_nhwc(null, null, 1, 64, null) == capi.DAB_EINVAL
    assert "null pointer" in capi.last_error()
    assert lib.dab_bitpack_nhwc(one, one, 4, 100, null) == capi.DAB_EINVAL
    assert "multiple of 64" in capi.last_error()
    assert lib.dab_bgemm(4, 4, 4, one, 2, one, 4, one, 4, null) == capi.DAB_EINVAL
    assert "leading dimension" in capi.last_error()
    assert lib.dab_bconv3x3(one, 1, 8, 8, 192, one, 8, 1, 1, one, null) == capi.DAB_EUNSUPPORTED
    assert lib.dab_bconv3x3(one, 1, 8, 8, 64, one, 5, 1, 1, one, null) == capi.DAB_EUNSUPPORTED
    assert lib.dab_bconv3x3(one, 1, 2, 2, 64, one, 8, 1, 0, one, null) == capi.DAB_EINVAL
    assert lib.dab_fused_binarize_im2col(one, 1, 1, 1, 60000, 1, 1, 0, 0, 1, 1, 1, 1, one, null) == capi.DAB_EINVAL
    assert "smaller than 60000" in capi.last_error()
    with pytest.raises(capi.DabUnsupported):
        capi.check(capi.DAB_EUNSUPPORTED)
    with pytest.raises(RuntimeError):
        capi.check(capi.DAB_EINVAL)


def test_workspace_and_row_words():
    from dabnn_amd import capi
    lib = capi.lib
    assert lib.dab_col_row_words(3, 3, 64) == 10  # 9 words rounded up to 128 bits
    assert lib.dab_col_row_words(3, 3, 128) == 18
    assert lib.dab_col_row_words(3, 3, 512) == 72
    assert lib.dab_col_row_words(5, 5, 128) == 50
    assert lib.dab_col_row_words(3, 3, 3) == 2
    # direct method needs the packed input, bgemm method the column matrix
    assert lib.dab_binconv_workspace_bytes(1, 56, 56, 64, 3, 3, 1, 1, 1, 1) == 56 * 56 * 10 * 8
    assert lib.dab_binconv_workspace_bytes(2, 7, 7, 512, 3, 3, 1, 1, 1, 1) == 2 * 49 * 72 * 8


# the 3x3 route and the general one: sizes of which every call behind dab_binconv_forward refuses the arguments, however small the problem
@pytest.mark.parametrize("cout", [64, 60])
@pytest.mark.parametrize("change", [dict(pad_h=-1, pad_w=-1), dict(pad_w=-1), dict(stride_h=0), dict(stride_w=-1), dict(workspace=20), dict(out=18)])
def test_binconv_forward_refuses_what_its_parts_refuse(cout, change):
    from dabnn_amd import capi
    a = dict(pad_h=1, pad_w=1, stride_h=1, stride_w=1, workspace=32, out=32)
    a.update(change)
    vp = ctypes.c_void_p
    rc = capi.lib.dab_binconv_forward(vp(16), 2, 8, 9, 64, vp(16), vp(16), 9, 3, 3, a["pad_h"], a["pad_w"], a["stride_h"], a["stride_w"], cout, vp(a["out"]),
                                      vp(a["workspace"]), 1 << 30, None, vp(None))
    assert rc == capi.DAB_EINVAL, capi.last_error()


def test_binconv_forward_refuses_images_smaller_than_the_direct_kernel():
    """Stride 2 over two padded rows or columns: (2 - 3) / 2 + 1 is one output pixel in C, but no 3x3 window fits."""
    from dabnn_amd import capi
    vp = ctypes.c_void_p
    for h, w, pad in [(2, 9, 0), (9, 2, 0), (2, 2, 0)]:
        rc = capi.lib.dab_binconv_forward(vp(16), 2, h, w, 64, vp(16), vp(16), 9, 3, 3, pad, pad, 2, 2, 64, vp(32), vp(32), 1 << 30, None, vp(None))
        assert rc == capi.DAB_EINVAL and "smaller than the kernel" in capi.last_error(), capi.last_error()


def test_shapes_that_two_layers_take_in_one_pass():
    """dab_bconv3x3_pair_takes says what the call refuses, at the edges that the header states."""
    from dabnn_amd import capi
    vp = ctypes.c_void_p
    takes = capi.lib.dab_bconv3x3_pair_takes
    for h in (2, 7, 56, 300):
        assert [w for w in range(1, 600) if takes(4, h, w)] == list(range(16, 129)) + [160]
    assert [w for w in range(1, 600) if takes(4, 1, w)] == list(range(16, 161))
    assert takes(2**22, 1, 16) and not takes(2**23, 1, 16) and not takes(2**20, 300, 64) and not takes(1, 2**23, 16)
    assert not takes(0, 8, 16) and not takes(1, 0, 16) and not takes(1, 8, -1)
    for n, h, w in [(4, 7, 15), (4, 7, 129), (4, 7, 159), (4, 7, 161), (2**23, 1, 16), (2**20, 300, 64)]:
        rc = capi.lib.dab_bconv3x3_pair(vp(16), vp(16), n, h, w, vp(16), vp(16), vp(16), vp(16), vp(16), vp(16), vp(32), vp(64), vp(None))
        assert rc == capi.DAB_EUNSUPPORTED and not takes(n, h, w), (n, h, w)


def test_shapes_of_the_down_sampling_passes():
    """dab_bconv3x3_down_takes and dab_bconv3x3_pair_pool_takes say what the calls refuse, at the edges that the header states."""
    from dabnn_amd import capi
    vp = ctypes.c_void_p
    takes = capi.lib.dab_bconv3x3_down_takes
    assert [c for c in range(1, 1100) if takes(2, 8, 8, c, 64)] == [64, 128, 256] and [c for c in range(1, 300) if takes(2, 8, 8, 64, c)] == [64, 128, 192, 256]
    assert not takes(2, 7, 8, 64, 64) and not takes(2, 8, 7, 64, 64) and not takes(0, 8, 8, 64, 64) and not takes(2**20, 64, 64, 64, 64)
    for n, h, w, cin, cout in [(2, 7, 8, 64, 64), (2, 8, 8, 512, 64), (2, 8, 8, 64, 72), (2**20, 64, 64, 64, 64)]:
        rc = capi.lib.dab_bconv3x3_down(vp(16), vp(32), 0, n, h, w, cin, vp(16), vp(16), vp(16), cout, vp(16), None, None, None, None, vp(64), vp(128), vp(None))
        assert rc == capi.DAB_EUNSUPPORTED, (n, h, w, cin, cout)
    rc = capi.lib.dab_bconv3x3_down(vp(16), vp(32), 0, 2, 8, 8, 64, vp(16), vp(16), vp(16), 64, vp(16), None, vp(16), None, None, vp(64), vp(128), vp(None))
    assert rc == capi.DAB_EINVAL and "both coefficient vectors" in capi.last_error()
    pool = capi.lib.dab_bconv3x3_pair_pool_takes
    assert [w for w in range(1, 200) if pool(4, 8, w)] == list(range(2, 65, 2)) and not pool(4, 7, 16) and not pool(0, 8, 16) and not pool(2**23, 2, 2)
    for n, h, w in [(4, 7, 16), (4, 8, 15), (4, 8, 66), (2**23, 2, 2)]:
        rc = capi.lib.dab_bconv3x3_pair_pool(vp(16), vp(16), n, h, w, vp(16), vp(16), vp(16), vp(16), vp(16), vp(16), vp(32), vp(64), vp(None))
        assert rc == capi.DAB_EUNSUPPORTED, (n, h, w)
