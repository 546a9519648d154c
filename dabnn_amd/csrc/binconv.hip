// BinConv::forward_impl (dabnn/layers/BinConv.cpp:144-191) as one call:
// binarise the fp32 input and run the binary convolution, choosing between
// the direct 3x3 kernel and im2col + bgemm the way BinConv::method() (:80-98)
// does on the reference's optimised targets.
#include <mutex>

#include "bgemm_core.h"

namespace dab {

// Scratch of dab_binconv_forward_static: the packed activations (direct arm) or the column matrix (bgemm arm) of one
// call.  One copy per GPU, held until the process ends; the array's name is only a handle for hipGetSymbolAddress in
// host code, the kernels get the device address that call returns.
static __device__ __align__(256) unsigned char scratch[DAB_BINCONV_STATIC_SCRATCH_BYTES];

constexpr int kMaxDevices = 64;
static void *scratch_ptr[kMaxDevices];  // device address of `scratch` on each GPU, resolved on the first call there
static std::mutex scratch_mutex;

// Device address of this GPU's copy of `scratch` (the current device's).
static int static_scratch(void **out) {
    int dev = 0;
    DAB_HIP(hipGetDevice(&dev));
    if (dev < 0 || dev >= kMaxDevices) return fail(DAB_EUNSUPPORTED, "dab_binconv_forward_static: device index %d", dev);
    std::lock_guard<std::mutex> lock(scratch_mutex);
    if (scratch_ptr[dev] == nullptr) {
        void *p = nullptr;
        DAB_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        if (p == nullptr) return fail(DAB_EHIP, "dab_binconv_forward_static: no device address for the scratch array");
        scratch_ptr[dev] = p;
    }
    *out = scratch_ptr[dev];
    return DAB_OK;
}


static bool direct_ok(int c, int kh, int kw, int pad_h, int pad_w, int stride_h, int stride_w, int cout) {
    // dabnn/layers/BinConv.cpp:100-126: 3x3, equal strides, 64/128/256/512/1024 input channels
    return kh == 3 && kw == 3 && stride_h == stride_w && pad_h == pad_w &&
           (c == 64 || c == 128 || c == 256 || c == 512 || c == 1024) && cout % 8 == 0;
}
// fused_binarize_im2col's own limit on a column (dabnn/fused_binarize_im2col.h:23)
static bool im2col_row_fits(int kh, int kw, int c) { return (long long)kh * kw * c < 60000; }
}  // namespace dab

extern "C" size_t dab_binconv_workspace_bytes(int n, int h, int w, int c, int kh, int kw, int pad_h, int pad_w,
                                              int stride_h, int stride_w) {
    using namespace dab;
    if (n <= 0 || h <= 0 || w <= 0 || c <= 0 || kh <= 0 || kw <= 0 || stride_h <= 0 || stride_w <= 0) return 0;
    const size_t packed = (size_t)n * h * w * ((c + 63) / 64) * 8;
    const int oh = out_dim(h, pad_h, kh, 1, stride_h), ow = out_dim(w, pad_w, kw, 1, stride_w);
    const size_t col = (size_t)n * (oh > 0 ? oh : 0) * (ow > 0 ? ow : 0) * dab_col_row_words(kh, kw, c) * 8;
    return packed > col ? packed : col;
}

extern "C" int dab_binconv_forward(const float *x, int n, int h, int w, int c, const uint64_t *wgt, const uint64_t *wgt_t,
                                   int hwc_words, int kh, int kw, int pad_h, int pad_w, int stride_h, int stride_w,
                                   int cout, float *out, void *workspace, size_t workspace_bytes, int *method_out,
                                   dab_stream_t stream) {
    using namespace dab;
    DAB_REQUIRE(x && out && workspace, "dab_binconv_forward: null pointer");
    DAB_REQUIRE(n > 0 && h > 0 && w > 0 && c > 0 && cout > 0 && kh > 0 && kw > 0, "dab_binconv_forward: non-positive dimension");
    DAB_REQUIRE(pad_h >= 0 && pad_w >= 0 && stride_h > 0 && stride_w > 0, "dab_binconv_forward: bad pad/stride");
    DAB_REQUIRE(c % 64 == 0, "dab_binconv_forward: c %d is not a multiple of 64", c);
    DAB_REQUIRE(workspace_bytes >= dab_binconv_workspace_bytes(n, h, w, c, kh, kw, pad_h, pad_w, stride_h, stride_w),
                "dab_binconv_forward: workspace too small");
    const int oh = out_dim(h, pad_h, kh, 1, stride_h), ow = out_dim(w, pad_w, kw, 1, stride_w);
    DAB_REQUIRE(oh > 0 && ow > 0, "dab_binconv_forward: empty output");

    if (direct_ok(c, kh, kw, pad_h, pad_w, stride_h, stride_w, cout)) {
        DAB_REQUIRE(wgt, "dab_binconv_forward: direct method needs wgt");
        DAB_REQUIRE(hwc_words == 9 * (c / 64), "dab_binconv_forward: %d words per filter, expected %d", hwc_words,
                    9 * (c / 64));
        DAB_REQUIRE(h + 2 * pad_h >= 3 && w + 2 * pad_w >= 3, "dab_binconv_forward: input smaller than the kernel");
        DAB_REQUIRE((reinterpret_cast<uintptr_t>(workspace) & 15) == 0 && (reinterpret_cast<uintptr_t>(wgt) & 7) == 0 && (reinterpret_cast<uintptr_t>(out) & 15) == 0,
                    "dab_binconv_forward: buffers must be 16-byte aligned");
        int rc = c <= 512 ? bconv_float_try(x, n, h, w, c, wgt, hwc_words, kh, kw, pad_h, pad_w, stride_h, stride_w, cout, out, oh, ow, as_stream(stream)) : 0;
        if (rc != 0) {
            if (rc > 0 && method_out) *method_out = 0;
            return rc > 0 ? DAB_OK : rc;
        }
        uint64_t *packed = static_cast<uint64_t *>(workspace);
        rc = dab_bitpack_nhwc(x, packed, (int64_t)n * h * w, c, stream);
        if (rc != DAB_OK) return rc;
        rc = dab_bconv3x3(packed, n, h, w, c, wgt, cout, stride_h, pad_h, out, stream);
        if (rc == DAB_OK && method_out) *method_out = 0;
        return rc;
    }

    DAB_REQUIRE(wgt_t, "dab_binconv_forward: bgemm method needs the transposed weights");
    const int row_words = dab_col_row_words(kh, kw, c);
    DAB_REQUIRE(hwc_words <= row_words && hwc_words * 64 >= kh * kw * c,
                "dab_binconv_forward: %d words per filter does not match a %dx%dx%d filter", hwc_words, kh, kw, c);
    const long long npix = (long long)n * oh * ow;
    if (npix >= (1ll << 31)) return fail(DAB_EUNSUPPORTED, "dab_binconv_forward: too many output pixels");
    if (wgt != nullptr && (reinterpret_cast<uintptr_t>(wgt) & 7) == 0 && im2col_row_fits(kh, kw, c) && bit_gemm_takes_images((long long)n * h * w * (c / 64), (long long)cout * hwc_words, npix, cout)) {
        // The column matrix is fused_binarize_im2col of the input, kh * kw times its packed copy: the convolution reads
        // the packed pixels of a window where they are instead (8 x 14 x 14 x 256, 5 x 5: 11 us against 26 with the
        // column matrix and its GEMM).
        DAB_REQUIRE((reinterpret_cast<uintptr_t>(workspace) & 7) == 0 && (reinterpret_cast<uintptr_t>(out) & 3) == 0, "dab_binconv_forward: misaligned pointer");
        int rc = bconv_float_try(x, n, h, w, c, wgt, hwc_words, kh, kw, pad_h, pad_w, stride_h, stride_w, cout, out, oh, ow, as_stream(stream));
        if (rc != 0) {
            if (rc > 0 && method_out) *method_out = 1;
            return rc > 0 ? DAB_OK : rc;
        }
        uint64_t *packed = static_cast<uint64_t *>(workspace);
        rc = dab_bitpack_nhwc(x, packed, (int64_t)n * h * w, c, stream);
        if (rc != DAB_OK) return rc;
        rc = dab_bconv(packed, c / 64, n, h, w, c, wgt, hwc_words, kh, kw, pad_h, pad_w, stride_h, stride_w, cout, nullptr, nullptr,
                       nullptr, out, cout, nullptr, 0, stream);
        if (rc == DAB_OK && method_out) *method_out = 1;
        return rc;
    }
    // output_mat->fill<float>(0.f) and the accumulation into it (BinConv.cpp:153-165) are one store: 0.f + count == count
    uint64_t *col = static_cast<uint64_t *>(workspace);
    int rc = dab_fused_binarize_im2col(x, n, h, w, c, kh, kw, pad_h, pad_w, stride_h, stride_w, 1, 1, col, stream);
    if (rc != DAB_OK) return rc;
    rc = dab_bgemm_overwrite(cout, (int)npix, hwc_words, wgt_t, cout, col, row_words, out, cout, stream);
    if (rc == DAB_OK && method_out) *method_out = 1;
    return rc;
}

extern "C" int dab_bconv(const uint64_t *x, int64_t x_ld, int n, int h, int w, int c, const uint64_t *wgt, int hwc_words, int kh,
                         int kw, int pad_h, int pad_w, int stride_h, int stride_w, int cout, const float *a, const float *b,
                         const float *shortcut, float *out, int64_t out_ld, uint64_t *out_packed, int64_t packed_ld,
                         dab_stream_t stream) {
    using namespace dab;
    const char *fn = "dab_bconv";
    DAB_REQUIRE(x && wgt && out, "%s: null pointer", fn);
    DAB_REQUIRE(n > 0 && h > 0 && w > 0 && c > 0 && cout > 0 && kh > 0 && kw > 0, "%s: non-positive dimension", fn);
    DAB_REQUIRE(pad_h >= 0 && pad_w >= 0 && stride_h > 0 && stride_w > 0, "%s: bad pad/stride", fn);
    DAB_REQUIRE(c % 64 == 0, "%s: c %d is not a multiple of 64", fn, c);
    const int cw = c / 64;
    DAB_REQUIRE(hwc_words >= kh * kw * cw && hwc_words <= dab_col_row_words(kh, kw, c), "%s: %d words per filter does not match a %dx%dx%d filter",
                fn, hwc_words, kh, kw, c);
    DAB_REQUIRE(x_ld >= cw && out_ld >= cout && (!out_packed || packed_ld * 64 >= cout), "%s: leading dimension smaller than the row", fn);
    DAB_REQUIRE((a == nullptr) == (b == nullptr) && (a || (!shortcut && !out_packed)), "%s: an epilogue needs both affine vectors", fn);
    DAB_REQUIRE((reinterpret_cast<uintptr_t>(x) & 7) == 0 && (reinterpret_cast<uintptr_t>(wgt) & 7) == 0 && (reinterpret_cast<uintptr_t>(out) & 3) == 0 &&
                    (reinterpret_cast<uintptr_t>(out_packed) & 7) == 0,
                "%s: misaligned pointer", fn);
    if (out_packed && cout % 64 != 0) return fail(DAB_EUNSUPPORTED, "%s: cout %d is not a multiple of 64", fn, cout);
    const int oh = out_dim(h, pad_h, kh, 1, stride_h), ow = out_dim(w, pad_w, kw, 1, stride_w);
    DAB_REQUIRE(oh > 0 && ow > 0, "%s: empty output", fn);
    const long long npix = (long long)n * oh * ow;
    if (!im2col_row_fits(kh, kw, c) || !bit_gemm_takes_images((long long)n * h * w * x_ld, (long long)cout * hwc_words, npix, cout))
        return fail(DAB_EUNSUPPORTED, "%s: tensor too large for 32-bit indexing", fn);
    BitGemm g = {};
    g.x = x, g.w = wgt, g.out = out;
    g.rows = npix, g.cols = cout;
    g.x_ld = x_ld, g.w_ld = hwc_words, g.out_ld = out_ld;
    g.words = kh * kw * cw, g.extra_word = hwc_words > kh * kw * cw;
    g.H = h, g.W = w, g.OH = oh, g.OW = ow, g.kw = kw;
    g.stride_h = stride_h, g.stride_w = stride_w, g.pad_h = pad_h, g.pad_w = pad_w;
    g.tap_words = cw;
    g.a = a, g.b = b, g.shortcut = shortcut;
    g.bits = reinterpret_cast<uint32_t *>(out_packed), g.bits_ld = (int)(2 * packed_ld);
    return bit_gemm(fn, g, kFilterRows, as_stream(stream));
}

extern "C" int dab_binconv_forward_static(const float *x, int n, int h, int w, int c, const uint64_t *wgt,
                                          const uint64_t *wgt_t, int hwc_words, int kh, int kw, int pad_h, int pad_w,
                                          int stride_h, int stride_w, int cout, float *out, int *method_out,
                                          dab_stream_t stream) {
    using namespace dab;
    DAB_REQUIRE(n > 0 && h > 0 && w > 0 && c > 0 && kh > 0 && kw > 0 && stride_h > 0 && stride_w > 0,
                "dab_binconv_forward_static: non-positive dimension");
    const size_t need = dab_binconv_workspace_bytes(n, h, w, c, kh, kw, pad_h, pad_w, stride_h, stride_w);
    if (need > (size_t)DAB_BINCONV_STATIC_SCRATCH_BYTES)
        return fail(DAB_EUNSUPPORTED,
                    "dab_binconv_forward_static: this problem needs %zu bytes of scratch, the static buffer holds %zu; "
                    "use dab_binconv_forward with a workspace of your own",
                    need, (size_t)DAB_BINCONV_STATIC_SCRATCH_BYTES);
    void *ws = nullptr;
    const int rc = static_scratch(&ws);
    if (rc != DAB_OK) return rc;
    // both arms overwrite every word of the scratch they read, so nothing of the previous call has to be cleared
    return dab_binconv_forward(x, n, h, w, c, wgt, wgt_t, hwc_words, kh, kw, pad_h, pad_w, stride_h, stride_w, cout, out,
                               ws, (size_t)DAB_BINCONV_STATIC_SCRATCH_BYTES, method_out, stream);
}
