/*
 * Probes of the MI355X (gfx950) backend: how large a problem is for the current device and which fused entry points of
 * dabnn_hip.h take it.  None of them has a counterpart in the reference and none computes anything: they exist so
 * that a caller that plans a layer sequence (Net::prepare) can link layers the way the kernels prefer, and so that a
 * parity test can name the build it means to cover.  The reference's surface, and the documented extensions of it,
 * are in dabnn_hip.h; a drop-in caller needs nothing from this file.
 */
#ifndef DABNN_HIP_TUNING_H
#define DABNN_HIP_TUNING_H

#include "dabnn_hip.h"

#ifdef __cplusplus
extern "C" {
#endif

/*
 * The kernel that dab_bconv3x3 (epilogue 0), dab_bconv3x3_affine_add (1) or dab_bconv3x3_affine_add_sign (2) runs for a
 * problem on the current device; -1 for one that the entry point refuses.
 */
enum {
    DAB_BCONV_SPLIT_16 = 0,     /* a block is one tile of 16 pixels, its three waves count a kernel row each */
    DAB_BCONV_SPLIT_32X32 = 1,  /* the same with tiles of 32 pixels x 32 channels */
    DAB_BCONV_SPLIT_32X64 = 2,  /* and 32 x 64 */
    DAB_BCONV_STREAM_32X32 = 3, /* 64 input channels: waves walk over tiles of 32 pixels x 32 channels */
    DAB_BCONV_STREAM_32X64 = 4, /* 32 x 64 */
    DAB_BCONV_STREAM_64X64 = 5, /* 64 x 64 */
    DAB_BCONV_WINDOW = 6        /* 128 to 512: the block's four waves share a tile's input window in LDS */
};
DAB_API int dab_bconv3x3_kernel(int n, int h, int w, int cin, int cout, int stride, int pad, int epilogue);

/*
 * Size classes of a direct convolution's problem (n_out_pixels = N*OH*OW; cin 64, 128, 256 or 512, cout a multiple of 8,
 * -1 otherwise), from the work a SIMD gets of it on the current device:
 *   0  few 64-pixel tiles (a SIMD gets less than one 64-pixel x 8-channel item, two with 512 input channels)
 *   1  mid-sized
 *   2  large: a SIMD gets many items
 *   3  256 and 512 input channels between the small and the mid-sized problems
 * A caller that plans a layer sequence goes by them: Net::prepare links a producer with 512 input channels to the
 * BinConv that reads its result (packed copy written by the producer) in the classes 0 and 3.  They are no answer to
 * which kernel runs: dab_bconv3x3_kernel is.
 */
/* of dab_bconv3x3_affine_add(_sign) at stride 1; never answers 3 */
DAB_API int dab_bconv3x3_build(int64_t n_out_pixels, int cin, int cout);
/* of dab_bconv3x3 */
DAB_API int dab_bconv3x3_counts_build(int64_t n_out_pixels, int cin, int cout, int stride);
/* of dab_bconv3x3_affine_add (with_sign = 0) and dab_bconv3x3_affine_add_sign (with_sign = 1) */
DAB_API int dab_bconv3x3_epilogue_build(int64_t n_out_pixels, int cin, int cout, int stride, int with_sign);
/* 1 for few tiles (class 0 before class 3 is asked), 0 otherwise and for other channel counts */
DAB_API int dab_bconv3x3_splits_depth(int64_t n_out_pixels, int cin, int cout);

/*
 * 1 for a first-stage block at a batch where the fp32 shortcut it reads and the result it writes are what bounds it (64
 * input channels, cout a multiple of 64, at least 32 tiles of 64 pixels per CU), 0 otherwise.
 */
DAB_API int dab_bconv3x3_fused_shares_tiles(int64_t n_out_pixels, int cin, int cout);

/*
 * 1 for the shapes dab_global_ave_pool_fconv1x1 covers (n <= 8, h * w <= 64, c a multiple of 4 up to 1024,
 * cout >= 64), 0 for those the two separate calls serve.
 */
DAB_API int dab_global_ave_pool_fconv1x1_takes(int n, int h, int w, int c, int cout);

/*
 * 1 when dab_fconv_maxpool takes the shape and the problem is large enough on the current device for the one pass to
 * beat dab_fconv_affine_relu + dab_max_pool_sign, 0 otherwise.
 */
DAB_API int dab_fconv_maxpool_pays(int n, int h, int w, int c, int kh, int kw, int pad_h, int pad_w, int stride_h,
                                   int stride_w, int dil_h, int dil_w, int cout);

#ifdef __cplusplus
}
#endif

#endif /* DABNN_HIP_TUNING_H */
