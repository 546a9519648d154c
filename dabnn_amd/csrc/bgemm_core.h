// The general binary GEMM of this library: out[row][col] = number of places where two rows of bits differ, rows = output
// pixels, columns = output channels.  dab_bgemm multiplies matrices of packed words with it, the BinConv layers that the
// direct 3x3 kernels do not take (other windows, strides or channel counts) convolve with it.  Bits on the matrix cores
// as in fp4_core.h.
//
// Depth is walked in units: 2 * CC consecutive dwords of a pixel (of one tap of its window), the first CC for the lower
// half of a wave's lanes, the others for the upper half, CC matrix instructions of 64 bits.  CC = 4 (16-byte loads)
// where the words of a pixel are a multiple of four, else 3, 2 or 1.
#pragma once

#include "fp4_core.h"

namespace dab {

struct BitGemm {
    const uint64_t *x;  // packed pixels, x_ld words from one to the next
    const uint64_t *w;  // filters: kFilterRows [col][w_ld] words, kFilterColumns [word][w_ld] (bgemm's column-major A)
    float *out;         // out_ld floats per pixel
    long long rows;     // pixels (below 2^31)
    int cols;           // channels
    long long x_ld, w_ld, out_ld;
    int words;          // words of a filter that meet words of a window; w_ld may leave one more, see extra_word
    int extra_word;     // kFilterRows: a filter holds one word past them (padding to 128 bits); it meets zeros
    // geometry of a window; a plain matrix is a window of one tap over an image of one row
    int H, W, OH, OW, kw, stride_h, stride_w, pad_h, pad_w;
    int tap_words;      // words of a tap (= words for a plain matrix)
    const float *a, *b, *shortcut;  // affine epilogue (shortcut has out's layout), null without
    uint32_t *bits;     // sign bits of the result, bits_ld dwords per pixel; null without
    int bits_ld;
    bool accumulate;    // out += counts
};
enum FilterLayout { kFilterRows, kFilterColumns };

// DAB_OK or an error code; `fn` names the caller in messages.
int bit_gemm(const char *fn, const BitGemm &g, FilterLayout layout, hipStream_t stream);
// Whether the limits of the window form (32-bit offsets within the packed images) hold.
bool bit_gemm_takes_images(long long image_words, long long filter_words, long long rows, int cols);

// bconv_float.hip: the convolution of fp32 input in one launch; 1 = done, 0 = not its problem (pack and convolve), negative = error.
int bconv_float_try(const float *x, int n, int h, int w, int c, const uint64_t *wgt, int words, int kh, int kw, int pad_h, int pad_w, int stride_h, int stride_w,
                    int cout, float *out, int oh, int ow, hipStream_t s);

}  // namespace dab
