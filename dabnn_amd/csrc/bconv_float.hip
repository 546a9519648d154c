// Binary convolution of fp32 input in one launch: pack_mat and the convolution over any window behind it
// (dabnn/layers/BinConv.cpp:144-165) for problems whose two launches would cost more than the work.
//
// A block makes R whole output rows of one image for 64 output channels.  It packs the input rows under them into LDS (a word
// is the lane mask of one compare, dabnn/bitpack.h:254-293), zero words around them, and the 64 filters beside them; then each
// wave multiplies tiles of 32 pixels x 64 channels on the fp4 matrix instruction (fp4_core.h), or a share of their depth
// where there are fewer tiles than waves.  Rows that two blocks need are packed by both, and once more for every 64 output
// channels: what that costs decides where this kernel ends (plan_float_conv).
// Bound by latency: one launch from the host (4.3 us with the call), one round trip for the input and filters, one pass over
// the depth, the store.  So all of a wave's input is asked for at once (48 words: with 32 at a time 16 x 56 x 56 x 64 took 8.1
// us instead of 6.6), in groups of 16 so that small strips do not pack what is not there (1 to 1.5 us of them).
#include <functional>

#include "bgemm_core.h"
#include "fp4_core.h"

namespace dab {

struct FloatBconvArgs {
    const float *x;
    const uint64_t *w;
    float *out;
    int H, W, CW, OH, OW, cout;
    int stride_h, stride_w, pad_h, pad_w;
    int kw, taps;
    int words;         // of a filter, the converter's padding word included
    int rows, bands;   // output rows of a block, blocks one below the other
    int in_rows;        // input rows in LDS
    int px_bytes, row_bytes, filter_bytes;  // LDS strides
    int groups;        // of 64 channels
    int filters_at, part_at;                // LDS offsets
    uint32_t w_words;  // in the filter tensor
    uint32_t row_words;  // packed words of an input row
    FastDiv div_groups, div_bands, div_words, div_row_words, div_cw, div_ow, div_kw;
};

constexpr size_t kFloatConvLds = 152u << 10;
// Where packing and convolving in two launches becomes the faster way.  Random layers, one call after another from the host, estimate /
// one launch / two: 4.0 k cycles 4.3 us / 7.2 (3 x 6 x 8 x 64 -> 40, 3x3), 4.7 k 4.9 / 7.4 (41 x 41 x 256 -> 128, 1x1), 5.5 k 5.7 / 8.6
// (227 x 6 x 6 x 128 -> 8, 5x5), 6.9 k 6.6 / 8.0 (16 x 56 x 56 x 64 -> 64, 3x3), 7.2 k 6.6 / 7.3, 7.5 k 7.2 / 7.3, 8.0 k 8.3 / 7.2.
constexpr double kFloatConvCycles = 7200;

constexpr int kFloatConvThreads = 512, kFloatConvWaves = kFloatConvThreads / 64;

// DS: waves that share a tile's depth.
template <int DS>
__global__ __launch_bounds__(kFloatConvThreads) void bconv_float_kernel(const FloatBconvArgs p) {
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    const int tid = threadIdx.x, lane = tid & 63, half = lane >> 5, l32 = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // the channel groups of a band, and neighbouring bands, on one XCD: they read the same input
    const uint32_t item = xcd_contiguous_block(blockIdx.x, gridDim.x);
    const uint32_t strip = p.div_groups.div(item);
    const int ch0 = (int)(item - strip * p.groups) * 64;
    const int img = (int)p.div_bands.div(strip), band = (int)strip - img * p.bands;
    const int oy0 = band * p.rows, rows = p.OH - oy0 < p.rows ? p.OH - oy0 : p.rows;

    // The rows of the input that lie in the image, as one run of words: wave by wave 48 at a time, the first ones and the first
    // filter words asked for before anything else is done.
    const int iy0 = oy0 * p.stride_h - p.pad_h, first = iy0 < 0 ? -iy0 : 0;
    const int need = p.in_rows - (p.rows - rows) * p.stride_h, last = iy0 + need > p.H ? p.H - iy0 : need;
    const int total = last > first ? (last - first) * (int)p.row_words : 0;
    const float *src = p.x + ((size_t)img * p.H + (iy0 + first)) * p.row_words * 64 + lane;
    constexpr int kAtOnce = 48;
    float v[kAtOnce];
    auto fetch = [&](int j0) {
#pragma unroll
        for (int g = 0; g < kAtOnce; g += 16) {
            if (j0 + g >= total) break;
#pragma unroll
            for (int k = g; k < g + 16; ++k) v[k] = src[(size_t)(j0 + k < total ? j0 + k : total - 1) * 64];
        }
    };
    fetch(wave * kAtOnce);
    // zero words where nothing is packed: around the image
    for (int i = tid * 16; i < p.filters_at; i += kFloatConvThreads * 16) *reinterpret_cast<u32x4 *>(lds + i) = u32x4{0u, 0u, 0u, 0u};
    // the filters: contiguous in memory, one row each in LDS
    const int filter_words = 64 * p.words;
    const uint32_t w_first = (uint32_t)ch0 * p.words;
#pragma unroll 16
    for (int i = tid; i < filter_words; i += kFloatConvThreads) {
        const uint32_t f = p.div_words.div(i);
        const uint64_t word = w_first + i < p.w_words ? p.w[w_first + i] : 0;
        *reinterpret_cast<uint64_t *>(lds + p.filters_at + f * p.filter_bytes + (i - f * p.words) * 8) = word;
    }
    __syncthreads();
    for (int j0 = wave * kAtOnce; j0 < total; j0 += kFloatConvWaves * kAtOnce) {
        uint32_t lo = 0, hi = 0;
#pragma unroll
        for (int g = 0; g < kAtOnce; g += 16) {
            if (j0 + g >= total) break;
#pragma unroll
            for (int k = g; k < g + 16; ++k) {
                const uint64_t mask = __ballot(v[k] > 0.f);
                lo = dab_writelane((uint32_t)mask, k, lo);
                hi = dab_writelane((uint32_t)(mask >> 32), k, hi);
            }
        }
        fetch(j0 + kFloatConvWaves * kAtOnce);
        const int j = j0 + lane;
        if (lane < kAtOnce && j < total) {
            const uint32_t r = p.div_row_words.div(j), in_row = j - r * p.row_words;
            const uint32_t col = p.div_cw.div(in_row), c = in_row - col * p.CW;
            *reinterpret_cast<u32x2 *>(lds + (first + r) * p.row_bytes + (col + p.pad_w) * p.px_bytes + c * 8) = u32x2{lo, hi};
        }
    }
    __syncthreads();

    const int pixels = rows * p.OW, tiles = (pixels + 31) / 32;
    const size_t out_first = ((size_t)img * p.OH + oy0) * p.OW * p.cout;
    const __amdgpu_buffer_rsrc_t ro = make_rsrc(p.out + out_first, (uint32_t)(pixels * p.cout) * 4u);
    int lane_off[2];
#pragma unroll
    for (int n = 0; n < 2; ++n) {
        const int ch = ch0 + n * 32 + l32;
        lane_off[n] = ch < p.cout ? (half * 4 * p.cout + ch) * 4 : (int)0x80000000;
    }
    const float half_depth = 32.f * p.words;  // both operands are +-1: differing bits are (depth - sum) / 2
    const int slice = wave % DS, depth = p.taps * p.CW;
    const int from = depth * slice / DS, to = depth * (slice + 1) / DS;
    const unsigned char *filter = lds + p.filters_at + l32 * p.filter_bytes + half * 4;
    const int n_off = 32 * p.filter_bytes;
    for (int t0 = 0; t0 < tiles; t0 += kFloatConvWaves / DS) {
        const int tile = t0 + wave / DS;
        f32x16m acc[2];
#pragma unroll
        for (int n = 0; n < 2; ++n)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[n][e] = 0.f;
        if (DS > 1 || tile < tiles) {
            int px = tile * 32 + l32;
            px = px < pixels ? px : pixels - 1;
            const int oy = (int)p.div_ow.div(px), ox = px - oy * p.OW;
            const unsigned char *window = lds + oy * p.stride_h * p.row_bytes + ox * p.stride_w * p.px_bytes + half * 4;
            // four words of the depth at a time, the next four on their way from LDS meanwhile
            constexpr int kWords = 4;
            struct Words {
                uint32_t a[kWords], b[2][kWords];
            };
            int tap = (int)p.div_cw.div(from), c = from - tap * p.CW;
            int ky = (int)p.div_kw.div(tap), kx = tap - ky * p.kw;
            int at = ky * p.row_bytes + kx * p.px_bytes + c * 8;  // of the window's next word
            auto read = [&](Words &q, int word) {
#pragma unroll
                for (int i = 0; i < kWords; ++i) {
                    if (word + i >= to) break;
                    q.a[i] = *reinterpret_cast<const uint32_t *>(window + at);
                    q.b[0][i] = *reinterpret_cast<const uint32_t *>(filter + (word + i) * 8);
                    q.b[1][i] = *reinterpret_cast<const uint32_t *>(filter + n_off + (word + i) * 8);
                    at += 8;
                    if (++c == p.CW) {
                        c = 0;
                        at += p.px_bytes - p.CW * 8;
                        if (++kx == p.kw) {
                            kx = 0;
                            at += p.row_bytes - p.kw * p.px_bytes;
                        }
                    }
                }
            };
            auto multiply = [&](uint32_t a_bits, uint32_t b0, uint32_t b1) {
                const i32x8 a = bitspm1(a_bits);
                mfma_fp4<32>(acc[0], a, bitspm1(b0));
                mfma_fp4<32>(acc[1], a, bitspm1(b1));
            };
            Words now, next;
            read(now, from);
            for (int word = from; word < to; word += kWords) {
                read(next, word + kWords);
#pragma unroll
                for (int i = 0; i < kWords; ++i) {
                    if (word + i >= to) break;
                    multiply(now.a[i], now.b[0][i], now.b[1][i]);
                }
                now = next;
            }
            if (slice == DS - 1 && p.words > depth)  // the filters' padding word meets a zero word
                multiply(0u, *reinterpret_cast<const uint32_t *>(filter + depth * 8), *reinterpret_cast<const uint32_t *>(filter + n_off + depth * 8));
        }
        const int tile_off = tile * 32 * p.cout * 4;
        auto store = [&](int n, int e, float sum) {
            __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, half_depth - 0.5f * sum), ro, lane_off[n],
                                                  tile_off + (8 * (e / 4) + e % 4) * p.cout * 4, kStoreThrough);
        };
        if constexpr (DS == 1) {
            if (tile < tiles) {
#pragma unroll
                for (int e = 0; e < 16; ++e)
#pragma unroll
                    for (int n = 0; n < 2; ++n) store(n, e, acc[n][e]);
            }
        } else {
            // every wave adds up and stores its share of the 32 registers
            float *part = reinterpret_cast<float *>(lds + p.part_at) + (wave / DS) * (DS * 32 * 64);
#pragma unroll
            for (int n = 0; n < 2; ++n)
#pragma unroll
                for (int e = 0; e < 16; ++e) part[(slice * 32 + n * 16 + e) * 64 + lane] = acc[n][e];
            __syncthreads();
            const int n = slice / (DS / 2), e0 = (slice % (DS / 2)) * (32 / DS);
            if (tile < tiles) {
#pragma unroll
                for (int k = 0; k < 32 / DS; ++k) {
                    float sum = 0.f;
#pragma unroll
                    for (int q = 0; q < DS; ++q) sum += part[(q * 32 + n * 16 + e0 + k) * 64 + lane];
                    store(n, e0 + k, sum);
                }
            }
            if (t0 + kFloatConvWaves / DS < tiles) __syncthreads();
        }
    }
}

template <int DS>
static int launch_float_conv(const FloatBconvArgs &a, unsigned grid, size_t lds, hipStream_t s) {
    if (lds > (64u << 10)) {
        const int rc = allow_dynamic_lds<bconv_float_kernel<DS>>("dab_binconv_forward", kFloatConvLds);
        if (rc != DAB_OK) return rc;
    }
    hipLaunchKernelGGL((bconv_float_kernel<DS>), dim3(grid), dim3(kFloatConvThreads), lds, s, a);
    DAB_LAUNCH_CHECK();
    return DAB_OK;
}

struct FloatConvPlan {
    FloatBconvArgs a;
    int ds;
    unsigned grid;
    size_t lds;
};

// The cheapest strip height, and whether the launch beats packing and convolving in two.  Estimated in cycles of a CU: what a
// block packs and loads at 48 bytes a cycle, 160 for 64 depths of a tile of 32 x 64, 600 to store one.
static bool plan_float_conv(FloatConvPlan &plan, const float *x, int n, int h, int w, int c, const uint64_t *wgt, int words, int kh, int kw, int pad_h, int pad_w,
                            int stride_h, int stride_w, int cout, float *out, int oh, int ow) {
    const int cw = c / 64, taps = kh * kw, groups = (cout + 63) / 64, cus = simd_count() / 4;
    const long long in_w = (long long)w + 2 * pad_w, px_bytes = (cw | 1) * 8ll, row_bytes = in_w * px_bytes, filter_bytes = (words | 1) * 8ll;
    if ((long long)h * w * cw >= (1 << 28) || (long long)cout * words >= (1 << 28) || (long long)oh * ow * cout >= (1 << 28) || in_w >= (1 << 20) || filter_bytes * 64 > (long long)kFloatConvLds)
        return false;
    const long long filters = 64 * filter_bytes;
    double best = 1e30;
    for (int r = 1; r < 2 * oh; r *= 2) {
        const int rows = r < oh ? r : oh, in_rows = (rows - 1) * stride_h + kh;
        const int tiles = (rows * ow + 31) / 32, ds = tiles > 4 ? 1 : tiles > 2 ? 2 : tiles > 1 ? 4 : 8;
        const long long packed = (in_rows * row_bytes + 8 + 15) / 16 * 16, lds = packed + filters + (ds > 1 ? kFloatConvWaves * 32 * 64 * 4 : 0);
        if (lds > (long long)kFloatConvLds) break;
        const int bands = (oh + rows - 1) / rows;
        const long long blocks = (long long)n * bands * groups;
        if (blocks >= (1ll << 23)) continue;
        const double packing = ((double)(in_rows < h ? in_rows : h) * w * cw * 256 + 64.0 * words * 8) / 48;
        const double counting = ((tiles * ds + kFloatConvWaves - 1) / kFloatConvWaves) * (160.0 * taps * cw / ds + 600);
        const double cycles = 3000 + (double)((blocks + cus - 1) / cus) * (packing + counting);
        if (cycles >= best) continue;
        best = cycles;
        plan.ds = ds, plan.lds = (size_t)lds, plan.grid = (unsigned)blocks;
        plan.a.rows = rows, plan.a.bands = bands, plan.a.in_rows = in_rows;
        plan.a.filters_at = (int)packed, plan.a.part_at = (int)(packed + filters);
    }
    if (best > kFloatConvCycles || best >= 1e30) return false;
    FloatBconvArgs &a = plan.a;
    a.x = x, a.w = wgt, a.out = out;
    a.H = h, a.W = w, a.CW = cw, a.OH = oh, a.OW = ow, a.cout = cout;
    a.stride_h = stride_h, a.stride_w = stride_w, a.pad_h = pad_h, a.pad_w = pad_w;
    a.kw = kw, a.taps = taps, a.words = words;
    a.px_bytes = (int)px_bytes, a.row_bytes = (int)row_bytes, a.filter_bytes = (int)filter_bytes;
    a.groups = groups, a.w_words = (uint32_t)((long long)cout * words), a.row_words = (uint32_t)(w * cw);
    a.div_groups = FastDiv((uint32_t)groups), a.div_bands = FastDiv((uint32_t)a.bands), a.div_words = FastDiv((uint32_t)words);
    a.div_row_words = FastDiv(a.row_words), a.div_cw = FastDiv((uint32_t)cw), a.div_ow = FastDiv((uint32_t)ow), a.div_kw = FastDiv((uint32_t)kw);
    return true;
}

int bconv_float_try(const float *x, int n, int h, int w, int c, const uint64_t *wgt, int words, int kh, int kw, int pad_h, int pad_w, int stride_h, int stride_w,
                    int cout, float *out, int oh, int ow, hipStream_t s) {
    FloatConvPlan p;
    // (with a stride of two and more the output of a window larger than the padded image is rounded up to one pixel)
    if (h + 2ll * pad_h < kh || w + 2ll * pad_w < kw) return 0;
    // A layer run in place, or into a buffer that its input reaches into: here blocks store while others still read their rows.
    const float *x_end = x + (size_t)n * h * w * c, *out_end = out + (size_t)n * oh * ow * cout;
    if (std::less<const float *>()(x, out_end) && std::less<const float *>()(out, x_end)) return 0;
    if ((reinterpret_cast<uintptr_t>(wgt) & 7) != 0 || (reinterpret_cast<uintptr_t>(out) & 3) != 0 || (reinterpret_cast<uintptr_t>(x) & 3) != 0) return 0;
    if (!plan_float_conv(p, x, n, h, w, c, wgt, words, kh, kw, pad_h, pad_w, stride_h, stride_w, cout, out, oh, ow)) return 0;
    const int rc = p.ds == 1   ? launch_float_conv<1>(p.a, p.grid, p.lds, s)
                   : p.ds == 2 ? launch_float_conv<2>(p.a, p.grid, p.lds, s)
                   : p.ds == 4 ? launch_float_conv<4>(p.a, p.grid, p.lds, s)
                               : launch_float_conv<8>(p.a, p.grid, p.lds, s);
    return rc == DAB_OK ? 1 : rc;
}

}  // namespace dab
