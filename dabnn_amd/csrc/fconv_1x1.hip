// FpConv2D (dabnn/fconv.h:14-76) with 1x1 windows over 64, 128, 192 or 256 channels, large problems, on the f16 matrix cores with
// split operands and fp32 accuracy (common.h): the shortcut branches of down-sampling blocks, with the AvePool 2x2 stride 2 before
// them (dabnn/layers/AvePool.cpp) in the loader, and the transitions of dense blocks, with the MaxPool 2x2 stride 2
// (dabnn/layers/MaxPool.cpp) there, Affine, Relu or PRelu and the sign bits.
//
// Bound: memory, which the fp32 kernel (float_glue.hip) does not reach: its matrix instruction takes five times as long as
// three of f16, every column of blocks reads and averages the input again, and each slice of depth ends in a barrier.  Here a
// block is persistent and has 256 output channels (or 128), so the input is read once or twice.  A wave
// holds its 16 or 32 filters, split, in registers; the tiles of 16 or 32 pixels pass through two LDS buffers that all eight waves
// read.  The loads of the next tile (with a pool: of its four taps) are under way during the products of this one, and the
// pixel's channels are with 16 or 32 neighbouring lanes, which find its power of two, split and store.  Output channels are the
// rows of the matrix instruction: a lane stores four of a pixel at once.
//
// Each pixel and each filter has a power of two of its own, and a pixel that needs fp32 (an infinity, or values too far below its
// largest) gets it alone, so a result does not depend on the tile that it is made in and the pooled form is bit for bit the
// convolution of the pooled tensor.
//
// Measured against the fp32 kernel, us a launch (pixels x channels -> channels):
//   averages  49152 x 128 -> 256:  37.9 -> 31.2    24576 x 256 -> 512: 62.7 -> 41.0    in a net, 4900 x 256 -> 512: 28.4 -> 20.7
//   maxima    32768 x 256 -> 128:  24.1 (the pool by itself) + 22.8 -> 28.8
//   plain     32768 x 256 -> 128:  22.8 -> 18.6    131072 x 128 -> 128: 51.2 -> 30.2    131072 x 256 -> 256: 143.5 -> 69.5
// The last reads and writes 268 MB, 3.9 TB/s.  Error against 64-bit sums, relative to the results' root mean square:
// 2.03e-7 -> 1.11e-7 for 128 channels, 2.87e-7 -> 1.32e-7 for 256.  Filters split into LDS by every block instead, with the waves loading
// their pixels themselves: the averages 40 to 60 % slower than the fp32 kernel, since a wave waited for each of its loads.
#include <float.h>

#include "common.h"

namespace dab {

struct Fconv1x1Args {
    const float *x, *w, *bias, *aff_a, *aff_b, *slope;
    float *out, *pooled;
    uint32_t *bits;
    int relu, slope_n, out_ld, bits_ld;
    bool wide_out;  // whether four channels of the result can be stored at once
    int M, cout;
    int h, wd;  // of the input before the pool
    int cols, tiles;  // column blocks, tiles of pixels
    FastDiv div_ow, div_oh, div_cols;
};

constexpr int k1x1Threads = 512;
constexpr int kSpecialPixel = 1 << 20;  // in an exponent's place

// G: groups of 32 input channels.  CT: tiles of 16 output channels a wave.  PX: pixels a tile.
template <int G, int CT, int PX>
struct Form1x1 {
    static constexpr int K = 32 * G, channels = 8 * 16 * CT, row = K + 8, plane = PX * row;
    static constexpr int lanes = k1x1Threads / PX, quads = K / 4 / lanes;  // threads of a pixel, and their quadruples of channels
    static constexpr size_t lds = 2 * 2 * plane * 2;
};

template <int G, int CT, int PX, Pool2 POOL, int WPE>
__global__ __launch_bounds__(k1x1Threads, WPE) void fconv_1x1_kernel(const Fconv1x1Args p) {
    using F = Form1x1<G, CT, PX>;
    constexpr int K = F::K, CH = F::channels, ROW = F::row, PLANE = F::plane, LANES = F::lanes, QUADS = F::quads, MT = PX / 16;
    typedef HalfFrag8::u4 u4;
    typedef float f4 __attribute__((ext_vector_type(4)));
    extern __shared__ __attribute__((aligned(16))) uint16_t planes[];  // [buffer][hi, lo][pixel][channel]
    __shared__ __attribute__((aligned(16))) int filter_exp[CH];
    __shared__ __attribute__((aligned(16))) float per_channel[4][CH];  // bias, a, b, slope
    __shared__ int pixel_exp[2][PX];
    const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4, f_i = lane & 15;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t item = xcd_contiguous_block(blockIdx.x, gridDim.x);  // the column blocks of a pixel range on one XCD
    const int group = (int)p.div_cols.div(item), groups = (int)p.div_cols.div(gridDim.x);
    const int ch0 = ((int)item - group * p.cols) * CH;
    const int s_px = tid / LANES, s_q = tid % LANES;

    // a pixel's address in x, pooled: of its window
    auto address = [&](int pix) __attribute__((always_inline)) -> const float * {
        const int at = pix < p.M ? pix : p.M - 1;
        if constexpr (POOL != Pool2::none) {
            const uint32_t t = p.div_ow.div((uint32_t)at);
            const int ox = at - (int)t * (int)p.div_ow.d;
            const uint32_t img = p.div_oh.div(t);
            const int oy = (int)(t - img * p.div_oh.d);
            return p.x + (((size_t)img * p.h + 2 * oy) * p.wd + 2 * ox) * K;
        } else {
            return p.x + (size_t)at * K;
        }
    };
    constexpr int TAPS = POOL != Pool2::none ? 4 : 1;
    f4 raw[QUADS][TAPS];
    auto load = [&](int tile) __attribute__((always_inline)) {
        const float *base = address(tile * PX + s_px) + 4 * s_q;
#pragma unroll
        for (int k = 0; k < QUADS; ++k)
#pragma unroll
            for (int t = 0; t < TAPS; ++t) raw[k][t] = *reinterpret_cast<const f4 *>(base + (t >> 1) * (size_t)p.wd * K + (t & 1) * K + 4 * LANES * k);
    };
    // as pool_vec4_kernel adds and scales, or compares
    auto of_window = [](const f4 (&v)[TAPS]) __attribute__((always_inline)) -> f4 {
        if constexpr (POOL == Pool2::average) {
            return ((((f4{0.f, 0.f, 0.f, 0.f} + v[0]) + v[1]) + v[2]) + v[3]) * 0.25f;
        } else if constexpr (POOL == Pool2::largest) {
            f4 m = {-FLT_MAX, -FLT_MAX, -FLT_MAX, -FLT_MAX};
#pragma unroll
            for (int t = 0; t < TAPS; ++t)
#pragma unroll
                for (int e = 0; e < 4; ++e) m[e] = v[t][e] > m[e] ? v[t][e] : m[e];
            return m;
        } else {
            return v[0];
        }
    };
    auto stage = [&](int tile, int buf) __attribute__((always_inline)) {
        f4 v[QUADS];
        float largest = 0.f;
        uint32_t smallest = ~0u;
#pragma unroll
        for (int k = 0; k < QUADS; ++k) {
            v[k] = of_window(raw[k]);
            largest = max3_magnitude(v[k].z, v[k].w, max3_magnitude(v[k].x, v[k].y, largest));
            smallest = smallest_magnitude(smallest_magnitude(smallest, v[k].x, v[k].y), v[k].z, v[k].w);
        }
        if constexpr (POOL == Pool2::average) {
            if (p.pooled != nullptr && ch0 == 0 && tile * PX + s_px < p.M) {
#pragma unroll
                for (int k = 0; k < QUADS; ++k) *reinterpret_cast<f4 *>(p.pooled + (size_t)(tile * PX + s_px) * K + 4 * (s_q + LANES * k)) = v[k];
            }
        }
#pragma unroll
        for (int step = 1; step < LANES; step *= 2) largest = max3_magnitude(__shfl_xor(largest, step), 0.f, largest);
        const int e = f16_scale_exponent(largest);
        const float up = exp2_int(e), up11 = exp2_int(e + 11);
        uint16_t *at = planes + buf * 2 * PLANE + s_px * ROW + 4 * s_q;
#pragma unroll
        for (int k = 0; k < QUADS; ++k) {
            const HalfPair a = split_pair_f16(v[k].x, v[k].y, up, up11), b = split_pair_f16(v[k].z, v[k].w, up, up11);
            *reinterpret_cast<uint2 *>(at + 4 * LANES * k) = make_uint2(a.hi, b.hi);
            *reinterpret_cast<uint2 *>(at + 4 * LANES * k + PLANE) = make_uint2(a.lo, b.lo);
        }
        const uint64_t odd = __builtin_amdgcn_ballot_w64(!(largest < __builtin_inff()) || too_small_for_f16(smallest, e));
        const uint64_t mine = (LANES == 64 ? ~0ull : ((1ull << (LANES & 63)) - 1)) << (lane & ~(LANES - 1));
        if (s_q == 0) pixel_exp[buf][s_px] = (odd & mine) != 0 ? kSpecialPixel : e;
    };

    const int first = group;
    load(first);
    for (int c = tid; c < CH; c += k1x1Threads) {
        const bool ok = ch0 + c < p.cout;
        per_channel[0][c] = ok && p.bias ? p.bias[ch0 + c] : 0.f;
        per_channel[1][c] = ok && p.aff_a ? p.aff_a[ch0 + c] : 0.f;
        per_channel[2][c] = ok && p.aff_a ? p.aff_b[ch0 + c] : 0.f;
        per_channel[3][c] = ok && p.slope ? p.slope[p.slope_n == 1 ? 0 : ch0 + c] : 0.f;
    }
    const int wave_ch = wave * 16 * CT;
    const bool idle = ch0 + wave_ch >= p.cout;
    HalfFrag8 filter[CT][G];
    bool w_special = false;
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) {
        const int c = wave_ch + ct * 16 + f_i;
        const bool ok = ch0 + c < p.cout;
        const f4 *src = reinterpret_cast<const f4 *>(p.w + (size_t)(ok ? ch0 + c : 0) * K + 8 * g);
        f4 v[2 * G];
        float largest = 0.f;
        uint32_t smallest = ~0u;
#pragma unroll
        for (int k = 0; k < 2 * G; ++k) v[k] = src[8 * (k >> 1) + (k & 1)];
#pragma unroll
        for (int k = 0; k < 2 * G; ++k) {
            if (!ok) v[k] = f4{0.f, 0.f, 0.f, 0.f};
            largest = max3_magnitude(v[k].z, v[k].w, max3_magnitude(v[k].x, v[k].y, largest));
            smallest = smallest_magnitude(smallest_magnitude(smallest, v[k].x, v[k].y), v[k].z, v[k].w);
        }
        largest = max3_magnitude(__shfl_xor(largest, 16), 0.f, largest);
        largest = max3_magnitude(__shfl_xor(largest, 32), 0.f, largest);
        const int e = f16_scale_exponent(largest);
        const float up = exp2_int(e), up11 = exp2_int(e + 11);
        w_special |= __builtin_amdgcn_ballot_w64(!(largest < __builtin_inff()) || too_small_for_f16(smallest, e)) != 0;
#pragma unroll
        for (int k = 0; k < G; ++k)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const f4 u = v[2 * k + h];
                const HalfPair a = split_pair_f16(u.x, u.y, up, up11), b = split_pair_f16(u.z, u.w, up, up11);
                filter[ct][k].hi[2 * h] = a.hi, filter[ct][k].hi[2 * h + 1] = b.hi;
                filter[ct][k].lo[2 * h] = a.lo, filter[ct][k].lo[2 * h + 1] = b.lo;
            }
        if (g == 0) filter_exp[c] = e;
    }
    stage(first, 0);
    __syncthreads();

    int buf = 0;
    for (int tile = first; tile < p.tiles; tile += groups) {
        const bool more = tile + groups < p.tiles;
        if (more) load(tile + groups);
        if (!idle) {
            f32x4w acc[CT][MT], cross[CT][MT];
#pragma unroll
            for (int ct = 0; ct < CT; ++ct)
#pragma unroll
                for (int m = 0; m < MT; ++m) acc[ct][m] = cross[ct][m] = f32x4w{0.f, 0.f, 0.f, 0.f};
            const uint16_t *at = planes + buf * 2 * PLANE + f_i * ROW + 8 * g;
            auto h8 = [](u4 w) { return __builtin_bit_cast(f16x8, w); };
#pragma unroll
            for (int k = 0; k < G; ++k) {
                HalfFrag8 px[MT];
#pragma unroll
                for (int m = 0; m < MT; ++m)
                    px[m] = {*reinterpret_cast<const u4 *>(at + m * 16 * ROW + 32 * k), *reinterpret_cast<const u4 *>(at + m * 16 * ROW + 32 * k + PLANE)};
#pragma unroll
                for (int ct = 0; ct < CT; ++ct)
#pragma unroll
                    for (int m = 0; m < MT; ++m)
                        cross[ct][m] = __builtin_amdgcn_mfma_f32_16x16x32_f16(h8(filter[ct][k].lo), h8(px[m].hi), cross[ct][m], 0, 0, 0);
#pragma unroll
                for (int ct = 0; ct < CT; ++ct)
#pragma unroll
                    for (int m = 0; m < MT; ++m)
                        acc[ct][m] = __builtin_amdgcn_mfma_f32_16x16x32_f16(h8(filter[ct][k].hi), h8(px[m].hi), acc[ct][m], 0, 0, 0);
#pragma unroll
                for (int ct = 0; ct < CT; ++ct)
#pragma unroll
                    for (int m = 0; m < MT; ++m)
                        cross[ct][m] = __builtin_amdgcn_mfma_f32_16x16x32_f16(h8(filter[ct][k].hi), h8(px[m].lo), cross[ct][m], 0, 0, 0);
            }
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                const int pe = pixel_exp[buf][m * 16 + f_i], pix = tile * PX + m * 16 + f_i;
                const bool special = w_special || pe == kSpecialPixel;
                const bool any = __builtin_amdgcn_ballot_w64(special) != 0;
#pragma unroll
                for (int ct = 0; ct < CT; ++ct) {
#pragma clang fp contract(off)
                    const int c = wave_ch + ct * 16 + 4 * g, co = ch0 + c;
                    const int4 fe = *reinterpret_cast<const int4 *>(filter_exp + c);
                    const int exps[4] = {fe.x, fe.y, fe.z, fe.w};
                    f32x4w v;
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        v[e] = __builtin_ldexpf(__builtin_fmaf(cross[ct][m][e], 1.f / 2048.f, acc[ct][m][e]), -(pe + exps[e]));
                    if (any) {
                        // a pixel with an infinity or values too far below its largest, or such a filter: in fp32, in two sums
                        const int row = ch0 + wave_ch + ct * 16 + f_i;
                        const float *w_at = p.w + (size_t)(row < p.cout ? row : 0) * K + 8 * g, *x_at = address(pix) + 8 * g;
                        f32x4w even = f32x4w{0.f, 0.f, 0.f, 0.f}, odd = even;
#pragma unroll 1
                        for (int k = 0; k < 2 * G; ++k) {
                            const size_t off = 32 * (k >> 1) + 4 * (k & 1);
                            f4 tap[TAPS];
#pragma unroll
                            for (int t = 0; t < TAPS; ++t) tap[t] = *reinterpret_cast<const f4 *>(x_at + (t >> 1) * (size_t)p.wd * K + (t & 1) * K + off);
                            const f4 u = of_window(tap), w = *reinterpret_cast<const f4 *>(w_at + off);
                            even = __builtin_amdgcn_mfma_f32_16x16x4f32(w.x, u.x, even, 0, 0, 0);
                            odd = __builtin_amdgcn_mfma_f32_16x16x4f32(w.y, u.y, odd, 0, 0, 0);
                            even = __builtin_amdgcn_mfma_f32_16x16x4f32(w.z, u.z, even, 0, 0, 0);
                            odd = __builtin_amdgcn_mfma_f32_16x16x4f32(w.w, u.w, odd, 0, 0, 0);
                        }
                        if (special) v = even + odd;
                    }
                    // the layers' order: bias, Affine (two roundings), Relu or PRelu
                    if (p.bias) v = v + *reinterpret_cast<const f32x4w *>(&per_channel[0][c]);
                    if (p.aff_a) {
                        v = v * *reinterpret_cast<const f32x4w *>(&per_channel[1][c]);
                        v = v + *reinterpret_cast<const f32x4w *>(&per_channel[2][c]);
                    }
                    if (p.slope) {
                        const f32x4w slope = *reinterpret_cast<const f32x4w *>(&per_channel[3][c]);
#pragma unroll
                        for (int e = 0; e < 4; ++e) v[e] = v[e] < 0.f ? v[e] * slope[e] : v[e];
                    } else if (p.relu) {
#pragma unroll
                        for (int e = 0; e < 4; ++e) v[e] = v[e] < 0.f ? 0.f : v[e];  // std::max(v, 0.f): a NaN stays
                    }
                    const bool ok = pix < p.M && co < p.cout;
                    if (ok) {
                        float *d = p.out + (size_t)pix * p.out_ld + co;
                        if (p.wide_out) {
                            *reinterpret_cast<f32x4w *>(d) = v;
                        } else {
#pragma unroll
                            for (int e = 0; e < 4; ++e) d[e] = v[e];
                        }
                    }
                    if (p.bits) {
                        // sixteen channels of a pixel are four lanes' nibbles
                        uint32_t all = sign_nibble(make_float4(v[0], v[1], v[2], v[3])) << (4 * g);
                        all |= (uint32_t)__shfl_xor((int)all, 16);
                        all |= (uint32_t)__shfl_xor((int)all, 32);
                        if (g == 0 && ok) reinterpret_cast<uint16_t *>(p.bits + (size_t)pix * p.bits_ld)[co >> 4] = (uint16_t)all;
                    }
                }
            }
        }
        if (more) stage(tile + groups, buf ^ 1);
        __syncthreads();
        buf ^= 1;
    }
}

// Loading and splitting a block's filters takes 2 (64 channels, 16 filters a wave) to 11 us (256 channels, 32 filters) before its first
// product, so a launch must have work enough to make up for it.  Times of the fp32 kernel over this one's, 64 to 512 output channels,
// plain and averages: from 192 channels on 1.02 to 1.27 at pixels * channels * outputs = 5 * 2^26, 0.93 to 1.05 at three quarters of
// that; with 64 and 128 channels 1.0 to 1.3 at 2^29 (outputs of 256 and more), 0.89 to 1.27 at 3/4; narrow outputs, which are bound
// by the input: 0.98 to 1.19 at pixels * channels = 4 M.
bool fconv_1x1_takes(long long M, int K, int cout) {
    if (K % 64 != 0 || K > 256 || cout < 64 || cout % 32 != 0 || M < 1024) return false;
    return M * K >= 4ll << 20 || M * K * cout >= (K >= 192 ? 5ll << 26 : 1ll << 29);
}

int fconv_1x1_try(const float *x, long long M, int K, const float *wgt, const float *bias, const float *aff_a, const float *aff_b, int relu, const float *slope,
                  int slope_n, int cout, float *out, int out_ld, uint32_t *bits, int bits_ld, float *pooled, Pool2 kind, const Pool2Window *pool, hipStream_t s) {
    if (!fconv_1x1_takes(M, K, cout)) return 0;
    if ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(wgt) | reinterpret_cast<uintptr_t>(pooled)) % 16 != 0) return 0;
    Fconv1x1Args a;
    a.x = x, a.w = wgt, a.bias = bias, a.aff_a = aff_a, a.aff_b = aff_b, a.slope = slope, a.out = out, a.pooled = pooled, a.bits = bits;
    a.relu = relu, a.slope_n = slope_n, a.out_ld = out_ld, a.bits_ld = bits_ld;
    a.wide_out = out_ld % 4 == 0 && reinterpret_cast<uintptr_t>(out) % 16 == 0;
    a.M = (int)M, a.cout = cout, a.h = 0, a.wd = 0;
    if (pool) a.h = pool->h, a.wd = pool->w, a.div_ow = FastDiv((uint32_t)pool->ow), a.div_oh = FastDiv((uint32_t)pool->oh);
    const int cus = simd_count() / 4;
    auto launch = [&](auto groups, auto channels, auto pixels, auto pooling, auto waves) {
        constexpr int G = decltype(groups)::value, CT = decltype(channels)::value, PX = decltype(pixels)::value, WPE = decltype(waves)::value;
        constexpr Pool2 POOL = decltype(pooling)::value;
        using F = Form1x1<G, CT, PX>;
        constexpr auto kernel = fconv_1x1_kernel<G, CT, PX, POOL, WPE>;
        a.cols = (cout + F::channels - 1) / F::channels, a.tiles = (int)((M + PX - 1) / PX);
        a.div_cols = FastDiv((uint32_t)a.cols);
        const int most = cus * (WPE / 2) / a.cols > 0 ? cus * (WPE / 2) / a.cols : 1, rounds = (a.tiles + most - 1) / most;
        const dim3 grid((unsigned)((a.tiles + rounds - 1) / rounds * a.cols));
        const int rc = allow_dynamic_lds<kernel>("fconv_1x1", F::lds);
        if (rc != DAB_OK) return rc;
        hipLaunchKernelGGL(kernel, grid, dim3(k1x1Threads), F::lds, s, a);
        return hipGetLastError() == hipSuccess ? 1 : fail(DAB_EHIP, "fconv_1x1: launch failed");
    };
    using std::integral_constant;
    constexpr integral_constant<int, 1> one;
    constexpr integral_constant<int, 2> two;
    constexpr integral_constant<int, 4> four;
    constexpr integral_constant<int, 16> px16;
    constexpr integral_constant<int, 32> px32;
    constexpr integral_constant<int, 6> six;
    constexpr integral_constant<int, 8> eight;
    constexpr integral_constant<Pool2, Pool2::none> plain;
    constexpr integral_constant<Pool2, Pool2::average> average;
    constexpr integral_constant<Pool2, Pool2::largest> largest;
    // Sixteen filters a wave where 32 do not fill the outputs, and where blocks of 256 channels would have three tiles of
    // pixels or fewer each: splitting half of the filters saves more than reading the pixels twice costs (us with 16 / 32 a
    // wave, 256 -> 256 channels: 8192 pixels 12.3 / 15.7, 16384 18.1 / 20.6; 256 -> 512 with averages: 8192 22.1 / 23.0,
    // 16384, four tiles, 35.8 / 32.6).
    // (64 output channels leave half of the waves without products; the time is the memory's)
    const bool narrow = cout <= 128 || (M + 31) / 32 * ((cout + 255) / 256) <= 3ll * cus;
    switch (kind) {
        case Pool2::none:
            if (K == 64) return narrow ? launch(two, one, px32, plain, four) : launch(two, two, px32, plain, four);
            if (K == 128) return narrow ? launch(four, one, px32, plain, four) : launch(four, two, px32, plain, two);
            if (K == 192) return narrow ? launch(six, one, px32, plain, two) : launch(six, two, px32, plain, two);
            return narrow ? launch(eight, one, px32, plain, two) : launch(eight, two, px32, plain, two);
        case Pool2::average:
            if (K == 64) return narrow ? launch(two, one, px32, average, four) : launch(two, two, px32, average, two);
            if (K == 128) return narrow ? launch(four, one, px32, average, two) : launch(four, two, px32, average, two);
            if (K == 192) return narrow ? launch(six, one, px32, average, two) : launch(six, two, px32, average, two);
            return narrow ? launch(eight, one, px16, average, two) : launch(eight, two, px16, average, two);
        default:
            if (K == 64) return narrow ? launch(two, one, px32, largest, four) : launch(two, two, px32, largest, two);
            if (K == 128) return narrow ? launch(four, one, px32, largest, two) : launch(four, two, px32, largest, two);
            if (K == 192) return narrow ? launch(six, one, px32, largest, two) : launch(six, two, px32, largest, two);
            return narrow ? launch(eight, one, px16, largest, two) : launch(eight, two, px16, largest, two);
    }
}

}  // namespace dab
