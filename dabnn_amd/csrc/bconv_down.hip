// The first layer of a down-sampling block with its shortcut branch, in one launch:
//   out = a * bconv3x3(sign(x), stride 2, pad 1) + b + (sa * (conv1x1(avepool2x2(x)) + bias) + sb)
// (dabnn/layers/BinConv.cpp:144-191, Affine.cpp:10-23, AvePool.cpp:84-123, FloatConv.cpp, Add.cpp:7-17), with the sign bits of
// the result.  64, 128 or 256 input channels, even height and width.
//
// As two launches the branch's blob is written by one and read by the other; here it stays in the accumulators of the fp32 matrix
// instruction, which lie like those of the fp4 one that counts (fp4_core.h): lane = channel, register = pixel.  Its values are only
// written for who asks for them (`sc_out`).
//
// Three kernels, chosen by the number of 32-pixel x 32-channel pieces of the output (pick_down has both sides of its lines):
//   staged  few pieces: a block is one tile, all its operands are asked for at once, four or eight waves share the branch's depth
//   tile    a block is 32 pixels x 128 channels, a wave 32 channels
//   walk    many pieces, 64 and 128 input channels: a wave keeps the filters of 32 channels, blocks walk over pixel tiles
// All of them add the branch's products in dab_ave_pool2_fconv1x1's order, so its values are that call's to the bit.
// One Bi-Real-18 pass, the three layers as two launches each / in one (us, in a graph): batch 1 5.9 + 6.9 + 8.1 / 3.7 + 3.5 + 4.0, batch
// 6 9.1 + 8.9 + 9.0 / 5.6 + 5.8 + 5.7, batch 40 21 + 18 + 21 / 14.1 + 11.8 + 10.5, batch 256 96 + 67 + 59 / 61 + 55 + 53.
#include "fp4_core.h"

namespace dab {

struct BconvDownArgs {
    const uint64_t *x;   // sign bits of xf
    const float *xf;     // or the pooled tensor, for the kernels built for that
    const uint64_t *w;   // of the binary convolution
    const float *ea, *eb;
    const float *sw;     // [cout][cin] of the branch
    const float *bias, *sa, *sb;  // may be null: bias, and sa with sb
    float *sc_out;       // the branch's result, or null
    float *out;
    uint32_t *bits;      // or null
    int total;           // output pixels
    int H, W, OH, OW, cout, cols;
    uint32_t x_bytes, w_bytes;
    FastDiv div_ow, div_oh, div_cols;
};

constexpr int kDownOutside = (int)0x80000000;  // beyond any descriptor

struct DownPixel {
    int n, oy, ox;
    __device__ __forceinline__ DownPixel(const BconvDownArgs &p, int pix) {
        const uint32_t t = p.div_ow.div((uint32_t)pix);
        ox = pix - (int)t * p.OW;
        n = (int)p.div_oh.div(t);
        oy = (int)t - n * p.OH;
    }
};

// ave_pool_fallback (dabnn/layers/AvePool.cpp:84-123) for a 2x2 window: the taps added to zero in row-major order, divided by 4
__device__ __forceinline__ f32x4m pool_taps(const f32x4m (&t)[4]) {
#pragma clang fp contract(off)
    f32x4m s = {0.f, 0.f, 0.f, 0.f};
    s = s + t[0];
    s = s + t[1];
    s = s + t[2];
    s = s + t[3];
    return s * 0.25f;
}
// Four channels of a pooled pixel as they are asked for: the four taps, or the pooled value where x is pooled already.
template <bool POOLED>
struct DownPiece {
    f32x4m t[POOLED ? 1 : 4];
    __device__ __forceinline__ void fetch(const BconvDownArgs &p, int pix, int c, int channels) {
        if constexpr (POOLED) {
            t[0] = *reinterpret_cast<const f32x4m *>(p.xf + (size_t)pix * channels + c);
        } else {
            const DownPixel at(p, pix);
            const float *src = p.xf + ((size_t)(at.n * p.H + 2 * at.oy) * p.W + 2 * at.ox) * channels + c;
            const size_t below = (size_t)p.W * channels;
            t[0] = *reinterpret_cast<const f32x4m *>(src), t[1] = *reinterpret_cast<const f32x4m *>(src + channels);
            t[2] = *reinterpret_cast<const f32x4m *>(src + below), t[3] = *reinterpret_cast<const f32x4m *>(src + below + channels);
        }
    }
    __device__ __forceinline__ f32x4m value() const {
        if constexpr (POOLED)
            return t[0];
        else
            return pool_taps(t);
    }
};
// bias, Affine of the branch; Affine of the counts; Add: every operation rounded by itself like the separate layers'
__device__ __forceinline__ float branch_value(float v, bool with_bias, float bias, bool with_affine, float sa, float sb) {
#pragma clang fp contract(off)
    if (with_bias) v = v + bias;
    if (with_affine) {
        v = sa * v;
        v = v + sb;
    }
    return v;
}
__device__ __forceinline__ float down_value(float cnt, float ea, float eb, float sc) {
#pragma clang fp contract(off)
    float r = ea * cnt;
    r = r + eb;
    return r + sc;
}

// ---------------------------------------------------------------- few pieces
// Bound by latency: a block is T pixels x 16 * NT channels.  Three waves ask for a kernel row's bits each, all eight for the
// block's floats and filters in whole lines, which meet in LDS; then the waves take 16 pixels and a part of the branch's depth each, and
// the partial sums meet in LDS too.  (Floats fetched by each lane for its own pixel and depths, without the staging: a load then
// touches 16 or 32 lines, and 256 input channels took 5.3 to 9 us instead of 4.0 to 5.8.)
// The branch's four parts are those of dab_ave_pool2_fconv1x1, and so is the order in each: 0, 4, 1, 5 of eight depths in one
// instruction, 2, 6, 3, 7 in the next (the hardware rounds behind every product, in the order of the depth slots).  LDS holds a
// part's 16 depths as the four lanes of a row want them: 0 2 8 10, 4 6 12 14, 1 3 9 11, 5 7 13 15.
template <int CW, int T, int NT>
__global__ __launch_bounds__(512) void bconv3x3_down_staged_kernel(const BconvDownArgs p) {
    constexpr int C = CW * 64, CH = 16 * NT, LD = CH + 4, AS = C + 4, THREADS = 512;
    constexpr int KB = 64 / T, ND = 2 * CW < KB ? 1 : 2 * CW / KB, NC = CH / T < 1 ? 1 : CH / T;  // counting: T pixels x T channels, NC of them
    constexpr bool kPair = 2 * CW < KB;
    constexpr int STEPS = kPair ? 2 : 3;
    constexpr int XP = T * (C / 4) / THREADS < 1 ? 1 : T * (C / 4) / THREADS, FP = CH * (C / 4) / THREADS < 1 ? 1 : CH * (C / 4) / THREADS;
    constexpr int PXG = T / 16, DG = 4;  // the branch: PXG groups of 16 pixels, DG parts of the depth
    __shared__ __attribute__((aligned(16))) float pooled[T][AS];
    __shared__ __attribute__((aligned(16))) float filt[CH][AS];
    __shared__ __attribute__((aligned(16))) float part[3 + DG][T * LD];
    const int tid = threadIdx.x, lane = tid & 63;
    const int r = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t tile = p.div_cols.div(blockIdx.x);
    const int ch0 = (int)(blockIdx.x - tile * p.cols) * CH;
    uint32_t act[STEPS][ND], wt[NC][STEPS][ND];
    const int lr = lane % T, kb = lane / T;
    if (r < 3) {
        const __amdgpu_buffer_rsrc_t rx = make_rsrc(p.x, p.x_bytes), rw = make_rsrc(p.w, p.w_bytes);
        int pix = (int)tile * T + lr;
        pix = pix < p.total ? pix : p.total - 1;
        const DownPixel at(p, pix);
        const int y0 = 2 * at.oy - 1, x0 = 2 * at.ox - 1;
        const int base = ((at.n * p.H + y0 + r) * p.W + x0) * (CW * 8);
        const bool row_ok = (unsigned)(y0 + r) < (unsigned)p.H;
        const int wbase = (ch0 + lr) * (CW * 72) + r * (CW * 24);
#pragma unroll
        for (int s = 0; s < STEPS; ++s) {
            const int kw = kPair ? s * 2 + (kb >> 1) : s;
            const int inner = kPair ? (kb & 1) * 4 : kb * (ND * 4);
            const bool ok = row_ok && (unsigned)(x0 + kw) < (unsigned)p.W && (!kPair || kw < 3);
            load_dwords<ND>(act[s], rx, ok ? base + kw * (CW * 8) + inner : kDownOutside);
#pragma unroll
            for (int n = 0; n < NC; ++n)
                load_dwords<ND>(wt[n][s], rw, (!kPair || kw < 3) ? wbase + n * T * (CW * 72) + kw * (CW * 8) + inner : kDownOutside);
        }
    }
    DownPiece<false> x[XP];
    f32x4m f[FP];
#pragma unroll
    for (int i = 0; i < XP; ++i) {
        const int piece = tid + THREADS * i, pix = (int)tile * T + piece / (C / 4);
        x[i].fetch(p, pix < p.total ? pix : p.total - 1, (piece % (C / 4)) * 4, C);
    }
#pragma unroll
    for (int i = 0; i < FP; ++i) {
        const int piece = tid + THREADS * i;
        if (piece < CH * (C / 4)) f[i] = *reinterpret_cast<const f32x4m *>(p.sw + (size_t)ch0 * C + piece * 4);
    }
    // the store pass's operands: thread t has four channels of a pixel
    constexpr int Q = T * CH / 4;
    const int opix = (int)tile * T + tid / (CH / 4), och = ch0 + (tid % (CH / 4)) * 4;
    const bool ok = tid < Q && opix < p.total;
    const f32x4m zero = {0.f, 0.f, 0.f, 0.f};
    f32x4m ea = zero, eb = zero, bias = zero, sa = zero, sb = zero;
    if (ok) {
        ea = *reinterpret_cast<const f32x4m *>(p.ea + och), eb = *reinterpret_cast<const f32x4m *>(p.eb + och);
        if (p.bias) bias = *reinterpret_cast<const f32x4m *>(p.bias + och);
        if (p.sa) sa = *reinterpret_cast<const f32x4m *>(p.sa + och), sb = *reinterpret_cast<const f32x4m *>(p.sb + och);
    }
    __builtin_amdgcn_sched_barrier(0);  // everything is asked for before anything is waited for
    if (r < 3) {
        typename Fp4Acc<T>::type acc[NC];
#pragma unroll
        for (int n = 0; n < NC; ++n)
#pragma unroll
            for (int v = 0; v < Fp4Acc<T>::regs; ++v) acc[n][v] = 0.f;
#pragma unroll
        for (int s = 0; s < STEPS; ++s)
#pragma unroll
            for (int d = 0; d < ND; ++d) {
                const i32x8 a = bitspm1(act[s][d]);
#pragma unroll
                for (int n = 0; n < NC; ++n) mfma_fp4<T>(acc[n], a, bitspm1(wt[n][s][d]));
            }
#pragma unroll
        for (int n = 0; n < NC; ++n)
#pragma unroll
            for (int v = 0; v < Fp4Acc<T>::regs; ++v) part[r][fp4_row<T>(kb, v) * LD + n * T + lr] = acc[n][v];
    }
    // depths 4 q .. 4 q + 3 of their 16: two places of two
    auto put = [](float *row, int q, f32x4m v) __attribute__((always_inline)) {
        typedef float f32x2m __attribute__((ext_vector_type(2)));
        float *to = row + (q & ~3) * 4 + (q & 1) * 4 + (q & 2);
        *reinterpret_cast<f32x2m *>(to) = f32x2m{v[0], v[2]};
        *reinterpret_cast<f32x2m *>(to + 8) = f32x2m{v[1], v[3]};
    };
#pragma unroll
    for (int i = 0; i < XP; ++i) {
        const int piece = tid + THREADS * i;
        if (piece < T * (C / 4)) put(pooled[piece / (C / 4)], piece % (C / 4), x[i].value());
    }
#pragma unroll
    for (int i = 0; i < FP; ++i) {
        const int piece = tid + THREADS * i;
        if (piece < CH * (C / 4)) put(filt[piece / (C / 4)], piece % (C / 4), f[i]);
    }
    __syncthreads();
    if (r < PXG * DG) {
        const int l16 = lane & 15, k4 = lane >> 4, px = r % PXG, dg = r / PXG;
        f32x4m acc[NT];
#pragma unroll
        for (int n = 0; n < NT; ++n) acc[n] = zero;
#pragma unroll
        for (int d = 0; d < C; d += 64) {
            const int k = d + dg * 16 + 4 * k4;
            const f32x4m a = *reinterpret_cast<const f32x4m *>(&pooled[px * 16 + l16][k]);
            f32x4m b[NT];
#pragma unroll
            for (int n = 0; n < NT; ++n) b[n] = *reinterpret_cast<const f32x4m *>(&filt[n * 16 + l16][k]);
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int n = 0; n < NT; ++n) acc[n] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[e], b[n][e], acc[n], 0, 0, 0);
        }
#pragma unroll
        for (int n = 0; n < NT; ++n)
#pragma unroll
            for (int v = 0; v < 4; ++v) part[3 + dg][(px * 16 + 4 * k4 + v) * LD + n * 16 + l16] = acc[n][v];
    }
    __syncthreads();
    if (tid >= Q) return;  // whole waves

    constexpr float kHalfDepth = 0.5f * (kPair ? 3 * 4 * 64 : 9 * C);
    const int o = (tid / (CH / 4)) * LD + (tid % (CH / 4)) * 4;
    f32x4m s[3 + DG], v, sc;
#pragma unroll
    for (int i = 0; i < 3 + DG; ++i) s[i] = *reinterpret_cast<f32x4m *>(&part[i][o]);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const float t = ((s[3][e] + s[4][e]) + s[5][e]) + s[6][e];
        sc[e] = branch_value(t, p.bias != nullptr, bias[e], p.sa != nullptr, sa[e], sb[e]);
        v[e] = down_value(kHalfDepth - 0.5f * (s[0][e] + s[1][e] + s[2][e]), ea[e], eb[e], sc[e]);
    }
    const size_t first = (size_t)opix * p.cout + och;
    if (ok) {
        *reinterpret_cast<f32x4m *>(p.out + first) = v;
        if (p.sc_out) *reinterpret_cast<f32x4m *>(p.sc_out + first) = sc;
    }
    if (p.bits) {
        constexpr int G = CH / 4 < 8 ? CH / 4 : 8;
        const int g = tid % G;
        uint32_t word = sign_nibble(make_float4(v[0], v[1], v[2], v[3])) << (4 * g);
        word = or_from_lane_above<1>(word);
        word = or_from_lane_above<2>(word);
        if constexpr (G == 8) word = or_from_lane_above<4>(word);
        if (ok && g == 0) {
            if constexpr (G == 8)
                p.bits[first >> 5] = word;
            else
                reinterpret_cast<uint16_t *>(p.bits)[first >> 4] = (uint16_t)word;
        }
    }
}

// ---------------------------------------------------------------- between
// A wave counts, the block pools its pixels into LDS, the wave multiplies on the fp32 matrix instruction -- 32 of 64 cycles per 64
// channels of depth, which is what bounds the kernel: 40 images of 28 x 28 x 128 to 256 take 12.0 us.  Two blocks share a CU, one
// multiplying while the other waits for its floats: with 256 input channels a thread's 32 taps take 128 registers, so half of them are
// asked for when the bits have been counted, into their registers.  14 x 14 x 256 to 512, us, all at once and one block a CU / so: 40
// images 11.1 / 10.4, 60 20.1 / 17.0, 100 29.6 / 23.6, 256 70.5 / 53.4; a block of eight waves, the floats read half as often, 65.5 there, and
// three blocks a CU, with spills, 72.5.
// SPLIT: four sums of a quarter of the depth each, one behind the other, as dab_ave_pool2_fconv1x1 has them for problems this small.
template <int CW, int WAVES, bool POOLED, bool SPLIT>
__global__ __launch_bounds__(WAVES * 64, 2) void bconv3x3_down_tile_kernel(const BconvDownArgs p) {
    constexpr int C = CW * 64, AS = C + 4, CH = 32 * WAVES, THREADS = 64 * WAVES;  // AS: rows 4 floats off a multiple of 64 banks
    constexpr int PIECES = 32 * (C / 4) / THREADS;  // 16-byte pieces of the pooled tile per thread
    constexpr int EARLY = !POOLED && PIECES > 4 ? PIECES / 2 : PIECES;  // of those: asked for before anything is counted
    constexpr int CHUNK = 8, CHUNKS = C / 8 / CHUNK;  // a wave's filters in steps of 8 depths, asked for CHUNK steps at a time
    __shared__ __attribute__((aligned(16))) float pooled[32][AS];
    const int tid = threadIdx.x, lane = tid & 63, half = lane >> 5, l32 = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t item = xcd_contiguous_block(blockIdx.x, gridDim.x);  // a pixel tile's channel blocks share an XCD's L2
    const uint32_t tile = p.div_cols.div(item);
    const int ch0 = (int)(item - tile * p.cols) * CH + wave * 32, ch = ch0 + l32;
    const int m0 = (int)tile * 32;
    const bool ch_ok = ch0 < p.cout;  // (32 channels are all there or none)
    const __amdgpu_buffer_rsrc_t rx = make_rsrc(p.x, p.x_bytes), rw = make_rsrc(p.w, p.w_bytes);

    // the bits first: loads come back in order, and counting covers the wait for the floats
    uint32_t act[9][CW], wt[9][CW];
    {
        const int pix = m0 + l32 < p.total ? m0 + l32 : p.total - 1;
        const DownPixel at(p, pix);
        const int y0 = 2 * at.oy - 1, x0 = 2 * at.ox - 1, base = ((at.n * p.H + y0) * p.W + x0) * (CW * 8) + half * (CW * 4);
#pragma unroll
        for (int t = 0; t < 9; ++t) {
            const bool ok = (unsigned)(y0 + t / 3) < (unsigned)p.H && (unsigned)(x0 + t % 3) < (unsigned)p.W;
            load_dwords<CW>(act[t], rx, ok ? base + ((t / 3) * p.W + t % 3) * (CW * 8) : kDownOutside);
        }
#pragma unroll
        for (int t = 0; t < 9; ++t) load_dwords<CW>(wt[t], rw, ch_ok ? ch * (CW * 72) + t * (CW * 8) + half * (CW * 4) : kDownOutside);
    }
    DownPiece<POOLED> x[PIECES];
    auto fetch_floats = [&](int from, int to) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < PIECES; ++i) {
            if (i < from || i >= to) continue;
            const int piece = tid + THREADS * i, pix = m0 + piece / (C / 4);
            x[i].fetch(p, pix < p.total ? pix : p.total - 1, (piece % (C / 4)) * 4, C);
        }
    };
    fetch_floats(0, EARLY);
    const float *filter = p.sw + (size_t)(ch_ok ? ch : 0) * C + half * 4;
    f32x4m f[CHUNKS > 1 ? 2 : 1][CHUNK];
    // the first depth of step i, of C / 8: in order, or all 16-deep pieces of a part and then the next part's
    constexpr int PART = C / 32;  // steps
    auto depth_of = [](int i) { return SPLIT ? (i % PART) / 2 * 64 + i / PART * 16 + i % 2 * 8 : i * 8; };
    auto fetch_filters = [&](int chunk) {
#pragma unroll
        for (int s = 0; s < CHUNK; ++s) f[chunk & 1][s] = *reinterpret_cast<const f32x4m *>(filter + depth_of(chunk * CHUNK + s));
    };
    fetch_filters(0);
    float ea = 0.f, eb = 0.f, bias = 0.f, sa = 0.f, sb = 0.f;
    if (ch_ok) {
        ea = p.ea[ch], eb = p.eb[ch];
        if (p.bias) bias = p.bias[ch];
        if (p.sa) sa = p.sa[ch], sb = p.sb[ch];
    }

    f32x16m cnt, sum, parts;
#pragma unroll
    for (int v = 0; v < 16; ++v) cnt[v] = 0.f, sum[v] = 0.f, parts[v] = 0.f;
#pragma unroll
    for (int t = 0; t < 9; ++t)
#pragma unroll
        for (int c = 0; c < CW; ++c) mfma_fp4<32>(cnt, bitspm1(act[t][c]), bitspm1(wt[t][c]));
    if constexpr (EARLY < PIECES) {
        __builtin_amdgcn_sched_barrier(0);
        fetch_floats(EARLY, PIECES);  // into the registers of the bits
        __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int i = 0; i < PIECES; ++i) {
        const int piece = tid + THREADS * i;
        *reinterpret_cast<f32x4m *>(&pooled[piece / (C / 4)][(piece % (C / 4)) * 4]) = x[i].value();
    }
    __syncthreads();
    // eight depths at a time, the pairs d and d + 4 in one instruction
#pragma unroll
    for (int chunk = 0; chunk < CHUNKS; ++chunk) {
        if (chunk + 1 < CHUNKS) fetch_filters(chunk + 1);
#pragma unroll
        for (int s = 0; s < CHUNK; ++s) {
            const int step = chunk * CHUNK + s;
            if (SPLIT && step > 0 && step % PART == 0) {
#pragma unroll
                for (int v = 0; v < 16; ++v) parts[v] = step == PART ? sum[v] : parts[v] + sum[v], sum[v] = 0.f;
            }
            const f32x4m a = *reinterpret_cast<const f32x4m *>(&pooled[l32][depth_of(step) + half * 4]);
#pragma unroll
            for (int e = 0; e < 4; ++e) sum = __builtin_amdgcn_mfma_f32_32x32x2f32(a[e], f[chunk & 1][s][e], sum, 0, 0, 0);
        }
    }
    if constexpr (SPLIT) {
#pragma unroll
        for (int v = 0; v < 16; ++v) sum[v] = parts[v] + sum[v];
    }

    constexpr float kHalfDepth = 0.5f * 9 * C;
    const size_t base = (size_t)m0 * p.cout;
    const int rows = p.total - m0 < 32 ? p.total - m0 : 32;
    const __amdgpu_buffer_rsrc_t ro = make_rsrc(p.out + base, (uint32_t)rows * p.cout * 4u);
    const __amdgpu_buffer_rsrc_t rs = make_rsrc(p.sc_out + (p.sc_out ? base : 0), p.sc_out ? (uint32_t)rows * p.cout * 4u : 0u);
    const int lane_off = ch_ok ? (half * 4 * p.cout + ch) * 4 : kDownOutside;
    uint32_t word = 0;
#pragma unroll
    for (int v = 0; v < 16; ++v) {
        const int row = 8 * (v / 4) + v % 4;
        const float sc = branch_value(sum[v], p.bias != nullptr, bias, p.sa != nullptr, sa, sb);
        const float r = down_value(kHalfDepth - 0.5f * cnt[v], ea, eb, sc);
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, r), ro, lane_off + row * p.cout * 4, 0, kStoreStream);
        if (p.sc_out) __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, sc), rs, lane_off + row * p.cout * 4, 0, 0);
        const uint64_t mask = __ballot(r > 0.f);
        word = dab_writelane((uint32_t)mask, row, word);
        word = dab_writelane((uint32_t)(mask >> 32), row + 4, word);
    }
    if (p.bits && half == 0 && m0 + l32 < p.total && ch_ok) p.bits[(size_t)(m0 + l32) * (p.cout / 32) + ch0 / 32] = word;
}

// ---------------------------------------------------------------- many pieces: blocks that walk over pixel tiles
// A wave keeps the filters of 32 channels for its lifetime, and a block walks over tiles of 32 pixels: it pools a tile into LDS while
// the next one's floats and bits are on their way.  Bound by its instructions, of which vector and matrix ones do not overlap here: 256
// images of 56 x 56 x 64 to 128 take 61 us (two launches 96, the tile kernel 66), 51 from the pooled tensor (tile kernel 57) -- of 125 000
// cycles, the fp32 matrix instructions of a SIMD have 50 000, counting 7 000, the vector instructions 31 000 and more.  With 128 input channels a
// block has eight waves, so that the floats are read once: 28 x 28 at 256 images 55 us (two launches 67, tile kernel 57).  (The same with the
// products on the bf16 matrix instruction, in three parts each: 60, 47 and 43 us, but not the separate launch's sums to the last bit.)
template <int CW, int WAVES, bool POOLED>
__global__ __launch_bounds__(WAVES * 64, CW == 1 ? 3 : 2) void bconv3x3_down_walk_kernel(const BconvDownArgs p) {
    constexpr int C = CW * 64, CH = 32 * WAVES, THREADS = 64 * WAVES;
    constexpr int PIECES = 32 * (C / 4) / THREADS, AS = C + 4;  // AS: rows 4 floats off a multiple of 64 banks
    __shared__ __attribute__((aligned(16))) float pooled[2][32][AS];
    const int tid = threadIdx.x, lane = tid & 63, half = lane >> 5, l32 = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int group = (int)p.div_cols.div(blockIdx.x), groups = (int)p.div_cols.div(gridDim.x);
    const int ch0 = ((int)blockIdx.x - group * p.cols) * CH + wave * 32, ch = ch0 + l32;
    const bool ch_ok = ch0 < p.cout;  // (32 channels are all there or none)
    const int tiles = (p.total + 31) / 32;
    const __amdgpu_buffer_rsrc_t rx = make_rsrc(p.x, p.x_bytes), rw = make_rsrc(p.w, p.w_bytes);

    DownPiece<POOLED> x[PIECES];
    uint32_t act[9][CW];
    auto fetch_floats = [&](int tile) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < PIECES; ++i) {
            const int piece = tid + THREADS * i, pix = tile * 32 + piece / (C / 4);
            x[i].fetch(p, pix < p.total ? pix : p.total - 1, (piece % (C / 4)) * 4, C);
        }
    };
    auto fetch_bits = [&](int tile) __attribute__((always_inline)) {
        const int pix = tile * 32 + l32 < p.total ? tile * 32 + l32 : p.total - 1;
        const DownPixel at(p, pix);
        const int y0 = 2 * at.oy - 1, x0 = 2 * at.ox - 1, base = ((at.n * p.H + y0) * p.W + x0) * (CW * 8) + half * (CW * 4);
#pragma unroll
        for (int t = 0; t < 9; ++t) {
            const bool ok = (unsigned)(y0 + t / 3) < (unsigned)p.H && (unsigned)(x0 + t % 3) < (unsigned)p.W;
            load_dwords<CW>(act[t], rx, ok ? base + ((t / 3) * p.W + t % 3) * (CW * 8) : kDownOutside);
        }
    };
    int tile = group;
    if (tile < tiles) fetch_bits(tile), fetch_floats(tile);

    uint32_t wt[9][CW];
#pragma unroll
    for (int t = 0; t < 9; ++t) load_dwords<CW>(wt[t], rw, ch_ok ? ch * (CW * 72) + t * (CW * 8) + half * (CW * 4) : kDownOutside);
    const float *filter = p.sw + (size_t)(ch_ok ? ch : 0) * C + half * 4;
    f32x4m f[C / 8];
#pragma unroll
    for (int i = 0; i < C / 8; ++i) f[i] = *reinterpret_cast<const f32x4m *>(filter + i * 8);
    uint32_t set = 0;
#pragma unroll
    for (int t = 0; t < 9; ++t)
#pragma unroll
        for (int c = 0; c < CW; ++c) set += __popc(wt[t][c]);
    set += __shfl_xor(set, 32);
    const float init = (float)set;
    float ea = 0.f, eb = 0.f, bias = 0.f, sa = 0.f, sb = 0.f;
    if (ch_ok) {
        ea = p.ea[ch], eb = p.eb[ch];
        if (p.bias) bias = p.bias[ch];
        if (p.sa) sa = p.sa[ch], sb = p.sb[ch];
    }

    // here, and not at their first use inside the loop: there the wait would be for the next tile's floats as well
#pragma unroll
    for (int i = 0; i < C / 8; ++i) asm volatile("" : "+v"(f[i]));
    asm volatile("" : "+v"(ea), "+v"(eb), "+v"(bias), "+v"(sa), "+v"(sb));

    for (int buf = 0; tile < tiles; tile += groups, buf ^= 1) {
#pragma unroll
        for (int i = 0; i < PIECES; ++i) {
            const int piece = tid + THREADS * i;
            *reinterpret_cast<f32x4m *>(&pooled[buf][piece / (C / 4)][(piece % (C / 4)) * 4]) = x[i].value();
        }
        const bool more = tile + groups < tiles;
        if (more) fetch_floats(tile + groups);
        __syncthreads();
        f32x16m sum;
#pragma unroll
        for (int v = 0; v < 16; ++v) sum[v] = 0.f;
#pragma unroll
        for (int i = 0; i < C / 8; ++i) {
            const f32x4m a = *reinterpret_cast<const f32x4m *>(&pooled[buf][l32][i * 8 + half * 4]);
#pragma unroll
            for (int e = 0; e < 4; ++e) sum = __builtin_amdgcn_mfma_f32_32x32x2f32(a[e], f[i][e], sum, 0, 0, 0);
        }
        f32x16m cnt;
#pragma unroll
        for (int v = 0; v < 16; ++v) cnt[v] = init;
#pragma unroll
        for (int t = 0; t < 9; ++t)
#pragma unroll
            for (int c = 0; c < CW; ++c) {
                asm volatile("" : "+v"(wt[t][c]));  // expanded here: hoisted out of the loop the expanded filters would not fit
                mfma_fp4<32>(cnt, bits01(act[t][c]), bitspm(wt[t][c]));
            }
        if (more) fetch_bits(tile + groups);

        const size_t base = (size_t)tile * 32 * p.cout;
        const int rows = p.total - tile * 32 < 32 ? p.total - tile * 32 : 32;
        const __amdgpu_buffer_rsrc_t ro = make_rsrc(p.out + base, (uint32_t)rows * p.cout * 4u);
        const __amdgpu_buffer_rsrc_t rs = make_rsrc(p.sc_out + (p.sc_out ? base : 0), p.sc_out ? (uint32_t)rows * p.cout * 4u : 0u);
        const int lane_off = ch_ok ? (half * 4 * p.cout + ch) * 4 : kDownOutside;
        uint32_t word = 0;
        auto finish = [&](auto usual) __attribute__((always_inline)) {  // a converter's block: an Affine and no bias, the branch's blob not wanted
            constexpr bool U = decltype(usual)::value;
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const int row = 8 * (v / 4) + v % 4;
                const float sc = U ? branch_value(sum[v], false, 0.f, true, sa, sb) : branch_value(sum[v], p.bias != nullptr, bias, p.sa != nullptr, sa, sb);
                const float r = down_value(cnt[v], ea, eb, sc);
                __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, r), ro, lane_off, row * p.cout * 4, kStoreStream);
                if (!U && p.sc_out) __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, sc), rs, lane_off, row * p.cout * 4, 0);
                const uint64_t mask = __ballot(r > 0.f);
                word = dab_writelane((uint32_t)mask, row, word);
                word = dab_writelane((uint32_t)(mask >> 32), row + 4, word);
            }
        };
        if (p.sa && !p.bias && !p.sc_out)
            finish(std::true_type{});
        else
            finish(std::false_type{});
        if (p.bits && half == 0 && l32 < rows && ch_ok) p.bits[((size_t)tile * 32 + l32) * (p.cout / 32) + ch0 / 32] = word;
    }
}

static bool down_geometry(BconvDownArgs &a, int n, int h, int w, int cin, int cout) {
    if (!(cin == 64 || cin == 128 || cin == 256) || cout % 64 != 0 || h % 2 != 0 || w % 2 != 0) return false;
    const long long in_pixels = (long long)n * h * w, total = in_pixels / 4;
    if (in_pixels >= (1ll << 31) - 64 || in_pixels * (cin / 8) >= (1ll << 31) || (long long)cout * cin * 9 / 8 >= (1ll << 31) || cout >= (1 << 20) ||
        total * cout >= (1ll << 40))
        return false;
    a.H = h, a.W = w, a.OH = h / 2, a.OW = w / 2, a.cout = cout, a.total = (int)total;
    a.x_bytes = (uint32_t)(in_pixels * (cin / 8)), a.w_bytes = (uint32_t)((long long)cout * 9 * cin / 8);
    a.div_ow = FastDiv((uint32_t)a.OW), a.div_oh = FastDiv((uint32_t)a.OH);
    return true;
}

enum class Down { staged16, staged32, tile_split, tile, walk };
// The branch's sums are dab_ave_pool2_fconv1x1's to the bit, so it follows from that call's rule whether the depth is split: for problems
// of up to about 768 pieces of 32 pixels x 32 channels (512 with 64 output channels).  us:
//   16 x 16 tiles up to 128 pieces of 128 and 256 input channels: 28 x 28 x 128 at batch 1 (56 pieces) 3.5 against 4.2, at batch 4
//   (200) 6.1 against 4.5; 14 x 14 x 256 at batch 2 (64) 4.0 against 5.6, at batch 6 (160) 6.8 against 5.7
//   32 x 32 tiles up to 700 pieces (64 input channels) and 512: 56 x 56 x 64 at batch 6 (588) 5.6 against the tile kernel's 6.4; 28 x 28 x
//   128 at batch 9 (448) 6.0 against 7.5; 14 x 14 x 256 at batch 16 (400) 9.7 against 10.8
// and in one sum, for which a block needs whole depths:
//   walking from 780 tiles of 32 pixels: 56 x 56 x 64 to 128 at batch 30 (735) 11.7 against the tile kernel's 11.4, at 40 14.1 / 14.5, at
//   100 28.9 / 29.8; 28 x 28 x 128 to 256 at batch 100 (613) 26.7 / 25.1, at 150 (919) 35.4 / 37.3; 64 to 256 channels at 735 20.6 / 18.4
static Down pick_down(long long total, int cin, int cout) {
    const long long tiles = (total + 31) / 32, pieces = tiles * (cout / 32);
    if (!pool2_fconv1x1_splits_depth(total, cout)) return cin <= 128 && tiles >= 780 ? Down::walk : Down::tile;
    if (cin >= 128 && pieces <= 128) return Down::staged16;
    return pieces <= (cin == 64 ? 700 : 512) ? Down::staged32 : Down::tile_split;
}

template <class Kernel>
static int launch_down(Kernel kernel, BconvDownArgs &a, int px, int ch, int threads, hipStream_t s) {
    a.cols = (a.cout + ch - 1) / ch;
    a.div_cols = FastDiv((uint32_t)a.cols);
    const long long blocks = ((long long)a.total + px - 1) / px * a.cols;
    if (blocks >= kMostBlocks) return fail(DAB_EUNSUPPORTED, "dab_bconv3x3_down: too many work units");
    hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(threads), 0, s, a);
    DAB_LAUNCH_CHECK();
    return DAB_OK;
}

template <int CW, int WAVES, bool POOLED>
static int launch_down_walk(BconvDownArgs &a, hipStream_t s) {
    constexpr int CH = 32 * WAVES;
    auto kernel = bconv3x3_down_walk_kernel<CW, WAVES, POOLED>;
    a.cols = (a.cout + CH - 1) / CH;
    a.div_cols = FastDiv((uint32_t)a.cols);
    static const int per_cu = [&] {
        int blocks = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&blocks, kernel, WAVES * 64, 0) != hipSuccess || blocks < 1) blocks = 1;
        return blocks;
    }();
    const int tiles = (int)(((long long)a.total + 31) / 32), most = simd_count() / 4 * per_cu / a.cols;
    const int groups = tiles < most ? tiles : most < 1 ? 1 : most;  // (equal shares on fewer blocks: 64 images 25.7 us instead of 22.3, 256 64 instead of 61)
    hipLaunchKernelGGL(kernel, dim3((unsigned)(groups * a.cols)), dim3(WAVES * 64), 0, s, a);
    DAB_LAUNCH_CHECK();
    return DAB_OK;
}

template <int CW, bool POOLED>
static int launch_bconv_down(BconvDownArgs &a, hipStream_t s) {
    const Down kernel = pick_down(a.total, CW * 64, a.cout);
    if constexpr (CW >= 2 && !POOLED)
        if (kernel == Down::staged16) return launch_down(bconv3x3_down_staged_kernel<CW, 16, 1>, a, 16, 16, 512, s);
    if constexpr (!POOLED)
        if (kernel == Down::staged32) return launch_down(bconv3x3_down_staged_kernel<CW, 32, 2>, a, 32, 32, 512, s);
    if constexpr (CW <= 2)
        if (kernel == Down::walk) return launch_down_walk<CW, 4 * CW, POOLED>(a, s);
    if (kernel != Down::tile) return launch_down(bconv3x3_down_tile_kernel<CW, 4, POOLED, true>, a, 32, 128, 256, s);
    return launch_down(bconv3x3_down_tile_kernel<CW, 4, POOLED, false>, a, 32, 128, 256, s);
}

}  // namespace dab

extern "C" int dab_bconv3x3_down_takes(int n, int h, int w, int cin, int cout) {
    dab::BconvDownArgs a;
    return n > 0 && h > 0 && w > 0 && cout > 0 && dab::down_geometry(a, n, h, w, cin, cout) &&
           ((long long)a.total + 31) / 32 * ((cout + 127) / 128) < dab::kMostBlocks;
}

extern "C" int dab_bconv3x3_down(const uint64_t *x_packed, const float *x, int x_pooled, int n, int h, int w, int cin, const uint64_t *wgt,
                                 const float *a, const float *b, int cout, const float *sc_wgt, const float *sc_bias, const float *sc_a, const float *sc_b,
                                 float *shortcut, float *out, uint64_t *out_packed, dab_stream_t stream) {
    using namespace dab;
    const char *fn = "dab_bconv3x3_down";
    DAB_REQUIRE(x_packed && x && wgt && a && b && sc_wgt && out, "%s: null pointer", fn);
    DAB_REQUIRE(n > 0 && h > 0 && w > 0 && cin > 0 && cout > 0, "%s: non-positive dimension", fn);
    DAB_REQUIRE((sc_a == nullptr) == (sc_b == nullptr), "%s: affine needs both coefficient vectors", fn);
    DAB_REQUIRE(out != x && shortcut != x && out != shortcut && out_packed != x_packed, "%s: the results must not alias the input or each other", fn);
    auto at = [](const void *q) { return reinterpret_cast<uintptr_t>(q); };
    DAB_REQUIRE(((at(x_packed) | at(x) | at(a) | at(b) | at(sc_wgt) | at(sc_bias) | at(sc_a) | at(sc_b) | at(shortcut) | at(out)) & 15) == 0 &&
                    ((at(wgt) | at(out_packed)) & 7) == 0,
                "%s: buffers must be 16-byte aligned", fn);
    BconvDownArgs p;
    if (!dab_bconv3x3_down_takes(n, h, w, cin, cout) || !down_geometry(p, n, h, w, cin, cout))
        return fail(DAB_EUNSUPPORTED, "%s: %d images of %d x %d x %d to %d channels are not covered", fn, n, h, w, cin, cout);
    p.x = x_packed, p.xf = x, p.w = wgt, p.ea = a, p.eb = b, p.sw = sc_wgt, p.bias = sc_bias, p.sa = sc_a, p.sb = sc_b;
    p.sc_out = shortcut, p.out = out, p.bits = reinterpret_cast<uint32_t *>(out_packed);
    hipStream_t s = as_stream(stream);
    switch (cin) {
        case 64: return x_pooled ? launch_bconv_down<1, true>(p, s) : launch_bconv_down<1, false>(p, s);
        case 128: return x_pooled ? launch_bconv_down<2, true>(p, s) : launch_bconv_down<2, false>(p, s);
        default: return x_pooled ? launch_bconv_down<4, true>(p, s) : launch_bconv_down<4, false>(p, s);
    }
}
