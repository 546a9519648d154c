// Direct 3x3 binary convolution for 64/128/256/512 (raw counts also 1024) input channels.
//
// Replaces the reference's pack -> pad -> bconv_3x3 chain
// (dabnn/layers/BinConv.cpp:145-150, dabnn/bconv.h:855-931) on packed input;
// results equal baseline_bconv (common/baseline.h:77-116) bit for bit.
//
// Data layout: x [N][H][W][CW] uint64 (CW = cin/64), weights in the reference's
// own order [cout][3][3][CW] (no repacking), out [N][OH][OW][cout] fp32.
//
// An implicit GEMM on the matrix cores (fp4_core.h): rows = output pixels, columns = output channels, depth = the 9 * cin
// bits of a window.  A lane fetches the bits of its pixel or filter and expands them in registers; out-of-image taps are
// fetched through a buffer descriptor with an out-of-range offset, which the hardware answers with zero -- the zero word
// that stands for 64 values of -1 (dabnn/pad.h:12).
//
// Three kernels, chosen by the number of 32-pixel x 32-channel pieces of the output (launch_bconv3x3):
//   split   few pieces: a block is one tile, its three waves take one kernel row each, the partial sums meet in LDS
//   stream  many pieces, 64 input channels: waves walk over pixel tiles, the filters of 64 channels stay in LDS
//   window  many pieces, 128 to 512 input channels: a wave keeps the filters of 32 channels in registers, the block's
//           four waves share the packed pixels of a tile in LDS
#include "fp4_core.h"

namespace dab {

struct BconvArgs {
    const uint64_t *x;
    const uint64_t *w;
    float *out;
    int total;  // N*OH*OW output pixels
    int H, W, OH, OW;
    int cout;
    int stride, pad;
    int cols;         // channel tiles
    int px_tiles;     // pixel tiles
    int window;       // window kernel: pixels of input that a tile's windows reach at most
    int buffers;      // and how many such windows fit LDS, one or two
    uint32_t x_bytes, w_bytes;
    FastDiv div_ow, div_oh, div_cols;
    // fused epilogue (MODE >= 1 kernels only): out = a*cnt + b (+ shortcut); MODE 2 also writes sign bits of out
    const float *epi_a;
    const float *epi_b;
    const float *epi_shortcut;
    uint32_t *epi_bits;
};

// MODE 0: raw counts.  1: + Affine (+ Add).  2: the same and a sign-packed copy of the result.
constexpr int kModeCounts = 0, kModeAffineAdd = 1, kModeAffineAddSign = 2;

constexpr int kOutside = (int)0x80000000;  // an offset beyond any descriptor: loads return zero, stores are dropped

// Top-left input position of an output pixel and its linear input pixel index (either may be outside the image).
__device__ __forceinline__ int window_origin(const BconvArgs &p, int pix, int &y0, int &x0) {
    const uint32_t t = p.div_ow.div(pix);
    const int ox = pix - t * p.OW;
    const uint32_t n = p.div_oh.div(t);
    const int oy = t - n * p.OH;
    y0 = oy * p.stride - p.pad, x0 = ox * p.stride - p.pad;
    return (int)(n * p.H + y0) * p.W + x0;
}

// a*cnt + b (+ shortcut), every operation rounded by itself like the reference's Affine and Add layers
__device__ __forceinline__ float affine_add(float cnt, float a, float b, float shortcut, bool with_shortcut) {
#pragma clang fp contract(off)
    float r = a * cnt;
    r = r + b;
    if (with_shortcut) r = r + shortcut;
    return r;
}

// ---------------------------------------------------------------- few pieces: the depth split over a block's waves
// Bound by latency: a launch is two dependent round trips to memory (arguments, operands) and the drain.  So a block is
// one T-pixel x (T * NT)-channel tile and wave r takes kernel row r of it: everything a wave needs -- three taps of its
// pixels and of its filters -- is asked for at once in wide loads (16 bytes a lane from 256 input channels up), then
// come 12 * NT (512 channels, T = 16) matrix instructions, one exchange through LDS and the store.  Both operands are
// +-1 here, so that no lane has to count the bits of its filters.  One image of the seven ResNet-18 stage shapes:
// 16.2 us together, 18.9 with epilogue and sign bits; the popcount kernels this replaced took 22.6 and 27.4.
template <int CW, int MODE, int T, int NT>
__global__ __launch_bounds__(192) void bconv3x3_split_kernel(const BconvArgs p) {
    constexpr int KB = 64 / T;               // lanes of a wave that share a row or column: 32 depths each
    constexpr bool kPair = 2 * CW < KB;      // 64 channels, T = 16: an instruction's depths are two taps
    constexpr int ND = kPair ? 1 : 2 * CW / KB;  // dwords per lane and step
    constexpr int STEPS = kPair ? 2 : 3;
    constexpr int CH = T * NT, LD = CH + 4;  // LD: 16-byte rows whose starts spread over the banks
    constexpr bool kThrough = T == 32;       // written through the L2 from a few hundred tiles up: 3 to 20 % a launch
    __shared__ __attribute__((aligned(16))) float part[3][T * LD];
    const int tid = threadIdx.x, lane = tid & 63, lr = lane % T, kb = lane / T;
    const int r = __builtin_amdgcn_readfirstlane(tid >> 6);  // this wave's kernel row
    const uint32_t tile = p.div_cols.div(blockIdx.x);
    const int ch0 = (int)(blockIdx.x - tile * p.cols) * CH;
    const __amdgpu_buffer_rsrc_t rx = make_rsrc(p.x, p.x_bytes), rw = make_rsrc(p.w, p.w_bytes);

    int pix = (int)tile * T + lr;
    pix = pix < p.total ? pix : p.total - 1;
    int y0, x0;
    const int base = (window_origin(p, pix, y0, x0) + r * p.W) * (CW * 8);
    const bool row_ok = (unsigned)(y0 + r) < (unsigned)p.H;
    const int wbase = (ch0 + lr) * (CW * 72) + r * (CW * 24);  // channels past cout lie past the descriptor
    uint32_t act[STEPS][ND], wt[NT][STEPS][ND];
#pragma unroll
    for (int s = 0; s < STEPS; ++s) {
        const int kw = kPair ? s * 2 + (kb >> 1) : s;
        const int inner = kPair ? (kb & 1) * 4 : kb * (ND * 4);
        const bool ok = row_ok && (unsigned)(x0 + kw) < (unsigned)p.W && (!kPair || kw < 3);
        load_dwords<ND>(act[s], rx, ok ? base + kw * (CW * 8) + inner : kOutside);
#pragma unroll
        for (int n = 0; n < NT; ++n)
            load_dwords<ND>(wt[n][s], rw, (!kPair || kw < 3) ? wbase + n * T * (CW * 72) + kw * (CW * 8) + inner : kOutside);
    }

    // The store pass's operands, asked for before the counting: thread t has float4 number t (+ 192) of the tile.
    constexpr int Q = T * CH / 4, QI = (Q + 191) / 192;
    f32x4m sc[QI], ea[QI], eb[QI];
    int opix[QI], och[QI];
    bool ok[QI];
#pragma unroll
    for (int i = 0; i < QI; ++i) {
        const int q = tid + i * 192;
        opix[i] = (int)tile * T + q / (CH / 4), och[i] = ch0 + (q % (CH / 4)) * 4;
        ok[i] = q < Q && opix[i] < p.total && och[i] < p.cout;
        if constexpr (MODE != kModeCounts) {
            const f32x4m zero = {0.f, 0.f, 0.f, 0.f};
            ea[i] = ok[i] ? *reinterpret_cast<const f32x4m *>(p.epi_a + och[i]) : zero;
            eb[i] = ok[i] ? *reinterpret_cast<const f32x4m *>(p.epi_b + och[i]) : zero;
            sc[i] = ok[i] && p.epi_shortcut ? *reinterpret_cast<const f32x4m *>(p.epi_shortcut + (size_t)opix[i] * p.cout + och[i]) : zero;
        }
    }

    typename Fp4Acc<T>::type acc[NT];
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int v = 0; v < Fp4Acc<T>::regs; ++v) acc[n][v] = 0.f;
#pragma unroll
    for (int s = 0; s < STEPS; ++s)
#pragma unroll
        for (int d = 0; d < ND; ++d) {
            const i32x8 a = bitspm1(act[s][d]);
#pragma unroll
            for (int n = 0; n < NT; ++n) mfma_fp4<T>(acc[n], a, bitspm1(wt[n][s][d]));
        }
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int v = 0; v < Fp4Acc<T>::regs; ++v) part[r][fp4_row<T>(kb, v) * LD + n * T + lr] = acc[n][v];
    __syncthreads();

    // depths of the three waves together (the fourth, empty tap slot of a pair counts as equal bits)
    constexpr float kHalfDepth = 0.5f * (kPair ? 3 * 4 * 64 : 9 * CW * 64);
#pragma unroll
    for (int i = 0; i < QI; ++i) {
        const int q = tid + i * 192;
        if (Q % 192 != 0 && q >= Q) break;  // whole waves
        const int o = (q / (CH / 4)) * LD + (q % (CH / 4)) * 4;
        const f32x4m s0 = *reinterpret_cast<f32x4m *>(&part[0][o]), s1 = *reinterpret_cast<f32x4m *>(&part[1][o]),
                     s2 = *reinterpret_cast<f32x4m *>(&part[2][o]);
        f32x4m v;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            v[e] = kHalfDepth - 0.5f * (s0[e] + s1[e] + s2[e]);
            if constexpr (MODE != kModeCounts) v[e] = affine_add(v[e], ea[i][e], eb[i][e], sc[i][e], p.epi_shortcut != nullptr);
        }
        if (ok[i]) {
            f32x4m *dst = reinterpret_cast<f32x4m *>(p.out + (size_t)opix[i] * p.cout + och[i]);
            if constexpr (kThrough)
                store_through(dst, v);
            else
                *dst = v;
        }
        if constexpr (MODE == kModeAffineAddSign) {
            // the CH / 4 lanes of a pixel lie in one row of 16 lanes; eight of them (four with a 16-channel tile) make a store
            constexpr int G = CH / 4 < 8 ? CH / 4 : 8;
            const int g = q % G;
            uint32_t word = sign_nibble(make_float4(v[0], v[1], v[2], v[3])) << (4 * g);
            word = or_from_lane_above<1>(word);
            word = or_from_lane_above<2>(word);
            if constexpr (G == 8) word = or_from_lane_above<4>(word);
            const size_t bit = (size_t)opix[i] * p.cout + och[i];
            if (ok[i] && g == 0) {
                if constexpr (G == 8)
                    p.epi_bits[bit >> 5] = word;
                else
                    reinterpret_cast<uint16_t *>(p.epi_bits)[bit >> 4] = (uint16_t)word;
            }
        }
    }
}

// ---------------------------------------------------------------- the output of a wave's tile, straight from the accumulators
// Accumulator registers hold 32 pixels x 32 channels with the channels along the lanes: every register is 128
// contiguous bytes of two pixels, so results leave (and shortcut values arrive) as whole lines without a pass through
// LDS, a lane needs one pair of Affine coefficients, and the sign bits of a register are the lane mask of one compare.
// A tile's descriptor starts at its first pixel and ends with the tensor: rows of a last, ragged tile are dropped.
struct TileView {
    size_t base;       // first element
    uint32_t bytes;    // from there to the end of the tensor, as far as a tile can reach
    __device__ __forceinline__ TileView(const BconvArgs &p, int first_pixel) {
        base = (size_t)first_pixel * p.cout;
        const size_t left = ((size_t)(p.total - first_pixel)) * p.cout * 4;
        bytes = left < 0x7fffffffu ? (uint32_t)left : 0x7fffffffu;
    }
};
// Byte offset of accumulator register v of 32-pixel group m within a tile; the lane's part is its channel and row.
__device__ __forceinline__ int tile_row_offset(const BconvArgs &p, int m, int v) { return (m * 32 + 8 * (v / 4) + v % 4) * p.cout * 4; }

__device__ __forceinline__ void fetch_shortcut(float (&sc)[16], __amdgpu_buffer_rsrc_t rs, const BconvArgs &p, int m, int lane_off) {
#pragma unroll
    for (int v = 0; v < 16; ++v)
        sc[v] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, lane_off, tile_row_offset(p, m, v), 0));
}
// Applies the epilogue to register v, stores it and puts its sign bits into lanes row and row + 4 of `word`.
template <int MODE>
__device__ __forceinline__ void finish_register(float cnt, __amdgpu_buffer_rsrc_t ro, const BconvArgs &p, int m, int v, int lane_off, float a,
                                                float b, float sc, uint32_t &word) {
    float r = cnt;
    if constexpr (MODE != kModeCounts) r = affine_add(cnt, a, b, sc, p.epi_shortcut != nullptr);
    // Counts are written through the L2; results of an epilogue stream past it (56x56x64 at batch 256 with shortcut and
    // sign bits: 67 us against 82 written through; 56x56x64 counts there: 33 us written through, 40 streamed).
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, r), ro, lane_off, tile_row_offset(p, m, v),
                                          MODE == kModeCounts ? kStoreThrough : kStoreStream);
    if constexpr (MODE == kModeAffineAddSign) {
        const uint64_t mask = __ballot(r > 0.f);
        const int row = 8 * (v / 4) + v % 4;
        word = dab_writelane((uint32_t)mask, row, word);
        word = dab_writelane((uint32_t)(mask >> 32), row + 4, word);
    }
}

// ---------------------------------------------------------------- 64 input channels, many pieces
// Bound by memory (56 x 56 x 64 -> 64 at batch 256 reads a 205 MB shortcut and writes 205 MB).  A block stages the
// filters of 32 * NT channels once (2.4 KB a 32, as bits), then its waves walk over tiles of 32 * MT pixels, all blocks
// on neighbouring tiles at the same time.  A wave asks for its tile's nine taps and shortcut values before it counts.
// Batch 256, counts / with Affine + Add + sign bits: 31 / 67 us (52 and 83 with the popcount kernels before).
template <int MODE, int MT, int NT>
__global__ __launch_bounds__(256, MT == 2 ? 2 : NT == 2 ? 3 : 4) void bconv3x3_stream_kernel(const BconvArgs p) {
    constexpr int kRow = 72, CH = 32 * NT, PX = 32 * MT;  // bytes per filter: 18 dwords, so 32 rows hit 32 even banks
    __shared__ __attribute__((aligned(16))) unsigned char filters[CH * kRow];
    __shared__ uint32_t pop[CH];  // set bits per filter
    const int tid = threadIdx.x, lane = tid & 63, half = lane >> 5, l32 = lane & 31;
    const int wib = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int group = (int)p.div_cols.div(blockIdx.x), groups = (int)p.div_cols.div(gridDim.x);
    const int ch0 = ((int)blockIdx.x - group * p.cols) * CH;
    const __amdgpu_buffer_rsrc_t rx = make_rsrc(p.x, p.x_bytes), rw = make_rsrc(p.w, p.w_bytes);
    if (tid < CH) pop[tid] = 0;
    __syncthreads();
    for (int c = tid; c < CH * 9; c += 256) {  // word c of the block's filters (zero past the last channel)
        const u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(rw, ch0 * kRow + c * 8, 0, 0);
        *reinterpret_cast<u32x2 *>(filters + c * 8) = v;
        atomicAdd(&pop[c / 9], __popc(v.x) + __popc(v.y));
    }
    __syncthreads();
    float init[NT], ea[NT], eb[NT];
    int lane_off[NT];
#pragma unroll
    for (int n = 0; n < NT; ++n) {
        init[n] = (float)pop[n * 32 + l32];
        const int ch = ch0 + n * 32 + l32;
        const bool ok = ch < p.cout;
        lane_off[n] = ok ? (half * 4 * p.cout + ch) * 4 : kOutside;
        ea[n] = 0.f, eb[n] = 0.f;
        if constexpr (MODE != kModeCounts)
            if (ok) ea[n] = p.epi_a[ch], eb[n] = p.epi_b[ch];
    }
    int wofs = l32 * kRow + half * 4;

    for (int tile = group * 4 + wib; tile < p.px_tiles; tile += groups * 4) {
        // With an epilogue the filters' expanded form would not fit the registers: the compiler may not move it out of
        // the loop.  (Raw counts keep it there: 36 registers per 32 channels.)
        if constexpr (MODE != kModeCounts) asm volatile("" : "+v"(wofs));
        uint32_t act[MT][9];
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            int pix = tile * PX + m * 32 + l32;
            pix = pix < p.total ? pix : p.total - 1;
            int y0, x0;
            const int base = window_origin(p, pix, y0, x0) * 8 + half * 4;
#pragma unroll
            for (int t = 0; t < 9; ++t) {
                const int kh = t / 3, kw = t % 3;
                const bool ok = (unsigned)(y0 + kh) < (unsigned)p.H && (unsigned)(x0 + kw) < (unsigned)p.W;
                act[m][t] = __builtin_amdgcn_raw_buffer_load_b32(rx, ok ? base + (kh * p.W + kw) * 8 : kOutside, 0, 0);
            }
        }
        const TileView view(p, tile * PX);
        float sc[MT][NT][16];
        if constexpr (MODE != kModeCounts) {
            if (p.epi_shortcut) {
                const __amdgpu_buffer_rsrc_t rs = make_rsrc(p.epi_shortcut + view.base, view.bytes);
#pragma unroll
                for (int m = 0; m < MT; ++m)
#pragma unroll
                    for (int n = 0; n < NT; ++n) fetch_shortcut(sc[m][n], rs, p, m, lane_off[n]);
            }
        }
        f32x16m acc[MT][NT];
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int n = 0; n < NT; ++n)
#pragma unroll
                for (int v = 0; v < 16; ++v) acc[m][n][v] = init[n];
#pragma unroll
        for (int t = 0; t < 9; ++t) {
            i32x8 a[MT];
#pragma unroll
            for (int m = 0; m < MT; ++m) a[m] = bits01(act[m][t]);
#pragma unroll
            for (int n = 0; n < NT; ++n) {
                const i32x8 b = bitspm(*reinterpret_cast<const uint32_t *>(filters + wofs + n * 32 * kRow + t * 8));
#pragma unroll
                for (int m = 0; m < MT; ++m) mfma_fp4<32>(acc[m][n], a[m], b);
            }
        }
        const __amdgpu_buffer_rsrc_t ro = make_rsrc(p.out + view.base, view.bytes);
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            uint32_t word[NT];
#pragma unroll
            for (int n = 0; n < NT; ++n) word[n] = 0;
#pragma unroll
            for (int v = 0; v < 16; ++v)
#pragma unroll
                for (int n = 0; n < NT; ++n) finish_register<MODE>(acc[m][n][v], ro, p, m, v, lane_off[n], ea[n], eb[n], sc[m][n][v], word[n]);
            if constexpr (MODE == kModeAffineAddSign) {
                const int pix = tile * PX + m * 32 + l32;
                if (half == 0 && pix < p.total) {
#pragma unroll
                    for (int n = 0; n < NT; ++n)
                        if (ch0 + n * 32 < p.cout) p.epi_bits[(size_t)pix * (p.cout / 32) + ch0 / 32 + n] = word[n];
                }
            }
        }
    }
}

// ---------------------------------------------------------------- 128 to 512 input channels, many pieces
// Bound by memory up to 128 channels at large batch, by the expansion of bits (vector instructions) and the matrix cores
// with 256 and 512.  A wave keeps the bits of 32 filters in registers (9 * CW a lane) for its lifetime; a block is four
// such waves, 128 channels, and walks over tiles of 32 * MT pixels.  The input pixels that a tile's windows reach are
// one contiguous run of memory (image rows included): the block copies it to LDS with coalesced loads while it counts
// the tile before, and a lane reads its taps from there -- from a zero row where the tap is outside the image.  With
// MT = 2 an expanded filter serves two matrix instructions.  Tried against it: filters in LDS and taps fetched by every
// wave (14 x 14 x 256 at batch 256 with epilogue: 30.0 us against 27.2, 28 x 28 x 128: 39.3 against 36.3; the popcount
// kernels before took 50 and 56), four pixel groups per wave (spills with an epilogue).
template <int CW>
struct WindowRow {
    static constexpr int bytes = CW * 32 + 16;  // of a pixel in LDS, expanded: an odd number of 16-byte slots
};
constexpr long long kWindowLdsBytes = 78 * 1024;  // of a block: two blocks of a CU
constexpr int kWindowPieces = 4;  // 16-byte pieces of the next window a thread holds in registers
template <int CW>
struct WindowTile {
    static constexpr int groups32 = CW == 2 ? 1 : 2;  // MT; 128 channels: finer tiles are 3-5 % ahead
};

template <int CW, int MODE>
__global__ __launch_bounds__(256, CW == 2 ? 3 : 2) void bconv3x3_window_kernel(const BconvArgs p) {
    constexpr int MT = WindowTile<CW>::groups32, PX = 32 * MT, RS = WindowRow<CW>::bytes, PP = CW / 2;
    extern __shared__ __attribute__((aligned(16))) unsigned char win[];  // two windows and the zero row
    const int tid = threadIdx.x, lane = tid & 63, half = lane >> 5, l32 = lane & 31;
    const int wib = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int group = (int)p.div_cols.div(blockIdx.x), groups = (int)p.div_cols.div(gridDim.x);
    const int ch32 = ((int)blockIdx.x - group * p.cols) * 4 + wib;  // this wave's 32 channels
    const int ch = ch32 * 32 + l32;
    const bool ch_ok = ch < p.cout;
    const __amdgpu_buffer_rsrc_t rx = make_rsrc(p.x, p.x_bytes), rw = make_rsrc(p.w, p.w_bytes);
    uint32_t w[9][CW];
#pragma unroll
    for (int t = 0; t < 9; ++t) load_dwords<CW>(w[t], rw, ch_ok ? ch * (CW * 72) + t * (CW * 8) + half * (CW * 4) : kOutside);
    const int wbytes = p.window * RS, pieces = p.window * PP;
    if (tid < RS / 16) reinterpret_cast<u32x4 *>(win + p.buffers * wbytes)[tid] = u32x4{0u, 0u, 0u, 0u};

    u32x4 next[kWindowPieces];
    auto fetch = [&](int tile) {
        int y, x;
        const int lo = window_origin(p, tile * PX, y, x) * (CW * 8);  // may lie before the tensor: reads as zero
#pragma unroll
        for (int i = 0; i < kWindowPieces; ++i) {
            const int c = tid + i * 256;
            next[i] = u32x4{0u, 0u, 0u, 0u};
            if (c < pieces) next[i] = __builtin_amdgcn_raw_buffer_load_b128(rx, lo + c * 16, 0, 0);
        }
    };
    auto put = [&](int buf) {
#pragma unroll
        for (int i = 0; i < kWindowPieces; ++i) {
            const int c = tid + i * 256;
            if (c < pieces) {
                i32x4 *d = reinterpret_cast<i32x4 *>(win + buf * wbytes + (c / PP) * RS + (c % PP) * 64);
                d[0] = lower_half(bits01(next[i].x)), d[1] = lower_half(bits01(next[i].y));
                d[2] = lower_half(bits01(next[i].z)), d[3] = lower_half(bits01(next[i].w));
            }
        }
    };
    float ea = 0.f, eb = 0.f;
    if constexpr (MODE != kModeCounts)
        if (ch_ok) ea = p.epi_a[ch], eb = p.epi_b[ch];
    const int lane_off = ch_ok ? (half * 4 * p.cout + ch) * 4 : kOutside;
    int tile = group;
    if (tile < p.px_tiles) fetch(tile);
    uint32_t set = 0;
#pragma unroll
    for (int t = 0; t < 9; ++t)
#pragma unroll
        for (int c = 0; c < CW; ++c) set += __popc(w[t][c]);
    set += __shfl_xor(set, 32);
    const float init = (float)set;
    put(0);
    __syncthreads();

    for (int buf = 0, next_buf; tile < p.px_tiles; tile += groups, buf = next_buf) {
        next_buf = p.buffers == 1 ? 0 : buf ^ 1;
        const bool more = tile + groups < p.px_tiles;
        int tap[MT][9];  // LDS addresses
        {
            int y, x;
            const int lo = window_origin(p, tile * PX, y, x), zero = p.buffers * wbytes;
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                int pix = tile * PX + m * 32 + l32;
                pix = pix < p.total ? pix : p.total - 1;
                int y0, x0;
                const int base = buf * wbytes + (window_origin(p, pix, y0, x0) - lo) * RS + half * (CW * 16);
#pragma unroll
                for (int t = 0; t < 9; ++t) {
                    const int kh = t / 3, kw = t % 3;
                    const bool ok = (unsigned)(y0 + kh) < (unsigned)p.H && (unsigned)(x0 + kw) < (unsigned)p.W;
                    tap[m][t] = ok ? base + (kh * p.W + kw) * RS : zero;
                }
            }
        }
        const TileView view(p, tile * PX);
        float sc[MT][16];
        if constexpr (MODE != kModeCounts) {
            if (p.epi_shortcut) {
                const __amdgpu_buffer_rsrc_t rs = make_rsrc(p.epi_shortcut + view.base, view.bytes);
#pragma unroll
                for (int m = 0; m < MT; ++m) fetch_shortcut(sc[m], rs, p, m, lane_off);
            }
        }
        if (more) fetch(tile + groups);
        f32x16m acc[MT];
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[m][v] = init;
#pragma unroll
        for (int t = 0; t < 9; ++t) {
#pragma unroll
            for (int c = 0; c < CW; ++c) {
                // expanded here, not ahead of the loop: only the 72 registers of 128 channels would fit
                if constexpr (CW >= 4) asm volatile("" : "+v"(w[t][c]));
                const i32x8 b = bitspm(w[t][c]);
#pragma unroll
                for (int m = 0; m < MT; ++m)
                    mfma_fp4<32>(acc[m], upper_zero(*reinterpret_cast<const i32x4 *>(win + tap[m][t] + c * 16)), b);
            }
        }
        if (p.buffers == 1) __syncthreads();  // every wave has read this window
        if (more) put(next_buf);
        const __amdgpu_buffer_rsrc_t ro = make_rsrc(p.out + view.base, view.bytes);
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            uint32_t word = 0;
#pragma unroll
            for (int v = 0; v < 16; ++v) finish_register<MODE>(acc[m][v], ro, p, m, v, lane_off, ea, eb, sc[m][v], word);
            if constexpr (MODE == kModeAffineAddSign) {
                const int pix = tile * PX + m * 32 + l32;
                if (half == 0 && pix < p.total && ch32 * 32 < p.cout) p.epi_bits[(size_t)pix * (p.cout / 32) + ch32] = word;
            }
        }
        __syncthreads();  // the next window is in LDS, this one is dead
    }
}

// Input pixels that the windows of PX consecutive output pixels reach at most, 0 if they are no monotone run (an output
// that reaches past the image so far that the next image's windows start before it).
static int window_pixels(const BconvArgs &a, int px) {
    if ((a.H - (a.OH - 1) * a.stride) * (long long)a.W < (long long)(a.OW - 1) * a.stride || a.W < a.OW - 1) return 0;
    const long long rows = (px - 1 + a.OW - 1) / a.OW, images = (rows + a.OH - 1) / a.OH;  // crossed by a tile at most
    const long long wide = a.W > a.OW ? a.W - a.OW : 0, tall = a.H > a.OH * a.stride ? (long long)(a.H - a.OH * a.stride) * a.W : 0;
    const long long span = (px - 1ll) * a.stride + rows * a.stride * wide + images * tall + 2ll * a.W + 3;
    return span < (1 << 20) ? (int)span : 0;
}

template <class Kernel>
static int resident_blocks_per_cu(Kernel kernel, int threads) {
    int blocks = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&blocks, kernel, threads, 0) != hipSuccess || blocks < 1) blocks = 1;
    return blocks;
}

// Blocks of a launch whose blocks walk over pixel tiles: one per channel tile and group, as many groups as are resident.
static int resident_groups(const BconvArgs &a, int blocks_per_cu, int tiles_per_step) {
    const int wanted = (a.px_tiles + tiles_per_step - 1) / tiles_per_step;
    const int most = (int)((long long)(simd_count() / 4) * blocks_per_cu / a.cols);
    return wanted < most ? wanted : most < 1 ? 1 : most;
}

template <int MODE, int MT, int NT>
static int launch_stream(BconvArgs &a, hipStream_t stream) {
    a.cols = (a.cout + 32 * NT - 1) / (32 * NT);
    a.px_tiles = (int)(((long long)a.total + 32 * MT - 1) / (32 * MT));
    a.div_cols = FastDiv((uint32_t)a.cols);
    static const int blocks_per_cu = resident_blocks_per_cu(bconv3x3_stream_kernel<MODE, MT, NT>, 256);
    int groups = resident_groups(a, blocks_per_cu, 4);
    // equal shares: the blocks that one tile more than the others' per wave would need are not started
    const int per_wave = (a.px_tiles + groups * 4 - 1) / (groups * 4);
    groups = (a.px_tiles + 4 * per_wave - 1) / (4 * per_wave);
    hipLaunchKernelGGL((bconv3x3_stream_kernel<MODE, MT, NT>), dim3((unsigned)(groups * a.cols)), dim3(256), 0, stream, a);
    DAB_LAUNCH_CHECK();
    return DAB_OK;
}

// False when the tile's window does not fit the kernel (wide images over many channels).
template <int CW, int MODE>
static bool window_fits(BconvArgs &a) {
    a.window = window_pixels(a, 32 * WindowTile<CW>::groups32);
    return a.window > 0 && a.window * (CW / 2) <= 256 * kWindowPieces && (a.window + 1ll) * WindowRow<CW>::bytes <= kWindowLdsBytes;
}

template <int CW, int MODE>
static int launch_window(BconvArgs &a, hipStream_t stream) {
    constexpr int PX = 32 * WindowTile<CW>::groups32;
    a.cols = (a.cout + 127) / 128;
    a.px_tiles = (int)(((long long)a.total + PX - 1) / PX);
    a.div_cols = FastDiv((uint32_t)a.cols);
    a.buffers = (2ll * a.window + 1) * WindowRow<CW>::bytes <= kWindowLdsBytes ? 2 : 1;
    const size_t lds = (size_t)(a.buffers * a.window + 1) * WindowRow<CW>::bytes;
    static const int by_registers = resident_blocks_per_cu(bconv3x3_window_kernel<CW, MODE>, 256);
    const int by_lds = (int)(160 * 1024 / (lds + 512));
    const int groups = resident_groups(a, by_registers < by_lds ? by_registers : by_lds, 1);
    static const bool whole_lds = hipFuncSetAttribute(reinterpret_cast<const void *>(bconv3x3_window_kernel<CW, MODE>),
                                                      hipFuncAttributeMaxDynamicSharedMemorySize, (int)kWindowLdsBytes) == hipSuccess;
    (void)whole_lds;
    hipLaunchKernelGGL((bconv3x3_window_kernel<CW, MODE>), dim3((unsigned)(groups * a.cols)), dim3(256), lds, stream, a);
    DAB_LAUNCH_CHECK();
    return DAB_OK;
}

template <int CW, int MODE, int T, int NT>
static int launch_split(BconvArgs &a, hipStream_t stream) {
    a.cols = (a.cout + T * NT - 1) / (T * NT);
    a.px_tiles = (int)(((long long)a.total + T - 1) / T);
    a.div_cols = FastDiv((uint32_t)a.cols);
    const long long blocks = (long long)a.px_tiles * a.cols;
    if (blocks >= (1ll << 31)) return fail(DAB_EUNSUPPORTED, "dab_bconv3x3: too many work units");
    hipLaunchKernelGGL((bconv3x3_split_kernel<CW, MODE, T, NT>), dim3((unsigned)blocks), dim3(192), 0, stream, a);
    DAB_LAUNCH_CHECK();
    return DAB_OK;
}

// Which kernel, by the number of 32-pixel x 32-channel pieces of the output.  Measured on the seven ResNet-18 stage
// shapes at batches 1 to 256 with counts and with Affine + Add + sign bits (us with the latter):
//   16-pixel tiles up to 160 pieces (224 with 64 input channels), where they give the chip more waves: 7x7x512 at batch
//   4 (112 pieces) 3.4 against 3.9, 14x14x256 there (200) 3.5 against 3.4; 56x56x64 at batch 1 (196) 2.66 against 2.72
//   then 32-pixel tiles of 32 channels, from 1280 pieces of 64: 14x14x256 at batch 16 (784) 4.7 against 5.2, at batch
//   32 (1568) 6.9 against 6.3; 7x7x512 at batch 64 (1568) 10.1 against 9.4
//   the walking kernels from 768 pieces (64 input channels) and 2048 (deeper): 56x56x64 at batch 4 (784) 3.8 either
//   way, at batch 8 4.5 against 4.8; 28x28x128 at batch 32 (3136) 7.4 against 7.6, 14x14x256 at batch 64 (3136) 8.7
//   against 9.9, 7x7x512 at batch 64 (1568) 9.0 against 9.3, the stride-2 layer into it there (1568) 6.9 against 6.6
template <int CW, int MODE>
static int launch_bconv3x3(BconvArgs &a, hipStream_t s) {
    const long long pieces = (((long long)a.total + 31) / 32) * ((a.cout + 31) / 32);
    if constexpr (CW == 1) {
        if (pieces >= 768) {
            // Counts: 32 channels a wave where that is half the output's channels or more, else 64; with an epilogue 64,
            // from 6000 pieces with two pixel groups (56x56x64 at batch 64: 19.3 us against 21.9, at batch 32 9.9
            // against 11; 56x56x64 -> 128 at stride 2, batch 64: 9.8 against 10.6).
            if constexpr (MODE == kModeCounts) {
                if (a.cout <= 64) return launch_stream<MODE, 1, 1>(a, s);
                return launch_stream<MODE, 1, 2>(a, s);
            } else {
                if (pieces >= 6000) return launch_stream<MODE, 2, 2>(a, s);
                return launch_stream<MODE, 1, 2>(a, s);
            }
        }
    } else if constexpr (CW <= 8) {
        if (pieces >= 2048 && window_fits<CW, MODE>(a)) return launch_window<CW, MODE>(a, s);
    }
    if constexpr (CW <= 8) {
        if (pieces <= (CW == 1 ? 224 : 160)) return launch_split<CW, MODE, 16, (CW <= 2 ? 2 : 1)>(a, s);
        if (pieces >= 1280) return launch_split<CW, MODE, 32, 2>(a, s);
    }
    return launch_split<CW, MODE, 32, 1>(a, s);
}

// ---------------------------------------------------------------- size classes
// What the probes of dabnn_hip_tuning.h answer: a problem's size class, 0 (few 64-pixel tiles), 1, 2 (many) or 3 (256 and
// 512 input channels between small and mid-sized), from the work per SIMD.  Net::prepare links the layers of a net by it.
static bool few_tiles(long long tiles, int cin, int cout) { return tiles * (cout / 8) <= (long long)simd_count() * (cin >= 512 ? 2 : 1); }

static bool deep_mid_sized(long long tiles, int cin, int cout, int stride, int mode) {
    if (cout % 8 != 0 || !(cin == 512 || cin == 256)) return false;
    const bool deep = cin == 512 || stride >= 2;  // 512 input channels, or 256 at stride 2
    const long long work = tiles * cout, simds = simd_count();
    if (mode == kModeCounts) return work <= (deep ? 28 : 16) * simds;
    if (mode == kModeAffineAdd) return work <= simds || (work >= 6 * simds && work <= (deep ? 28 : 16) * simds);
    return cout % 64 == 0 && work >= (cin == 512 ? 8 : 6) * simds && work <= 28 * simds;
}

static int size_class(long long tiles, int cin, int cout, int stride, int mode) {
    if (deep_mid_sized(tiles, cin, cout, stride, mode)) return 3;
    if (few_tiles(tiles, cin, cout)) return 0;
    const long long simds = simd_count();
    if (cin <= 128) {
        const long long units = tiles * (cout / 8);
        if (mode != kModeCounts) return units >= (cin == 64 ? 4ll : 8ll) * simds * 4 ? 2 : 1;
        if (cin == 64) return stride == 1 && units >= 24 * simds && units < 44 * simds ? 2 : 1;
        return units >= (stride >= 2 ? 4 : 16) * simds ? 2 : 1;
    }
    const long long big_units = tiles * (cout / (cin == 256 ? 8 : 4));
    const long long per_wave = (mode == kModeCounts && cin == 512) ? 3 : 6;
    return cout % 8 == 0 && big_units >= per_wave * simds * (cin == 256 ? 4 : 3) ? 2 : 1;
}

}  // namespace dab

static int bconv3x3_impl(const char *fn, const uint64_t *x, int n, int h, int w, int cin, const uint64_t *wgt, int cout,
                         int stride, int pad, const float *a_coef, const float *b_coef, const float *shortcut, int mode,
                         float *out, uint64_t *out_packed, dab_stream_t stream) {
    using namespace dab;
    DAB_REQUIRE(x && wgt && out, "%s: null pointer", fn);
    DAB_REQUIRE(n > 0 && h > 0 && w > 0 && cin > 0 && cout > 0, "%s: non-positive dimension", fn);
    DAB_REQUIRE(stride > 0 && pad >= 0, "%s: stride %d pad %d", fn, stride, pad);
    DAB_REQUIRE(cin % 64 == 0, "%s: cin %d is not a multiple of 64", fn, cin);
    DAB_REQUIRE(h + 2 * pad >= 3 && w + 2 * pad >= 3, "%s: input smaller than the kernel", fn);
    const bool counts_1024 = cin == 1024 && mode == kModeCounts;  // no fused epilogue for 1024 input channels
    if (!(cin == 64 || cin == 128 || cin == 256 || cin == 512 || counts_1024) || cout % 8 != 0)
        return fail(DAB_EUNSUPPORTED, "%s: cin %d / cout %d not covered by the direct kernel", fn, cin, cout);
    DAB_REQUIRE((reinterpret_cast<uintptr_t>(x) & 15) == 0 && (reinterpret_cast<uintptr_t>(wgt) & 7) == 0 &&
                    (reinterpret_cast<uintptr_t>(out) & 15) == 0,
                "%s: buffers must be 16-byte aligned", fn);
    const bool fused = mode != kModeCounts;
    if (mode == kModeAffineAddSign) {
        DAB_REQUIRE(out_packed, "%s: null pointer", fn);
        DAB_REQUIRE((reinterpret_cast<uintptr_t>(out_packed) & 7) == 0, "%s: buffers must be 16-byte aligned", fn);
        if (cout % 64 != 0) return fail(DAB_EUNSUPPORTED, "%s: cout %d is not a multiple of 64", fn, cout);
    }
    if (fused) {
        DAB_REQUIRE(a_coef && b_coef, "%s: null affine coefficients", fn);
        DAB_REQUIRE((reinterpret_cast<uintptr_t>(a_coef) & 15) == 0 && (reinterpret_cast<uintptr_t>(b_coef) & 15) == 0 &&
                        (reinterpret_cast<uintptr_t>(shortcut) & 15) == 0,
                    "%s: coefficient and shortcut buffers must be 16-byte aligned", fn);
    }

    BconvArgs a;
    a.x = x, a.w = wgt, a.out = out;
    a.epi_a = a_coef, a.epi_b = b_coef, a.epi_shortcut = shortcut;
    a.epi_bits = reinterpret_cast<uint32_t *>(out_packed);
    a.H = h, a.W = w;
    a.OH = out_dim(h, pad, 3, 1, stride), a.OW = out_dim(w, pad, 3, 1, stride);
    const long long total = (long long)n * a.OH * a.OW;
    const long long x_bytes = (long long)n * h * w * (cin / 64) * 8, w_bytes = (long long)cout * 9 * (cin / 64) * 8;
    if (total >= (1ll << 31) - 64 || x_bytes >= (1ll << 31) || total * cout >= (1ll << 40) || w_bytes >= (1ll << 31) || cout >= (1 << 22))
        return fail(DAB_EUNSUPPORTED, "%s: tensor too large for 32-bit pixel indexing", fn);
    a.total = (int)total;
    a.cout = cout, a.stride = stride, a.pad = pad;
    a.x_bytes = (uint32_t)x_bytes, a.w_bytes = (uint32_t)w_bytes;
    a.div_ow = FastDiv((uint32_t)a.OW), a.div_oh = FastDiv((uint32_t)a.OH);
    a.cols = a.px_tiles = a.window = 0;
    hipStream_t s = as_stream(stream);
    switch (mode * 32 + cin / 64) {
        case kModeCounts * 32 + 1: return launch_bconv3x3<1, kModeCounts>(a, s);
        case kModeCounts * 32 + 2: return launch_bconv3x3<2, kModeCounts>(a, s);
        case kModeCounts * 32 + 4: return launch_bconv3x3<4, kModeCounts>(a, s);
        case kModeCounts * 32 + 8: return launch_bconv3x3<8, kModeCounts>(a, s);
        case kModeCounts * 32 + 16: return launch_bconv3x3<16, kModeCounts>(a, s);
        case kModeAffineAdd * 32 + 1: return launch_bconv3x3<1, kModeAffineAdd>(a, s);
        case kModeAffineAdd * 32 + 2: return launch_bconv3x3<2, kModeAffineAdd>(a, s);
        case kModeAffineAdd * 32 + 4: return launch_bconv3x3<4, kModeAffineAdd>(a, s);
        case kModeAffineAdd * 32 + 8: return launch_bconv3x3<8, kModeAffineAdd>(a, s);
        case kModeAffineAddSign * 32 + 1: return launch_bconv3x3<1, kModeAffineAddSign>(a, s);
        case kModeAffineAddSign * 32 + 2: return launch_bconv3x3<2, kModeAffineAddSign>(a, s);
        case kModeAffineAddSign * 32 + 4: return launch_bconv3x3<4, kModeAffineAddSign>(a, s);
        case kModeAffineAddSign * 32 + 8: return launch_bconv3x3<8, kModeAffineAddSign>(a, s);
    }
    return fail(DAB_EINVAL, "%s: bad mode", fn);
}
extern "C" int dab_bconv3x3(const uint64_t *x, int n, int h, int w, int cin, const uint64_t *wgt, int cout, int stride,
                            int pad, float *out, dab_stream_t stream) {
    return bconv3x3_impl("dab_bconv3x3", x, n, h, w, cin, wgt, cout, stride, pad, nullptr, nullptr, nullptr, dab::kModeCounts,
                         out, nullptr, stream);
}

extern "C" int dab_bconv3x3_affine_add(const uint64_t *x, int n, int h, int w, int cin, const uint64_t *wgt, int cout,
                                       int stride, int pad, const float *a, const float *b, const float *shortcut,
                                       float *out, dab_stream_t stream) {
    return bconv3x3_impl("dab_bconv3x3_affine_add", x, n, h, w, cin, wgt, cout, stride, pad, a, b, shortcut,
                         dab::kModeAffineAdd, out, nullptr, stream);
}

extern "C" int dab_bconv3x3_affine_add_sign(const uint64_t *x, int n, int h, int w, int cin, const uint64_t *wgt, int cout,
                                            int stride, int pad, const float *a, const float *b, const float *shortcut,
                                            float *out, uint64_t *out_packed, dab_stream_t stream) {
    return bconv3x3_impl("dab_bconv3x3_affine_add_sign", x, n, h, w, cin, wgt, cout, stride, pad, a, b, shortcut,
                         dab::kModeAffineAddSign, out, out_packed, stream);
}

extern "C" int dab_bconv3x3_splits_depth(int64_t n_out_pixels, int cin, int cout) {
    if (n_out_pixels <= 0 || cout <= 0 || cout % 8 != 0 || !(cin == 64 || cin == 128 || cin == 256 || cin == 512)) return 0;
    return dab::few_tiles((n_out_pixels + 63) / 64, cin, cout) ? 1 : 0;
}

extern "C" int dab_bconv3x3_fused_shares_tiles(int64_t n_out_pixels, int cin, int cout) {
    if (n_out_pixels <= 0 || cout <= 0) return 0;
    // a first-stage block at a batch where its shortcut and result are what bounds it: 32 tiles of 64 pixels per CU
    return cin == 64 && cout % 64 == 0 && (n_out_pixels + 63) / 64 >= 32ll * (dab::simd_count() / 4) ? 1 : 0;
}

static bool has_size_class(int64_t n_out_pixels, int cin, int cout, int stride) {
    return n_out_pixels > 0 && cout > 0 && cout % 8 == 0 && stride > 0 && (cin == 64 || cin == 128 || cin == 256 || cin == 512);
}

extern "C" int dab_bconv3x3_build(int64_t n_out_pixels, int cin, int cout) {
    if (!has_size_class(n_out_pixels, cin, cout, 1)) return -1;
    return dab::size_class((n_out_pixels + 63) / 64, cin, cout, 1, dab::kModeAffineAdd);
}

extern "C" int dab_bconv3x3_epilogue_build(int64_t n_out_pixels, int cin, int cout, int stride, int with_sign) {
    if (!has_size_class(n_out_pixels, cin, cout, stride) || (with_sign && cout % 64 != 0)) return -1;
    return dab::size_class((n_out_pixels + 63) / 64, cin, cout, stride, with_sign ? dab::kModeAffineAddSign : dab::kModeAffineAdd);
}

extern "C" int dab_bconv3x3_counts_build(int64_t n_out_pixels, int cin, int cout, int stride) {
    if (!has_size_class(n_out_pixels, cin, cout, stride)) return -1;
    return dab::size_class((n_out_pixels + 63) / 64, cin, cout, stride, dab::kModeCounts);
}
