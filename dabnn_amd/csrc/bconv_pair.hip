// Two residual layers of a first-stage block in one pass: v1 = a1 * bconv3x3(sign(v0)) + b1 + v0, v2 = a2 * bconv3x3(sign(v1)) + b2 + v1,
// 64 channels, stride 1, pad 1 (dabnn/layers/BinConv.cpp:144-191, Affine.cpp:10-23, Add.cpp:7-17, twice).
//
// One such layer is bound by memory: at batch 256 of 56 x 56 it reads a 205 MB shortcut and writes a 205 MB result in 72 to 80
// us.  Here v1 never leaves the chip: a block makes R rows of v2 of one image, and with them the rows of v1 that they need --
// R + 2, two of which its neighbours make too.  v1 stays in the accumulator layout in registers, where it is the second layer's
// shortcut; its sign bits go through LDS, where they are the second layer's input.
//
// Pixels are tiles of 32 that lie one behind the other in memory, full rows, so that a tile's values and sign bits are contiguous.
// Tile `above` starts with the strip's first pixel; the tiles before it hold the row above the strip.  A wave owns four tiles
// and all 64 channels (128 registers of v1), and multiplies two of them at a time by the filters, which LDS holds in the matrix
// instruction's form (fp4_core.h): an expanded pixel serves two channel groups, a fetched filter two tiles.
#include "fp4_core.h"

namespace dab {

struct BconvPairArgs {
    const uint64_t *x;        // sign bits of v0
    const float *shortcut;    // v0
    const uint64_t *w[2];
    const float *a[2], *b[2];
    float *out;
    uint64_t *bits;           // of v2, or null
    int H, W;
    int rows, bands;          // of a strip, strips of an image
    int above;                // tiles before the strip: ceil(W / 32)
    FastDiv div_bands, div_w;
};

constexpr int kPairTiles = 16;  // of a block: four waves with four each
constexpr int kPairFilterBytes = 9 * 2 * 64 * 16;

// The packed rows of a strip and the filters of both layers, which LDS holds before anything is counted.  They are asked for
// before the floats: loads come back in the order they were asked for, and the floats are only wanted behind the first tile's counts.
// (The floats first, us in a graph by itself: 56 x 56 at 40 images 18.1 instead of 17.6, at 100 43 / 38, at 256 90 either way; the pooled form at
// 256 77 instead of 66.  The results are written through the L2: the pass behind this one reads them, and both together take 2 to 4 % less
// than with streaming stores.)
struct PairStage {
    // (at most 800 words: five rows of 160)
    uint64_t rows[4], filters[5];
    float coefficient;  // a1, b1, a2, b2: one per thread
    // src: `words` words of the packed rows; bits, w: LDS
    __device__ __forceinline__ void fetch(const uint64_t *src, int words, const uint64_t *const (&w)[2], const float *const (&a)[2], const float *const (&b)[2], int tid) {
        coefficient = (tid < 64 ? a[0] : tid < 128 ? b[0] : tid < 192 ? a[1] : b[1])[tid & 63];
#pragma unroll
        for (int i = 0; i < 4; ++i) rows[i] = tid + 256 * i < words ? src[tid + 256 * i] : 0;
#pragma unroll
        for (int i = 0; i < 5; ++i) {
            const int j = tid + 256 * i;
            filters[i] = j < 64 * 9 ? w[0][j] : j < 2 * 64 * 9 ? w[1][j - 64 * 9] : 0;
        }
    }
    // first: of the row that the first word belongs to; the filters expanded, [layer][tap][32 channels][half][channel] of 16 bytes
    __device__ __forceinline__ void put(unsigned char *first, int words, int pitch, int width, const FastDiv &div_w, unsigned char *lds, uint32_t (*pop)[64], float *coef, int tid) const {
        coef[tid] = coefficient;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int j = tid + 256 * i, row = (int)div_w.div(j), col = j - row * width;
            if (j < words) *reinterpret_cast<uint64_t *>(first + row * pitch + (col + 1) * 8) = rows[i];
        }
#pragma unroll
        for (int i = 0; i < 5; ++i) {
            const int j = tid + 256 * i;
            if (j >= 2 * 64 * 9) break;
            const int layer = j >= 64 * 9, c = j - layer * (64 * 9), ch = c / 9, tap = c - ch * 9;
            unsigned char *d = lds + layer * kPairFilterBytes + ((tap * 2 + (ch >> 5)) * 64 + (ch & 31)) * 16;
            *reinterpret_cast<i32x4 *>(d) = lower_half(bitspm((uint32_t)filters[i]));
            *reinterpret_cast<i32x4 *>(d + 32 * 16) = lower_half(bitspm((uint32_t)(filters[i] >> 32)));
            atomicAdd(&pop[layer][ch], (uint32_t)__popcll(filters[i]));
        }
    }
};

template <bool SIGN>
__global__ __launch_bounds__(256, 2) void bconv3x3_pair_kernel(const BconvPairArgs p) {
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    __shared__ uint32_t pop[2][64];  // set bits per filter
    __shared__ float coef[2][2][64];  // a and b of the layers
    const int tid = threadIdx.x, lane = tid & 63, half = lane >> 5, l32 = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t item = xcd_contiguous_block(blockIdx.x, gridDim.x);  // neighbouring strips share rows: on one XCD
    const int img = (int)p.div_bands.div(item), r0 = ((int)item - img * p.bands) * p.rows;
    const int rows = p.H - r0 < p.rows ? p.H - r0 : p.rows;
    const int pitch = (p.W + 2) * 8;                           // of a row of packed pixels in LDS, zero words either side
    unsigned char *const bits0 = lds + 2 * kPairFilterBytes;   // image rows r0 - 2 .. r0 + rows + 1
    unsigned char *const bits1 = bits0 + (p.rows + 4) * pitch;  // of v1: r0 - 1 .. r0 + rows
    const size_t strip = ((size_t)img * p.H + r0) * p.W;       // its first pixel

    const int in0 = r0 >= 2 ? r0 - 2 : 0, in1 = r0 + rows + 2 < p.H ? r0 + rows + 2 : p.H, words = (in1 - in0) * p.W;
    PairStage stage;
    stage.fetch(p.x + ((size_t)img * p.H + in0) * p.W, words, p.w, p.a, p.b, tid);
    __builtin_amdgcn_sched_barrier(0);
    // v0 of the wave's tiles; 0 where there is nothing (above the image, past its end)
    auto tile_of = [&](int i) { return 2 * wave + (i & 1) + 8 * (i >> 1); };
    const int lane_off = half * 4 * 256 + l32 * 4;
    auto row_off = [](int n, int v) { return (8 * (v / 4) + v % 4) * 256 + n * 128; };
    const int image_left = (p.H - r0) * p.W;  // pixels from the strip's first to the image's end
    float val[4][2][16];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int first = (tile_of(i) - p.above) * 32;
        const bool there = (first >= 0 || r0 > 0) && first < image_left;
        const __amdgpu_buffer_rsrc_t rs = make_rsrc(p.shortcut + (strip + (there ? first : 0)) * 64, there ? (uint32_t)(image_left - first) * 256u : 0u);
#pragma unroll
        for (int n = 0; n < 2; ++n)
#pragma unroll
            for (int v = 0; v < 16; ++v) val[i][n][v] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, lane_off, row_off(n, v), 0));
    }

    if (tid < 128) pop[tid >> 6][tid & 63] = 0;
    const int bit_bytes = (2 * p.rows + 6) * pitch;
    for (int i = tid * 8; i < bit_bytes; i += 256 * 8) *reinterpret_cast<uint64_t *>(bits0 + i) = 0;
    __syncthreads();
    stage.put(bits0 + (in0 - (r0 - 2)) * pitch, words, pitch, p.W, p.div_w, lds, pop, &coef[0][0][0], tid);
    __syncthreads();

    auto layer = [&](auto which) __attribute__((always_inline)) {
        constexpr int L = decltype(which)::value;
        float init[2], ea[2], eb[2];
#pragma unroll
        for (int n = 0; n < 2; ++n) {
            init[n] = (float)pop[L][n * 32 + l32];
            ea[n] = coef[L][0][n * 32 + l32], eb[n] = coef[L][1][n * 32 + l32];
        }
        const unsigned char *filter = lds + L * kPairFilterBytes + lane * 16;
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            // two neighbouring tiles; first0: the first one's first pixel, counted from the strip's
            const int first0 = (tile_of(2 * s) - p.above) * 32;
            if (L == 0 ? first0 >= (rows + 1) * p.W : (first0 + 64 <= 0 || first0 >= rows * p.W)) continue;
            int row[2], col[2];  // row: from r0 - 2 on
            f32x16m acc[2][2];
            const unsigned char *window[2];
#pragma unroll
            for (int m = 0; m < 2; ++m) {
                const int u = first0 + m * 32 + l32 + 2 * p.W;
                row[m] = (int)p.div_w.div(u < 0 ? 0 : u), col[m] = u - row[m] * p.W;
                // v1's rows are 1 .. rows + 2, v2's 2 .. rows + 1; what lies outside is computed from some window and not used
                const int lowest = 1 + L, highest = rows + 2 - L, r = row[m] < lowest ? lowest : row[m] > highest ? highest : row[m];
                window[m] = (L == 0 ? bits0 : bits1) + (r - lowest) * pitch + col[m] * 8 + half * 4;
#pragma unroll
                for (int n = 0; n < 2; ++n)
#pragma unroll
                    for (int v = 0; v < 16; ++v) acc[m][n][v] = init[n];
            }
#pragma unroll
            for (int tap = 0; tap < 9; ++tap) {
                i32x8 a[2];
#pragma unroll
                for (int m = 0; m < 2; ++m) a[m] = bits01(*reinterpret_cast<const uint32_t *>(window[m] + (tap / 3) * pitch + (tap % 3) * 8));
#pragma unroll
                for (int n = 0; n < 2; ++n) {
                    const i32x8 b = upper_zero(*reinterpret_cast<const i32x4 *>(filter + (tap * 2 + n) * 64 * 16));
#pragma unroll
                    for (int m = 0; m < 2; ++m) mfma_fp4<32>(acc[m][n], a[m], b);
                }
            }
#pragma unroll
            for (int m = 0; m < 2; ++m) {
                const int i = 2 * s + m, first = first0 + m * 32;
                const bool inside = L == 1 && first >= 0 && first < rows * p.W;  // (a tile of v2)
                const __amdgpu_buffer_rsrc_t ro = make_rsrc(p.out + (strip + (inside ? first : 0)) * 64, inside ? (uint32_t)(rows * p.W - first) * 256u : 0u);
                uint32_t word[2] = {0, 0};
#pragma unroll
                for (int v = 0; v < 16; ++v)
#pragma unroll
                    for (int n = 0; n < 2; ++n) {
#pragma clang fp contract(off)
                        float r = ea[n] * acc[m][n][v];
                        r = r + eb[n];
                        r = r + val[i][n][v];
                        if constexpr (L == 0)
                            val[i][n][v] = r;
                        else
                            __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, r), ro, lane_off, row_off(n, v), kStoreThrough);
                        if constexpr (L == 0 || SIGN) {
                            const uint64_t mask = __ballot(r > 0.f);
                            word[n] = dab_writelane((uint32_t)mask, 8 * (v / 4) + v % 4, word[n]);
                            word[n] = dab_writelane((uint32_t)(mask >> 32), 8 * (v / 4) + v % 4 + 4, word[n]);
                        }
                    }
                if constexpr (L == 0) {
                    const int y = r0 - 2 + row[m];
                    if (half == 0 && row[m] >= 1 && row[m] <= rows + 2 && y >= 0 && y < p.H)
                        *reinterpret_cast<u32x2 *>(bits1 + (row[m] - 1) * pitch + (col[m] + 1) * 8) = u32x2{word[0], word[1]};
                } else if constexpr (SIGN) {
                    if (half == 0 && inside && first + l32 < rows * p.W) p.bits[strip + first + l32] = ((uint64_t)word[1] << 32) | word[0];
                }
            }
        }
    };
    layer(std::integral_constant<int, 0>{});
    __syncthreads();
    layer(std::integral_constant<int, 1>{});
}

// Rows of a strip for images of h x w: as many as 16 tiles hold with the row above and the row below, or fewer where a launch
// would leave CUs without a block; 0 if the kernel does not take them.
static int pair_rows(int n, int h, int w) {
    const int above = (w + 31) / 32;
    if (above * 32 > 2 * w) return 0;  // a tile's first pixel is at most two rows above the strip
    int most = ((kPairTiles - above) * 32) / w - 1;
    if (most > h) most = h;
    if (most < 1) return 0;
    if (most * w < above * 32 && most < h) return 0;  // the tiles before the second strip would start before the tensor
    const int cus = simd_count() / 4;
    // equal strips
    int bands = (h + most - 1) / most;
    while ((long long)n * bands < cus && (h + bands) / (bands + 1) * w >= above * 32 && (h + bands) / (bands + 1) >= 2) ++bands;
    return (h + bands - 1) / bands;
}

// Strips of an image, or 0 where the kernel does not take the problem.
static int pair_bands(int n, int h, int w) {
    const int rows = pair_rows(n, h, w);
    if (rows == 0) return 0;
    const int bands = (h + rows - 1) / rows;
    return (long long)h * w * 256 < (1ll << 31) && (long long)n * bands < kMostBlocks ? bands : 0;
}

// ---------------------------------------------------------------- the same for a pass whose result is only pooled
// Before a down-sampling block the second layer's result is read by an AvePool 2x2 and, as sign bits, by a binary convolution:
// the pass writes the pooled tensor and the bits, a quarter of the bytes, and its reader fetches a quarter.  A tile's 32 pixels are
// eight 2x2 windows, in the order of the pooled tensor, one window the four registers of an accumulator quad, so that pooling
// takes no exchange.  A strip has an even number of rows; the rows above and below it, of which only the sign bits are wanted, are a
// fifth tile of each wave that no register outlives, so that a strip has eight rows of 56 where the kernel above has seven.
// 56 x 56 at batch 256, and the block's first layer behind it (bconv_down.hip), us in a graph: the pass 66 (unpooled 90 to 93), that layer 51
// (62), one behind the other 125 (159).
struct BconvPairPoolArgs {
    const uint64_t *x;
    const float *shortcut;
    const uint64_t *w[2];
    const float *a[2], *b[2];
    float *pooled;
    uint64_t *bits;
    int H, W;
    int rows, bands;
    uint32_t image_bytes;  // of the shortcut
    FastDiv div_bands, div_w, div_half_w;
};

__global__ __launch_bounds__(256, 2) void bconv3x3_pair_pool_kernel(const BconvPairPoolArgs p) {
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    __shared__ uint32_t pop[2][64];
    __shared__ float coef[2][2][64];
    const int tid = threadIdx.x, lane = tid & 63, half = lane >> 5, l32 = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t item = xcd_contiguous_block(blockIdx.x, gridDim.x);
    const int img = (int)p.div_bands.div(item), r0 = ((int)item - img * p.bands) * p.rows;
    const int rows = p.H - r0 < p.rows ? p.H - r0 : p.rows, half_w = p.W >> 1, windows = (rows >> 1) * half_w;
    const int pitch = (p.W + 2) * 8;
    unsigned char *const bits0 = lds + 2 * kPairFilterBytes;   // image rows r0 - 2 .. r0 + rows + 1
    unsigned char *const bits1 = bits0 + (p.rows + 4) * pitch;  // of v1: r0 - 1 .. r0 + rows
    const size_t image = (size_t)img * p.H * p.W;               // its first pixel
    auto tile_of = [&](int i) { return 2 * wave + (i & 1) + 8 * (i >> 1); };
    const __amdgpu_buffer_rsrc_t rs = make_rsrc(p.shortcut + image * 64, p.image_bytes);
    constexpr int kNowhere = (int)0x80000000;  // beyond the image: loads return zero

    const int in0 = r0 >= 2 ? r0 - 2 : 0, in1 = r0 + rows + 2 < p.H ? r0 + rows + 2 : p.H, words = (in1 - in0) * p.W;
    PairStage stage;
    stage.fetch(p.x + image + (size_t)in0 * p.W, words, p.w, p.a, p.b, tid);
    __builtin_amdgcn_sched_barrier(0);
    // v0: the row above the strip and the one below it (pixel j of the two, one behind the other) ...
    float edge[2][16];
#pragma unroll
    for (int v = 0; v < 16; ++v) {
        const int j = wave * 32 + 8 * (v / 4) + 4 * half + v % 4;
        const int pix = (r0 - 1) * p.W + j + (j >= p.W ? rows * p.W : 0);
        const int off = j < 2 * p.W && pix >= 0 ? pix * 256 + l32 * 4 : kNowhere;
#pragma unroll
        for (int n = 0; n < 2; ++n) edge[n][v] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, off + n * 128, 0, 0));
    }
    // ... and of the wave's four tiles
    float val[4][2][16];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int win = tile_of(i) * 8 + 2 * q + half, rp = (int)p.div_half_w.div((uint32_t)win);
            const int off = win < windows ? ((r0 + 2 * rp) * p.W + 2 * (win - rp * half_w)) * 256 + l32 * 4 : kNowhere;
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int n = 0; n < 2; ++n)
                    val[i][n][4 * q + e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, off + (e & 1) * 256 + n * 128, (e >> 1) * p.W * 256, 0));
        }

    if (tid < 128) pop[tid >> 6][tid & 63] = 0;
    const int bit_bytes = (2 * p.rows + 6) * pitch;
    for (int i = tid * 8; i < bit_bytes; i += 256 * 8) *reinterpret_cast<uint64_t *>(bits0 + i) = 0;
    __syncthreads();
    stage.put(bits0 + (in0 - (r0 - 2)) * pitch, words, pitch, p.W, p.div_w, lds, pop, &coef[0][0][0], tid);
    __syncthreads();

    auto value = [](float cnt, float a, float b, float add) {
#pragma clang fp contract(off)
        float r = a * cnt;
        r = r + b;
        return r + add;
    };
    auto layer = [&](auto which) __attribute__((always_inline)) {
        constexpr int L = decltype(which)::value;
        float init[2], ea[2], eb[2];
#pragma unroll
        for (int n = 0; n < 2; ++n) {
            init[n] = (float)pop[L][n * 32 + l32];
            ea[n] = coef[L][0][n * 32 + l32], eb[n] = coef[L][1][n * 32 + l32];
        }
        const unsigned char *filter = lds + L * kPairFilterBytes + lane * 16;
        // counts of M tiles whose lanes' windows are at `window`
        auto count = [&](auto tiles, const unsigned char *const *window, f32x16m (*acc)[2]) __attribute__((always_inline)) {
            constexpr int M = decltype(tiles)::value;
#pragma unroll
            for (int m = 0; m < M; ++m)
#pragma unroll
                for (int n = 0; n < 2; ++n)
#pragma unroll
                    for (int v = 0; v < 16; ++v) acc[m][n][v] = init[n];
#pragma unroll
            for (int tap = 0; tap < 9; ++tap) {
                i32x8 a[M];
#pragma unroll
                for (int m = 0; m < M; ++m) a[m] = bits01(*reinterpret_cast<const uint32_t *>(window[m] + (tap / 3) * pitch + (tap % 3) * 8));
#pragma unroll
                for (int n = 0; n < 2; ++n) {
                    const i32x8 b = upper_zero(*reinterpret_cast<const i32x4 *>(filter + (tap * 2 + n) * 64 * 16));
#pragma unroll
                    for (int m = 0; m < M; ++m) mfma_fp4<32>(acc[m][n], a[m], b);
                }
            }
        };
        auto put_sign = [](uint32_t (&word)[2], int n, int v, float r) __attribute__((always_inline)) {
            const uint64_t mask = __ballot(r > 0.f);
            word[n] = dab_writelane((uint32_t)mask, 8 * (v / 4) + v % 4, word[n]);
            word[n] = dab_writelane((uint32_t)(mask >> 32), 8 * (v / 4) + v % 4 + 4, word[n]);
        };
        if constexpr (L == 0) {
            const int j = wave * 32 + l32, below = j >= p.W, col = j - (below ? p.W : 0);
            const bool there = j < 2 * p.W && (below ? r0 + rows < p.H : r0 > 0);
            if (wave * 32 < 2 * p.W) {
                const unsigned char *window[1] = {bits0 + (there && below ? rows + 1 : 0) * pitch + (there ? col : 0) * 8 + half * 4};
                f32x16m acc[1][2];
                count(std::integral_constant<int, 1>{}, window, acc);
                uint32_t word[2] = {0, 0};
#pragma unroll
                for (int v = 0; v < 16; ++v)
#pragma unroll
                    for (int n = 0; n < 2; ++n) put_sign(word, n, v, value(acc[0][n][v], ea[n], eb[n], edge[n][v]));
                if (half == 0 && there) *reinterpret_cast<u32x2 *>(bits1 + (below ? rows + 1 : 0) * pitch + (col + 1) * 8) = u32x2{word[0], word[1]};
            }
        }
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            if (tile_of(2 * s) * 8 >= windows) continue;
            int row[2], col[2];  // of the lane's pixel, from r0 on
            bool there[2];
            const unsigned char *window[2];
            f32x16m acc[2][2];
#pragma unroll
            for (int m = 0; m < 2; ++m) {
                const int win = tile_of(2 * s + m) * 8 + l32 / 4;
                there[m] = win < windows;
                const int rp = (int)p.div_half_w.div((uint32_t)(there[m] ? win : 0));
                row[m] = 2 * rp + ((l32 >> 1) & 1), col[m] = 2 * ((there[m] ? win : 0) - rp * half_w) + (l32 & 1);
                window[m] = (L == 0 ? bits0 + pitch : bits1) + row[m] * pitch + col[m] * 8 + half * 4;
            }
            count(std::integral_constant<int, 2>{}, window, acc);
#pragma unroll
            for (int m = 0; m < 2; ++m) {
                const int i = 2 * s + m;
                const size_t first = (size_t)img * (p.H >> 1) * half_w + (size_t)(r0 >> 1) * half_w;  // the strip's first pooled pixel
                const __amdgpu_buffer_rsrc_t ro = make_rsrc(p.pooled + first * 64, (uint32_t)windows * 256u);
                uint32_t word[2] = {0, 0};
#pragma unroll
                for (int n = 0; n < 2; ++n)
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
#pragma clang fp contract(off)
                        float sum = 0.f;  // ave_pool_fallback's order (dabnn/layers/AvePool.cpp:84-123)
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            const int v = 4 * q + e;
                            const float r = value(acc[m][n][v], ea[n], eb[n], val[i][n][v]);
                            if constexpr (L == 0)
                                val[i][n][v] = r;
                            else
                                sum = sum + r;
                            put_sign(word, n, v, r);
                        }
                        if constexpr (L == 1)
                            __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, sum * 0.25f), ro,
                                                                  (tile_of(i) * 8 + 2 * q + half) * 256 + l32 * 4 + n * 128, 0, kStoreThrough);
                    }
                if (half == 0 && there[m]) {
                    if constexpr (L == 0)
                        *reinterpret_cast<u32x2 *>(bits1 + (row[m] + 1) * pitch + (col[m] + 1) * 8) = u32x2{word[0], word[1]};
                    else
                        p.bits[image + (size_t)(r0 + row[m]) * p.W + col[m]] = ((uint64_t)word[1] << 32) | word[0];
                }
            }
        }
    };
    layer(std::integral_constant<int, 0>{});
    __syncthreads();
    layer(std::integral_constant<int, 1>{});
}

// Rows of a strip, even, or 0 where the kernel does not take the problem.
static int pair_pool_rows(int n, int h, int w) {
    if (h % 2 != 0 || w % 2 != 0 || w > 64 || (long long)h * w * 256 >= (1ll << 31)) return 0;
    int most = (kPairTiles * 32 / w) & ~1;
    if (most > h) most = h;
    const int cus = simd_count() / 4;
    auto even_rows = [&](int bands) { return ((h + bands - 1) / bands + 1) & ~1; };
    int bands = (h + most - 1) / most;
    while ((long long)n * bands < cus && even_rows(bands) > 2) ++bands;
    const int rows = even_rows(bands) < most ? even_rows(bands) : most;
    return (long long)n * ((h + rows - 1) / rows) < kMostBlocks ? rows : 0;
}

}  // namespace dab

extern "C" int dab_bconv3x3_pair_takes(int n, int h, int w) { return n > 0 && h > 0 && w > 0 && dab::pair_bands(n, h, w) > 0; }

extern "C" int dab_bconv3x3_pair(const uint64_t *x, const float *shortcut, int n, int h, int w, const uint64_t *w1, const float *a1, const float *b1,
                                 const uint64_t *w2, const float *a2, const float *b2, float *out, uint64_t *out_packed, dab_stream_t stream) {
    using namespace dab;
    const char *fn = "dab_bconv3x3_pair";
    DAB_REQUIRE(x && shortcut && w1 && a1 && b1 && w2 && a2 && b2 && out, "%s: null pointer", fn);
    DAB_REQUIRE(n > 0 && h > 0 && w > 0, "%s: non-positive dimension", fn);
    DAB_REQUIRE(out != shortcut && out_packed != x, "%s: the result must not alias the input", fn);
    DAB_REQUIRE((reinterpret_cast<uintptr_t>(x) & 7) == 0 && (reinterpret_cast<uintptr_t>(w1) & 7) == 0 && (reinterpret_cast<uintptr_t>(w2) & 7) == 0 &&
                    (reinterpret_cast<uintptr_t>(out_packed) & 7) == 0 && (reinterpret_cast<uintptr_t>(out) & 3) == 0 && (reinterpret_cast<uintptr_t>(shortcut) & 3) == 0,
                "%s: misaligned pointer", fn);
    const int bands = pair_bands(n, h, w);
    if (bands == 0) return fail(DAB_EUNSUPPORTED, "%s: %d images of %d x %d are not covered", fn, n, h, w);
    const int rows = pair_rows(n, h, w);
    BconvPairArgs p;
    p.x = x, p.shortcut = shortcut, p.out = out, p.bits = out_packed;
    p.w[0] = w1, p.w[1] = w2, p.a[0] = a1, p.a[1] = a2, p.b[0] = b1, p.b[1] = b2;
    p.H = h, p.W = w, p.rows = rows, p.bands = bands, p.above = (w + 31) / 32;
    p.div_bands = FastDiv((uint32_t)bands), p.div_w = FastDiv((uint32_t)w);
    const size_t lds = 2 * kPairFilterBytes + (size_t)(2 * rows + 6) * (w + 2) * 8;
    const dim3 grid((unsigned)(n * bands));
    if (out_packed)
        hipLaunchKernelGGL(bconv3x3_pair_kernel<true>, grid, dim3(256), lds, as_stream(stream), p);
    else
        hipLaunchKernelGGL(bconv3x3_pair_kernel<false>, grid, dim3(256), lds, as_stream(stream), p);
    DAB_LAUNCH_CHECK();
    return DAB_OK;
}

extern "C" int dab_bconv3x3_pair_pool_takes(int n, int h, int w) { return n > 0 && h > 0 && w > 0 && dab::pair_pool_rows(n, h, w) > 0; }

extern "C" int dab_bconv3x3_pair_pool(const uint64_t *x, const float *shortcut, int n, int h, int w, const uint64_t *w1, const float *a1, const float *b1,
                                      const uint64_t *w2, const float *a2, const float *b2, float *pooled, uint64_t *out_packed, dab_stream_t stream) {
    using namespace dab;
    const char *fn = "dab_bconv3x3_pair_pool";
    DAB_REQUIRE(x && shortcut && w1 && a1 && b1 && w2 && a2 && b2 && pooled && out_packed, "%s: null pointer", fn);
    DAB_REQUIRE(n > 0 && h > 0 && w > 0, "%s: non-positive dimension", fn);
    DAB_REQUIRE(pooled != shortcut && out_packed != x, "%s: the result must not alias the input", fn);
    auto at = [](const void *q) { return reinterpret_cast<uintptr_t>(q); };
    DAB_REQUIRE(((at(x) | at(w1) | at(w2) | at(out_packed)) & 7) == 0 && ((at(pooled) | at(shortcut)) & 3) == 0, "%s: misaligned pointer", fn);
    const int rows = pair_pool_rows(n, h, w);
    if (rows == 0) return fail(DAB_EUNSUPPORTED, "%s: %d images of %d x %d are not covered", fn, n, h, w);
    BconvPairPoolArgs p;
    p.x = x, p.shortcut = shortcut, p.pooled = pooled, p.bits = out_packed;
    p.w[0] = w1, p.w[1] = w2, p.a[0] = a1, p.a[1] = a2, p.b[0] = b1, p.b[1] = b2;
    p.H = h, p.W = w, p.rows = rows, p.bands = (h + rows - 1) / rows, p.image_bytes = (uint32_t)(h * w) * 256u;
    p.div_bands = FastDiv((uint32_t)p.bands), p.div_w = FastDiv((uint32_t)w), p.div_half_w = FastDiv((uint32_t)w / 2);
    const size_t lds = 2 * kPairFilterBytes + (size_t)(2 * rows + 6) * (w + 2) * 8;
    hipLaunchKernelGGL(bconv3x3_pair_pool_kernel, dim3((unsigned)(n * p.bands)), dim3(256), lds, as_stream(stream), p);
    DAB_LAUNCH_CHECK();
    return DAB_OK;
}
