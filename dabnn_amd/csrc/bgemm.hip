// Binary GEMM: C(i,j) += popcount(A(i,h) ^ B(h,j)), all operands column-major
// as in the reference (dabnn/bgemm.h:22-24,46-66,587-597):
//   A(i,h) = a[h*lda + i]   m x k words, the transposed filter bank
//   B(h,j) = b[j*ldb + h]   k x n words, one contiguous K-row per output pixel
//   C(i,j) = c[j*ldc + i]   m x n floats, i.e. NHWC output
// and the convolution over any window that shares its kernels (bgemm_core.h).
//
// Rows of the matrix instruction are pixels (columns j of C), columns are channels (rows i of C), so an accumulator
// register is 32 consecutive floats of two pixels and the output needs no transposition.
#include "bgemm_core.h"

namespace dab {

struct BitGemmArgs {
    BitGemm g;
    int units, chunks;  // units of 2 * CC dwords; of one tap
    uint32_t x_bytes;   // window form: the packed images
    uint32_t w_bytes;   // kFilterRows: the filters
    int col_tiles;
    long long row_tiles;
    long long first_tile;  // split kernel: the launch's first row tile
    FastDiv div_ow, div_oh, div_chunks, div_kw, div_col_tiles, div_row_pieces;
};

// four dwords that start at any word
typedef uint32_t u32x4u __attribute__((ext_vector_type(4), aligned(8)));

constexpr int kBeyond = (int)0x80000000;  // an offset outside every descriptor: loads return zero

// kFilterColumns goes with a plain matrix (rows of x in memory order), kFilterRows with windows of images.  A plain matrix is read
// through descriptors too, whose scalar offset walks the depth, so that a unit costs no vector address arithmetic, but for LONG
// ones: rows of 2^26 bytes, or filters of 2^31, and more.
template <FilterLayout L, bool LONG>
struct PixelRows {
    __amdgpu_buffer_rsrc_t rsrc;  // windows: the packed images
    int base, y0, x0;
    const uint64_t *row;          // plain matrix
    __device__ __forceinline__ void start(const BitGemmArgs &p, long long tile_row, int l32, int half) {
        long long r = tile_row + l32;
        r = r < p.g.rows ? r : p.g.rows - 1;
        if constexpr (L == kFilterColumns && LONG) {
            row = p.g.x + r * p.g.x_ld;
        } else if constexpr (L == kFilterColumns) {
            rsrc = make_rsrc(p.g.x + tile_row * p.g.x_ld, 0x7fffffffu);
            base = (int)(r - tile_row) * (int)(p.g.x_ld * 8) + half * 16;
        } else {
            rsrc = make_rsrc(p.g.x, p.x_bytes);
            const uint32_t t = p.div_ow.div((uint32_t)r);
            const int ox = (int)r - (int)t * p.g.OW;
            const uint32_t n = p.div_oh.div(t);
            const int oy = (int)t - (int)n * p.g.OH;
            y0 = oy * p.g.stride_h - p.g.pad_h, x0 = ox * p.g.stride_w - p.g.pad_w;
            base = (((int)n * p.g.H + y0) * p.g.W + x0) * (int)(p.g.x_ld * 8);
        }
    }
    // the lane's CC dwords of unit u (wave-uniform); zero outside the image and past the last word
    template <int CC>
    __device__ __forceinline__ void load(uint32_t (&d)[CC], const BitGemmArgs &p, int u, int half) const {
        if constexpr (L == kFilterColumns) {
            static_assert(CC == 4, "a plain matrix is walked four words at a time");
            const int word = u * 4 + half * 2;
            if constexpr (!LONG) {
                if (u * 4 + 4 <= p.g.words) {
                    load_dwords<4>(d, rsrc, base, u * 32);
                } else {
                    const u32x2 v0 = __builtin_amdgcn_raw_buffer_load_b64(rsrc, word < p.g.words ? base : kBeyond, u * 32, 0);
                    const u32x2 v1 = __builtin_amdgcn_raw_buffer_load_b64(rsrc, word + 1 < p.g.words ? base + 8 : kBeyond, u * 32, 0);
                    d[0] = v0.x, d[1] = v0.y, d[2] = v1.x, d[3] = v1.y;
                }
                return;
            }
            d[0] = d[1] = d[2] = d[3] = 0u;
            if (word + 1 < p.g.words) {
                const u32x4u v = *reinterpret_cast<const u32x4u *>(row + word);
                d[0] = v.x, d[1] = v.y, d[2] = v.z, d[3] = v.w;
            } else if (word < p.g.words) {
                const u32x2 v = *reinterpret_cast<const u32x2 *>(row + word);
                d[0] = v.x, d[1] = v.y;
            }
        } else {
            const int tap = (int)p.div_chunks.div((uint32_t)u), chunk = u - tap * p.chunks;
            const int kh = (int)p.div_kw.div((uint32_t)tap), kw = tap - kh * p.g.kw;
            const bool ok = (unsigned)(y0 + kh) < (unsigned)p.g.H && (unsigned)(x0 + kw) < (unsigned)p.g.W;
            const int off = ok ? base + (kh * p.g.W + kw) * (int)(p.g.x_ld * 8) + (chunk * 2 + half) * (CC * 4) : kBeyond;
            if constexpr (CC == 3) {
                const u32x3 v = __builtin_amdgcn_raw_buffer_load_b96(rsrc, off, 0, 0);
                d[0] = v.x, d[1] = v.y, d[2] = v.z;
            } else {
                load_dwords<CC>(d, rsrc, off);
            }
        }
    }
};

// CC dwords of unit u of filter `col` for one half of the lanes
template <int CC, FilterLayout L, bool LONG>
__device__ __forceinline__ void load_filter(uint32_t (&d)[CC], const BitGemmArgs &p, __amdgpu_buffer_rsrc_t rw, int col, int u, int half) {
    if constexpr (L == kFilterColumns && !LONG) {
        const int word = u * 4 + half * 2, ld = (int)p.g.w_ld * 8, off = col < p.g.cols ? col * 8 + half * 2 * ld : kBeyond;
        const bool whole = u * 4 + 4 <= p.g.words;
        const u32x2 v0 = __builtin_amdgcn_raw_buffer_load_b64(rw, whole || word < p.g.words ? off : kBeyond, u * 4 * ld, 0);
        const u32x2 v1 = __builtin_amdgcn_raw_buffer_load_b64(rw, whole || word + 1 < p.g.words ? off : kBeyond, u * 4 * ld + ld, 0);
        d[0] = v0.x, d[1] = v0.y, d[2] = v1.x, d[3] = v1.y;
    } else if constexpr (L == kFilterColumns) {
        const int word = u * 4 + half * 2;
        const uint64_t *src = p.g.w + (long long)word * p.g.w_ld + col;
        const bool ok = col < p.g.cols;
        const uint64_t v0 = ok && word < p.g.words ? src[0] : 0ull, v1 = ok && word + 1 < p.g.words ? src[p.g.w_ld] : 0ull;
        d[0] = (uint32_t)v0, d[1] = (uint32_t)(v0 >> 32), d[2] = (uint32_t)v1, d[3] = (uint32_t)(v1 >> 32);
    } else {
        const int off = col < p.g.cols && u < p.units ? col * (int)(p.g.w_ld * 8) + (u * 2 + half) * (CC * 4) : kBeyond;
        if constexpr (CC == 3) {
            const u32x3 v = __builtin_amdgcn_raw_buffer_load_b96(rw, off, 0, 0);
            d[0] = v.x, d[1] = v.y, d[2] = v.z;
        } else {
            load_dwords<CC>(d, rw, off);
        }
    }
}
// Set bits of the word that pads filter `col` to 128 bits
__device__ __forceinline__ uint32_t extra_bits(const BitGemmArgs &p, __amdgpu_buffer_rsrc_t rw, int col) {
    const u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(rw, col < p.g.cols ? (col * (int)p.g.w_ld + p.g.words) * 8 : kBeyond, 0, 0);
    return __popc(v.x) + __popc(v.y);
}

// The output (or a tensor laid out like it) from a tile's first pixel to the tensor's end: offsets past it load zero and
// store nothing.  For rows below 64 MB (kLongRow): the offsets of a tile's 32 rows stay below 2^31.  Longer rows of a plain
// matrix (LONG) are addressed by pointer, element by element under a test of row and channel.
constexpr long long kLongRow = 1ll << 24;
__device__ __forceinline__ __amdgpu_buffer_rsrc_t tile_rsrc(const float *t, const BitGemmArgs &p, long long row0) {
    const long long left = ((p.g.rows - 1 - row0) * p.g.out_ld + p.g.cols) * 4;
    return make_rsrc(t + row0 * p.g.out_ld, left < 0x7fffffff ? (uint32_t)left : 0x7fffffffu);
}

enum Epilogue { kStoreCounts, kAddCounts, kAffine, kAffineSign };

// Few tiles, or a depth that does not fit LDS as filters: a block is one tile of 32 pixels x 32 * NT channels, its four
// (eight) waves take every fourth (eighth) unit of the depth each and load their operands straight from memory, kUnitsAtOnce units at a
// time; the partial sums meet in LDS.  Both operands +-1 (fp4_core.h).  Bound by their expansion: m512 k72 n3136, accumulating, 7.9 us.
// (Two units asked for while two are multiplied: 8.0 there, 900 x 1000 x 50 6.3 instead of 5.8, 7 x 47 x 47 x 192 -> 120, 3 x 3, 5.5 instead of 5.1.)
// SHALLOW: up to kUnitsAtOnce units a wave, without the loop, and what C holds is asked for before them: behind them its wait shows in
// launches this short (189 x 26 x 13, accumulating, 2.52 us instead of 2.75, 300 x 300 x 40 3.03 instead of 3.19), while deeper ones begin with the
// units (m512 k72 n3136 8.4 the other way round; 1 x 14 x 14 x 256 -> 256, 5 x 5, 3.60 instead of 3.69) -- but for windows with 64 channels a
// block, whose loop is a shorter one without units in front of it (3 x 49 x 49 x 256 -> 208, 5 x 5, 9.0 us instead of 9.4).
constexpr int kUnitsAtOnce = 3;
template <int CC, FilterLayout L, int E, int NT, int WAVES, bool LONG, bool SHALLOW = false>
__global__ __launch_bounds__(64 * WAVES, 4) void bit_gemm_split_kernel(const BitGemmArgs p) {
    constexpr int CH = 32 * NT, LD = CH + 1;
    __shared__ float part[WAVES][32 * LD];
    const int tid = threadIdx.x, lane = tid & 63, half = lane >> 5, l32 = lane & 31;
    const int wib = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t block_tile = p.div_col_tiles.div(blockIdx.x);
    const int ch0 = (int)(blockIdx.x - block_tile * p.col_tiles) * CH;
    const long long row0 = (block_tile + p.first_tile) * 32;
    const __amdgpu_buffer_rsrc_t rw = make_rsrc(p.g.w, L == kFilterRows ? p.w_bytes : 0x7fffffffu);
    PixelRows<L, LONG> px;
    px.start(p, row0, l32, half);

    // this thread's outputs: channel tid % CH of pixels tid / CH + i * (256 / CH)
    constexpr int RPI = 64 * WAVES / CH, ROWS = 32 / RPI;
    const int ch = ch0 + tid % CH, r0 = tid / CH;
    const bool ch_ok = ch < p.g.cols;
    float old[ROWS], ea = 0.f, eb = 0.f;
    uint32_t extra = 0;
    if (L == kFilterRows && p.g.extra_word) extra = extra_bits(p, rw, ch);
    if (E == kAffine || E == kAffineSign)
        if (ch_ok) ea = p.g.a[ch], eb = p.g.b[ch];
    const int out_off = ch_ok ? (r0 * (int)p.g.out_ld + ch) * 4 : kBeyond, out_step = RPI * (int)p.g.out_ld * 4;
    auto element = [&](int i) { return p.g.out + (row0 + r0 + i * RPI) * p.g.out_ld + ch; };  // LONG: output i
    uint32_t a[kUnitsAtOnce][CC], w[kUnitsAtOnce][NT][CC];
    auto fetch = [&](int u0) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < kUnitsAtOnce; ++i)
            if (u0 + WAVES * i < p.units) {
                px.load(a[i], p, u0 + WAVES * i, half);
#pragma unroll
                for (int n = 0; n < NT; ++n) load_filter<CC, L, LONG>(w[i][n], p, rw, ch0 + n * 32 + l32, u0 + WAVES * i, half);
            }
    };
    constexpr bool kFirst = !SHALLOW && (L == kFilterColumns || NT == 1);
    if constexpr (kFirst) fetch(wib);
    const float *second = E == kAddCounts ? p.g.out : p.g.shortcut;
    if constexpr (LONG) {
        static_assert(L == kFilterColumns, "a plain matrix");
        if constexpr (E == kAddCounts) {
#pragma unroll
            for (int i = 0; i < ROWS; ++i) old[i] = ch_ok && row0 + r0 + i * RPI < p.g.rows ? *element(i) : 0.f;
        }
    } else if (E != kStoreCounts && second != nullptr) {
        const __amdgpu_buffer_rsrc_t rs = tile_rsrc(second, p, row0);
#pragma unroll
        for (int i = 0; i < ROWS; ++i) old[i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, out_off, i * out_step, 0));
    }
    if constexpr (SHALLOW) fetch(wib);
    f32x16m acc[NT];
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[n][v] = 0.f;
    auto multiply = [&](int u0) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < kUnitsAtOnce; ++i)
            if (u0 + WAVES * i < p.units) {
#pragma unroll
                for (int c = 0; c < CC; ++c) {
                    const i32x8 av = bitspm1(a[i][c]);
#pragma unroll
                    for (int n = 0; n < NT; ++n) mfma_fp4<32>(acc[n], av, bitspm1(w[i][n][c]));
                }
            }
    };
    if constexpr (SHALLOW) {
        multiply(wib);
    } else {
        for (int u0 = wib; u0 < p.units; u0 += WAVES * kUnitsAtOnce) {
            if (!kFirst || u0 != wib) fetch(u0);
            multiply(u0);
        }
    }
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int v = 0; v < 16; ++v) part[wib][fp4_row<32>(half, v) * LD + n * 32 + l32] = acc[n][v];
    __syncthreads();

    const __amdgpu_buffer_rsrc_t ro = tile_rsrc(p.g.out, p, row0);
    const float half_depth = (float)(p.units * CC) * 32.f;  // of the units; words past the last are zero on both sides and equal
#pragma unroll
    for (int i = 0; i < ROWS; ++i) {
        const int row = r0 + i * RPI;
        const long long r = row0 + row;
        const int o = row * LD + tid % CH;
        float sum = (part[0][o] + part[1][o]) + (part[2][o] + part[3][o]);
        if constexpr (WAVES == 8) sum = sum + ((part[4][o] + part[5][o]) + (part[6][o] + part[7][o]));
        float v = half_depth - 0.5f * sum + (float)extra;
        if constexpr (E == kAddCounts) v = old[i] + v;
        if constexpr (E == kAffine || E == kAffineSign) {
#pragma clang fp contract(off)
            v = ea * v;
            v = v + eb;
            if (p.g.shortcut) v = v + old[i];
        }
        const bool ok = ch_ok && r < p.g.rows;
        if constexpr (LONG) {
            if (ok) store_through(element(i), v);
        } else {
            __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v), ro, out_off, i * out_step, kStoreThrough);
        }
        if constexpr (E == kAffineSign) {
            const uint64_t mask = __ballot(v > 0.f);
            if (ok && (tid & 31) == 0)
                p.g.bits[r * p.g.bits_ld + (ch >> 5)] = (lane & 32) ? (uint32_t)(mask >> 32) : (uint32_t)mask;
        }
    }
}

// Many tiles, or one to three units of depth: a block keeps the filters of 32 * NT channels in LDS as bits, in the order its lanes read them, and its
// four waves walk over tiles of 32 pixels, four units of their pixels ahead of the multiplication.
template <int CC, FilterLayout L, int E, int NT, bool LONG>
__global__ __launch_bounds__(256, NT == 2 ? 3 : 4) void bit_gemm_stream_kernel(const BitGemmArgs p) {
    constexpr int CH = 32 * NT, SLOT = CC == 3 ? 16 : CC * 4;  // bytes of a (unit, channel, half)
    extern __shared__ __attribute__((aligned(16))) unsigned char filters[];
    __shared__ uint32_t pop[CH];  // set bits per filter
    const int tid = threadIdx.x, lane = tid & 63, half = lane >> 5, l32 = lane & 31;
    const int wib = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int group = (int)p.div_col_tiles.div(blockIdx.x), groups = (int)p.div_col_tiles.div(gridDim.x);
    const int ch0 = ((int)blockIdx.x - group * p.col_tiles) * CH;
    const __amdgpu_buffer_rsrc_t rw = make_rsrc(p.g.w, L == kFilterRows ? p.w_bytes : 0x7fffffffu);
    if (tid < CH) pop[tid] = L == kFilterRows && p.g.extra_word ? extra_bits(p, rw, ch0 + tid) : 0u;
    __syncthreads();
    constexpr int kBatch = 3;  // pieces a thread asks for before it puts the first of them away
    const int n_pieces = p.units * CH * 2;
    for (int s0 = tid; s0 < n_pieces; s0 += 256 * kBatch) {
        uint32_t d[kBatch][CC];
        int slot[kBatch], chan[kBatch];
#pragma unroll
        for (int j = 0; j < kBatch; ++j) {
            // consecutive threads take consecutive channels of column-major filters, consecutive units of filter rows
            const int s = s0 + j * 256;
            int u, c, h;
            if constexpr (L == kFilterColumns) {
                // (the same unit in all lanes of a wave, whose 64 pieces never straddle 2 * CH)
                c = s % CH, h = (s / CH) & 1, u = __builtin_amdgcn_readfirstlane(s / (2 * CH));
            } else {
                c = (int)p.div_row_pieces.div((uint32_t)s);
                const int r = s - c * p.units * 2;
                u = r >> 1, h = r & 1;
            }
            chan[j] = c, slot[j] = (u * CH + c) * 2 + h;
            if (s < n_pieces) load_filter<CC, L, LONG>(d[j], p, rw, ch0 + c, u, h);
        }
#pragma unroll
        for (int j = 0; j < kBatch; ++j) {
            if (s0 + j * 256 < n_pieces) {
                uint32_t *dst = reinterpret_cast<uint32_t *>(filters + slot[j] * SLOT);
                uint32_t set = 0;
#pragma unroll
                for (int i = 0; i < CC; ++i) dst[i] = d[j][i], set += __popc(d[j][i]);
                atomicAdd(&pop[chan[j]], set);
            }
        }
    }
    __syncthreads();
    float init[NT], ea[NT], eb[NT];
    int out_off[NT];
    const int row_bytes = (int)p.g.out_ld * 4;
#pragma unroll
    for (int n = 0; n < NT; ++n) {
        const int ch = ch0 + n * 32 + l32;
        out_off[n] = ch < p.g.cols ? half * 4 * row_bytes + ch * 4 : kBeyond;
        init[n] = (float)pop[n * 32 + l32];
        ea[n] = 0.f, eb[n] = 0.f;
        if (E == kAffine || E == kAffineSign)
            if (ch < p.g.cols) ea[n] = p.g.a[ch], eb[n] = p.g.b[ch];
    }
    const unsigned char *mine = filters + (l32 * 2 + half) * SLOT;

    for (long long tile = (long long)group * 4 + wib; tile < p.row_tiles; tile += (long long)groups * 4) {
        const long long row0 = tile * 32;
        PixelRows<L, LONG> px;
        px.start(p, row0, l32, half);
        uint32_t a[4][CC];
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (i < p.units) px.load(a[i], p, i, half);
        float old[NT][16];
        // LONG: output v of channel group n, and whether the matrix has it
        auto element = [&](int n, int v) { return p.g.out + (row0 + fp4_row<32>(half, v)) * p.g.out_ld + ch0 + n * 32 + l32; };
        auto inside = [&](int n, int v) { return ch0 + n * 32 + l32 < p.g.cols && row0 + fp4_row<32>(half, v) < p.g.rows; };
        if constexpr (LONG) {
            static_assert(L == kFilterColumns, "a plain matrix");
            if constexpr (E == kAddCounts) {
#pragma unroll
                for (int v = 0; v < 16; ++v)
#pragma unroll
                    for (int n = 0; n < NT; ++n) old[n][v] = inside(n, v) ? *element(n, v) : 0.f;
            }
        } else if constexpr (E != kStoreCounts) {
            const float *second = E == kAddCounts ? p.g.out : p.g.shortcut;
            if (second != nullptr) {
                const __amdgpu_buffer_rsrc_t rs = tile_rsrc(second, p, row0);
#pragma unroll
                for (int v = 0; v < 16; ++v)
#pragma unroll
                    for (int n = 0; n < NT; ++n)
                        old[n][v] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, out_off[n], fp4_row<32>(0, v) * row_bytes, 0));
            }
        }
        f32x16m acc[NT];
#pragma unroll
        for (int n = 0; n < NT; ++n)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[n][v] = init[n];
        for (int u0 = 0; u0 < p.units; u0 += 4) {
            uint32_t next[4][CC];
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (u0 + 4 + i < p.units) px.load(next[i], p, u0 + 4 + i, half);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if (u0 + i < p.units) {
                    const unsigned char *fu = mine + (u0 + i) * (CH * 2 * SLOT);
                    uint32_t w[NT][CC];
#pragma unroll
                    for (int n = 0; n < NT; ++n) {
                        if constexpr (CC == 3) {
                            const u32x4 v = *reinterpret_cast<const u32x4 *>(fu + n * 64 * SLOT);
                            w[n][0] = v.x, w[n][1] = v.y, w[n][2] = v.z;
                        } else {
                            lds_dwords<CC>(w[n], fu + n * 64 * SLOT);
                        }
                    }
#pragma unroll
                    for (int c = 0; c < CC; ++c) {
                        const i32x8 av = bits01(a[i][c]);
#pragma unroll
                        for (int n = 0; n < NT; ++n) mfma_fp4<32>(acc[n], av, bitspm(w[n][c]));
                    }
                }
            }
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int c = 0; c < CC; ++c) a[i][c] = next[i][c];
        }
        const __amdgpu_buffer_rsrc_t ro = tile_rsrc(p.g.out, p, row0);
        uint32_t word[NT];
#pragma unroll
        for (int n = 0; n < NT; ++n) word[n] = 0;
#pragma unroll
        for (int v = 0; v < 16; ++v) {
#pragma unroll
            for (int n = 0; n < NT; ++n) {
                float res = acc[n][v];
                if constexpr (E == kAddCounts) res = old[n][v] + res;
                if constexpr (E == kAffine || E == kAffineSign) {
#pragma clang fp contract(off)
                    res = ea[n] * res;
                    res = res + eb[n];
                    if (p.g.shortcut) res = res + old[n][v];
                }
                if constexpr (LONG) {
                    if (inside(n, v)) store_through(element(n, v), res);
                } else {
                    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, res), ro, out_off[n], fp4_row<32>(0, v) * row_bytes, kStoreThrough);
                }
                if constexpr (E == kAffineSign) {
                    const uint64_t mask = __ballot(res > 0.f);
                    word[n] = dab_writelane((uint32_t)mask, fp4_row<32>(0, v), word[n]);
                    word[n] = dab_writelane((uint32_t)(mask >> 32), fp4_row<32>(1, v), word[n]);
                }
            }
        }
        if constexpr (E == kAffineSign) {
            const long long r = row0 + l32;
            if (half == 0 && r < p.g.rows) {
#pragma unroll
                for (int n = 0; n < NT; ++n)
                    if (ch0 + n * 32 < p.g.cols) p.g.bits[r * p.g.bits_ld + ch0 / 32 + n] = word[n];
            }
        }
    }
}

// A shallow and small product: a lane per channel and a wave per four pixels, whose words are the same for all lanes, and
// xor and popcount of them; nothing is staged and no wave waits for another.  Bound by the launch: 1.9 to 2.8 us, the walking
// kernel with its filters in LDS 2.4 to 3.6 (m 256, n 4, k 1 accumulated 2.1 against 2.9; n 64, k 8 2.5 against 3.3).
constexpr int kDirectPixels = 4;
template <int E>
__global__ __launch_bounds__(256) void bit_gemm_direct_kernel(const BitGemmArgs p) {
    const int lane = threadIdx.x & 63, wib = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t block_tile = p.div_col_tiles.div(blockIdx.x);
    const int ch = (int)(blockIdx.x - block_tile * p.col_tiles) * 64 + lane;
    const long long row0 = ((long long)block_tile * 4 + wib) * kDirectPixels;
    if (row0 >= p.g.rows) return;
    const int col = ch < p.g.cols ? ch : p.g.cols - 1;
    float old[kDirectPixels];
#pragma unroll
    for (int i = 0; i < kDirectPixels; ++i) {
        old[i] = 0.f;
        if constexpr (E == kAddCounts)
            if (row0 + i < p.g.rows) old[i] = p.g.out[(row0 + i) * p.g.out_ld + col];
    }
    uint32_t count[kDirectPixels] = {};
#pragma unroll 4
    for (int h = 0; h < p.g.words; ++h) {
        const uint64_t w = p.g.w[h * p.g.w_ld + col];
#pragma unroll
        for (int i = 0; i < kDirectPixels; ++i) {
            const long long r = row0 + i < p.g.rows ? row0 + i : p.g.rows - 1;
            count[i] += __popcll(w ^ p.g.x[r * p.g.x_ld + h]);
        }
    }
#pragma unroll
    for (int i = 0; i < kDirectPixels; ++i)
        if (ch < p.g.cols && row0 + i < p.g.rows) p.g.out[(row0 + i) * p.g.out_ld + ch] = E == kAddCounts ? old[i] + (float)count[i] : (float)count[i];
}

// LDS that a block's filters may take: two blocks of a CU
constexpr long long kFilterLdsBytes = 72 * 1024;

template <int CC, FilterLayout L, int E, bool LONG = false>
static int launch_bit_gemm(const char *fn, BitGemmArgs &p, hipStream_t s) {
    p.row_tiles = (p.g.rows + 31) / 32;
    const int tiles32 = (p.g.cols + 31) / 32;
    const long long pieces = p.row_tiles * tiles32;
    const long long per_channel = (long long)p.units * 2 * (CC == 3 ? 16 : CC * 4);
    // The walking kernel where its filters fit and its waves find tiles for every SIMD; also for one to three units of
    // depth, which are no work for four waves.
    struct Walk {
        int channels, col_tiles;
        size_t lds;
        long long groups;
        long long rounds;  // tiles that the waves of the fullest CU walk
    };
    auto fits = [&](int ch) { return per_channel * ch <= kFilterLdsBytes; };
    auto walk = [&](int ch) {
        Walk w;
        w.channels = ch, w.col_tiles = (p.g.cols + ch - 1) / ch;
        w.lds = (size_t)(per_channel * ch);
        const int cus = simd_count() / 4, by_registers = ch == 64 ? 3 : 4, by_lds = (int)(160 * 1024 / (w.lds + 1024));
        const long long most = (long long)cus * (by_lds < by_registers ? by_lds : by_registers) / w.col_tiles, want = (p.row_tiles + 3) / 4;
        w.groups = want < most ? want : most < 1 ? 1 : most;
        // Equal shares, on as few blocks as that takes -- but for windows whose fullest CU would then walk a sixteenth more tiles than the
        // average one, where all resident blocks share them out: 64 x 28 x 28 x 192 -> 192, 3 x 3, 17.4 -> 15.2 us (12 tiles against 9.2),
        // 50 x 30 x 30 x 256 -> 256, 5 x 5, 49 -> 44 (12 / 11), 256 x 32 x 32 x 128 -> 64 into slices 23.3 -> 21.3 (9 / 8); with 128 images,
        // 4 tiles either way, 13.5 -> 15.  40 random layers 1.05 times as fast, 0.98 to 1.2; with one to three words a filter, bound by
        // the stores, 0.96 to 1.  (Plain matrices 0.9 to 1.2 times as fast: they keep equal shares.)
        const long long per_wave = (p.row_tiles + w.groups * 4 - 1) / (w.groups * 4), equal = (p.row_tiles + 4 * per_wave - 1) / (4 * per_wave);
        w.rounds = (equal * w.col_tiles + cus - 1) / cus * per_wave;
        if (L == kFilterColumns || p.g.words < 4 || w.rounds * 64 * cus < 17 * p.row_tiles * w.col_tiles) w.groups = equal;
        return w;
    };
    // 64 channels a wave for plain matrices (m128 k18 n50176: 12.6 us against 16.4).  For windows, whose lanes spend more on addresses
    // than on filters, with 33 to 64 channels, so that every window is fetched once, from 4096 pieces on (2048 with all 64: 582 x 8 x 8 x
    // 128 -> 40 7.8 us with 32 against 8.9).  A tile of 64 takes 1.5 to 1.9 times as long as one of 32, so not where the fullest CU walks
    // two thirds as many of them (45 such layers: 0.95).  570 random layers: into slices of their output 1.17 times as fast (0.93 to 1.8),
    // into an output of their own 1.06 (30 words a filter and more 0.94 to 1.3; fewer, bound by the stores, 0.89 to 1.6).  3x3 over 128
    // channels -> 64, into slices of 256, 131 072 pixels: 18.5 -> 15.3 us.  With more channels 32 (100 x 25 x 25 x 192 -> 472, 5 x 5, stride 2:
    // 34 us against 43).
    const bool wide = L == kFilterColumns ? p.g.cols > 32 && pieces >= 2048 : p.g.cols > 32 && p.g.cols <= 64 && pieces >= (p.g.cols == 64 ? 2048 : 4096);
    // Where 64 filters do not fit (above 144 words, or 108 in chunks of three), windows leave the walking kernel for the one that splits the
    // depth, 64 channels a block: 23 x 56 x 56 x 384 -> 40, 5x5, 50 us with 32 channels a wave, 32 split; 41 x 56 x 56 x 384 -> 64, 6x6, 113 and
    // 85.  Not in chunks of one word or two from 8000 pieces on, but for few channels and pieces (82 x 56 x 56 x 320 -> 64, 6x6, 269 and 375;
    // -> 40 270 and 256, 459 x 33 x 33 458 and 500).
    const bool split = wide && !fits(64) && (L == kFilterColumns || CC >= 3 || pieces < 8000 || (p.g.cols <= 40 && pieces < 20000));
    if ((pieces >= 2048 || p.units < 4) && fits(32) && !split) {
        Walk w = walk(32);
        if (wide && fits(64)) {
            const Walk by64 = walk(64);
            if (L == kFilterColumns || 2 * w.rounds > 3 * by64.rounds) w = by64;
        }
        p.col_tiles = w.col_tiles;
        p.div_col_tiles = FastDiv((uint32_t)p.col_tiles);
        const size_t lds = w.lds;
        const long long groups = w.groups;
        auto launch = [&](auto nt) {
            constexpr auto kernel = bit_gemm_stream_kernel<CC, L, E, decltype(nt)::value, LONG>;
            if (lds > 64 * 1024) {
                const int rc = allow_dynamic_lds<kernel>(fn, kFilterLdsBytes);
                if (rc != DAB_OK) return rc;
            }
            hipLaunchKernelGGL(kernel, dim3((unsigned)(groups * p.col_tiles)), dim3(256), lds, s, p);
            return DAB_OK;
        };
        int rc = DAB_OK;
        rc = w.channels == 64 ? launch(std::integral_constant<int, 2>{}) : launch(std::integral_constant<int, 1>{});
        if (rc != DAB_OK) return rc;
    } else {
        const int split_ch = p.g.cols > 32 && pieces >= 1024 ? 64 : 32;
        p.col_tiles = (p.g.cols + split_ch - 1) / split_ch;
        p.div_col_tiles = FastDiv((uint32_t)p.col_tiles);
        const long long blocks = p.row_tiles * p.col_tiles;
        if (blocks >= (1ll << 31)) return fail(DAB_EUNSUPPORTED, "%s: too many work units", fn);
        // Eight waves where they have depth for it and a CU no more than two blocks: 200 x 1000 x 150 5.5 -> 5.0 us, 300 x 300 x 100 4.5 ->
        // 4.2, 1 x 14 x 14 x 256 -> 256, 5 x 5, 4.1 -> 3.7, at 8 images 5.3 -> 5.1; 64 x 12000 x 50 (750 blocks) 5.0 -> 5.1, 60 x 14 x 14 x
        // 256 -> 40, 5 x 5 (736) 6.1 -> 6.3, 4 x 28 x 28 x 192 -> 192, 3 x 3 (nine units) 4.1 -> 4.2.
        const bool eight = p.units >= 12 && blocks <= simd_count() / 2;
        const long long most = kMostBlocks / p.col_tiles > 1 ? kMostBlocks / p.col_tiles : 1;  // row tiles of a launch
        for (p.first_tile = 0; p.first_tile < p.row_tiles; p.first_tile += most) {
            const long long tiles = p.row_tiles - p.first_tile < most ? p.row_tiles - p.first_tile : most;
            const dim3 grid((unsigned)(tiles * p.col_tiles));
            if (split_ch == 64)
                hipLaunchKernelGGL((bit_gemm_split_kernel<CC, L, E, 2, 4, LONG>), grid, dim3(256), 0, s, p);
            else if (eight)
                hipLaunchKernelGGL((bit_gemm_split_kernel<CC, L, E, 1, 8, LONG>), grid, dim3(512), 0, s, p);
            else if (!LONG && p.units <= 4 * kUnitsAtOnce)
                hipLaunchKernelGGL((bit_gemm_split_kernel<CC, L, E, 1, 4, LONG, !LONG>), grid, dim3(256), 0, s, p);
            else
                hipLaunchKernelGGL((bit_gemm_split_kernel<CC, L, E, 1, 4, LONG>), grid, dim3(256), 0, s, p);
        }
    }
    DAB_LAUNCH_CHECK();
    return DAB_OK;
}

bool bit_gemm_takes_images(long long image_words, long long filter_words, long long rows, int cols) {
    return image_words * 8 < (1ll << 31) && filter_words * 8 < (1ll << 31) && rows < (1ll << 31) - 64 && cols < (1 << 22);
}

// The direct kernel: plain matrices of up to three units of depth (16 words: 2.5 us against the split kernel's 2.1) and 2048
// waves (512 x 1024 x 12: 3.46 against 3.54; twice that, 256 x 4096: 3.2 to 4.8 us against 3.2 to 3.9).
static bool takes_direct(const BitGemm &g) {
    return g.words <= 12 && (g.rows + kDirectPixels - 1) / kDirectPixels * ((g.cols + 63) / 64) <= 2048;
}
template <int E>
static int launch_direct(BitGemmArgs &p, hipStream_t s) {
    p.col_tiles = (p.g.cols + 63) / 64;
    p.div_col_tiles = FastDiv((uint32_t)p.col_tiles);
    const long long blocks = (p.g.rows + 4 * kDirectPixels - 1) / (4 * kDirectPixels) * p.col_tiles;
    hipLaunchKernelGGL(bit_gemm_direct_kernel<E>, dim3((unsigned)blocks), dim3(256), 0, s, p);
    DAB_LAUNCH_CHECK();
    return DAB_OK;
}

// Columns of one launch: channel numbers stay well inside an int, and 32 columns a block make fewer than 2^32 threads.
constexpr long long kMostColumns = 1ll << 28;

int bit_gemm(const char *fn, const BitGemm &g, FilterLayout layout, hipStream_t stream) {
    if (layout == kFilterRows && g.out_ld >= kLongRow) {
        if (g.rows > 1) return fail(DAB_EUNSUPPORTED, "%s: output rows too long", fn);
        BitGemm one = g;
        one.out_ld = g.cols;
        return bit_gemm(fn, one, layout, stream);
    }
    if (layout == kFilterColumns && g.cols > kMostColumns) {
        BitGemm part = g;
        for (long long c = 0; c < g.cols; c += kMostColumns) {
            part.cols = (int)(g.cols - c < kMostColumns ? g.cols - c : kMostColumns);
            part.w = g.w + c, part.out = g.out + c;
            const int rc = bit_gemm(fn, part, layout, stream);
            if (rc != DAB_OK) return rc;
        }
        return DAB_OK;
    }
    BitGemmArgs p = {};
    p.g = g;
    if (layout == kFilterColumns && takes_direct(g)) return g.accumulate ? launch_direct<kAddCounts>(p, stream) : launch_direct<kStoreCounts>(p, stream);
    if (layout == kFilterColumns) {
        p.units = (g.words + 3) / 4, p.chunks = p.units;
        if (g.out_ld >= kLongRow || g.x_ld * 8 >= (1ll << 26) || g.words * g.w_ld * 8 >= (1ll << 31))
            return g.accumulate ? launch_bit_gemm<4, kFilterColumns, kAddCounts, true>(fn, p, stream)
                                : launch_bit_gemm<4, kFilterColumns, kStoreCounts, true>(fn, p, stream);
        return g.accumulate ? launch_bit_gemm<4, kFilterColumns, kAddCounts>(fn, p, stream)
                            : launch_bit_gemm<4, kFilterColumns, kStoreCounts>(fn, p, stream);
    }
    const int cw = g.tap_words, cc = cw % 4 == 0 ? 4 : cw % 3 == 0 ? 3 : cw % 2 == 0 ? 2 : 1;
    p.chunks = cw / cc;
    p.units = g.words / cc;
    p.x_bytes = (uint32_t)(((g.rows / ((long long)g.OH * g.OW)) * g.H * g.W) * g.x_ld * 8);
    p.w_bytes = (uint32_t)(g.cols * g.w_ld * 8);
    p.div_ow = FastDiv((uint32_t)g.OW), p.div_oh = FastDiv((uint32_t)g.OH);
    p.div_chunks = FastDiv((uint32_t)p.chunks), p.div_kw = FastDiv((uint32_t)g.kw);
    p.div_row_pieces = FastDiv((uint32_t)(2 * p.units));
    auto with_epilogue = [&](auto cc_) {
        constexpr int CC = decltype(cc_)::value;
        if (g.bits) return launch_bit_gemm<CC, kFilterRows, kAffineSign>(fn, p, stream);
        if (g.a) return launch_bit_gemm<CC, kFilterRows, kAffine>(fn, p, stream);
        return launch_bit_gemm<CC, kFilterRows, kStoreCounts>(fn, p, stream);
    };
    switch (cc) {
        case 4: return with_epilogue(std::integral_constant<int, 4>{});
        case 3: return with_epilogue(std::integral_constant<int, 3>{});
        case 2: return with_epilogue(std::integral_constant<int, 2>{});
        default: return with_epilogue(std::integral_constant<int, 1>{});
    }
}

constexpr int kMaxCount = (1 << 23) - 1;  // exact in fp32, twice over

}  // namespace dab

static int bgemm_impl(int m, int n, int k, const uint64_t *a, int lda, const uint64_t *b, int ldb, float *c, int ldc,
                      bool overwrite, dab_stream_t stream) {
    using namespace dab;
    DAB_REQUIRE(a && b && c, "dab_bgemm: null pointer");
    DAB_REQUIRE(m > 0 && n > 0 && k > 0, "dab_bgemm: m %d n %d k %d", m, n, k);
    DAB_REQUIRE(lda >= m && ldb >= k && ldc >= m, "dab_bgemm: leading dimension smaller than the matrix (lda %d ldb %d ldc %d)",
                lda, ldb, ldc);
    DAB_REQUIRE((reinterpret_cast<uintptr_t>(a) & 7) == 0 && (reinterpret_cast<uintptr_t>(b) & 7) == 0 &&
                    (reinterpret_cast<uintptr_t>(c) & 3) == 0,
                "dab_bgemm: misaligned pointer");
    if ((long long)k * 64 > kMaxCount) return fail(DAB_EUNSUPPORTED, "dab_bgemm: k %d words exceeds the exact-count range", k);
    if ((long long)ldb * 8 * 8 >= (1ll << 32)) return fail(DAB_EUNSUPPORTED, "dab_bgemm: ldb too large");
    BitGemm g = {};
    g.x = b, g.w = a, g.out = c;
    g.rows = n, g.cols = m;
    g.x_ld = ldb, g.w_ld = lda, g.out_ld = ldc;
    g.words = k, g.tap_words = k;
    g.accumulate = !overwrite;
    return bit_gemm("dab_bgemm", g, kFilterColumns, as_stream(stream));
}

extern "C" int dab_bgemm(int m, int n, int k, const uint64_t *a, int lda, const uint64_t *b, int ldb, float *c, int ldc,
                         dab_stream_t stream) {
    return bgemm_impl(m, n, k, a, lda, b, ldb, c, ldc, false, stream);
}

extern "C" int dab_bgemm_overwrite(int m, int n, int k, const uint64_t *a, int lda, const uint64_t *b, int ldb, float *c,
                                   int ldc, dab_stream_t stream) {
    return bgemm_impl(m, n, k, a, lda, b, ldb, c, ldc, true, stream);
}
