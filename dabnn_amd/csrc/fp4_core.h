// Sign bits on the matrix cores.
//
// There is no 1-bit matrix instruction, but v_mfma_f32_32x32x64_f8f6f4 / 16x16x128 multiply 4-bit floats (e2m1: sign,
// two exponent bits, one mantissa bit; 0, 0.5, 1, 1.5, 2, 3, 4, 6) into fp32 accumulators at four times the bf16 rate:
// 65 536 products of bits per 32 x 32 x 64 instruction, issued every 32-40 cycles, where v_xor_b32 + v_bcnt_u32_b32
// takes 6.4 cycles for 2 048.  Whole numbers up to 2^24 are exact in the accumulators, so a dot product of bits is the
// integer it should be.
//
// A lane of the instruction holds 32 consecutive depths of one row or column: four dwords of eight 4-bit floats, made
// from one dword of packed bits in registers.  Which bit lands in which depth does not matter as long as both operands
// use the same order, so dword j takes bits j, j + 4, j + 8, ... -- the bits of `x & (0x11111111 << j)` as they lie.
// A single bit at position 0, 1 or 2 of its nibble is the value 0.5, 1 or 2; position 3 is the sign, so that dword is
// shifted down.
//   bits01:  bit -> {0, m}, m = 0.5, 1, 2, 0.5 in the four dwords.  5 vector instructions.
//   bitspm:  bit -> {+m', -m'}, m' = 2, 1, 0.5, 2: every product with a bits01 value is 0 or +-1.  7 instructions.
//   bitspm1: bit -> {+1, -1} in all dwords, for products of two such operands.  7 instructions.
// With x as bits01 and w as bitspm, popcount(w) + sum x * (+-1 for w = 0 / 1) is the number of places where x and w
// differ; with both as bitspm1 it is (K - sum) / 2.  A zero word in both operands (the reference's padding word,
// dabnn/pad.h:12) counts no difference either way.
#pragma once

#include "common.h"

namespace dab {

typedef int i32x8 __attribute__((ext_vector_type(8)));  // the instruction's operand; 4-bit floats use the first four
typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4m __attribute__((ext_vector_type(4)));
typedef float f32x16m __attribute__((ext_vector_type(16)));

__device__ __forceinline__ i32x8 bits01(uint32_t x) {
    i32x8 r = {0, 0, 0, 0, 0, 0, 0, 0};
    r[0] = x & 0x11111111u, r[1] = x & 0x22222222u, r[2] = x & 0x44444444u, r[3] = (x >> 3) & 0x11111111u;
    return r;
}
// (x & y) | z in one instruction.  These expansions are what bounds the deep convolutions: vector instructions and
// fp4 matrix instructions of a SIMD do not overlap here, and each of the former costs 4 to 5 cycles with 2 or 3 waves.
__device__ __forceinline__ uint32_t and_or(uint32_t x, uint32_t y, uint32_t z) { return __builtin_amdgcn_bitop3_b32(x, y, z, 0xEA); }
__device__ __forceinline__ i32x8 bitspm(uint32_t w) {
    i32x8 r = {0, 0, 0, 0, 0, 0, 0, 0};
    r[0] = and_or(w << 3, 0x88888888u, 0x44444444u), r[1] = and_or(w << 2, 0x88888888u, 0x22222222u);
    r[2] = and_or(w << 1, 0x88888888u, 0x11111111u), r[3] = and_or(w, 0x88888888u, 0x44444444u);
    return r;
}
__device__ __forceinline__ i32x8 bitspm1(uint32_t w) {
    i32x8 r = {0, 0, 0, 0, 0, 0, 0, 0};
    r[0] = and_or(w << 3, 0x88888888u, 0x22222222u), r[1] = and_or(w << 2, 0x88888888u, 0x22222222u);
    r[2] = and_or(w << 1, 0x88888888u, 0x22222222u), r[3] = and_or(w, 0x88888888u, 0x22222222u);
    return r;
}

// Expanded dwords in memory hold only the four that 4-bit floats use.
__device__ __forceinline__ i32x4 lower_half(const i32x8 &v) { return i32x4{v[0], v[1], v[2], v[3]}; }
__device__ __forceinline__ i32x8 upper_zero(const i32x4 &v) { return i32x8{v[0], v[1], v[2], v[3], 0, 0, 0, 0}; }

// acc += A * B.  T = 32: 32 x 32 outputs over 64 depths, lane l holds row / column l % 32, depths 32 * (l / 32) ..;
// T = 16: 16 x 16 over 128 depths, row / column l % 16, depths 32 * (l / 16) ...
// Accumulator register v of lane l: column l % T, row fp4_row<T>(l / T, v).
template <int T>
struct Fp4Acc;
template <>
struct Fp4Acc<16> {
    typedef f32x4m type;
    static constexpr int regs = 4;
};
template <>
struct Fp4Acc<32> {
    typedef f32x16m type;
    static constexpr int regs = 16;
};
template <int T>
__device__ __forceinline__ void mfma_fp4(typename Fp4Acc<T>::type &acc, const i32x8 &a, const i32x8 &b) {
    if constexpr (T == 16)
        acc = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a, b, acc, 4, 4, 0, 0, 0, 0);
    else
        acc = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a, b, acc, 4, 4, 0, 0, 0, 0);
}
template <int T>
__device__ __forceinline__ constexpr int fp4_row(int kb, int v) {
    return T == 16 ? 4 * kb + v : 8 * (v / 4) + 4 * kb + v % 4;
}

// N dwords through a buffer descriptor / from LDS
template <int N>
__device__ __forceinline__ void load_dwords(uint32_t (&d)[N], __amdgpu_buffer_rsrc_t r, int off, int scalar = 0) {
    static_assert(N == 1 || N == 2 || N % 4 == 0, "whole loads");
    if constexpr (N == 1) {
        d[0] = __builtin_amdgcn_raw_buffer_load_b32(r, off, scalar, 0);
    } else if constexpr (N == 2) {
        const u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(r, off, scalar, 0);
        d[0] = v.x, d[1] = v.y;
    } else {
#pragma unroll
        for (int i = 0; i < N / 4; ++i) {
            const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(r, off, scalar + i * 16, 0);
            d[4 * i] = v.x, d[4 * i + 1] = v.y, d[4 * i + 2] = v.z, d[4 * i + 3] = v.w;
        }
    }
}
template <int N>
__device__ __forceinline__ void lds_dwords(uint32_t (&d)[N], const unsigned char *p) {
    if constexpr (N == 1) {
        d[0] = *reinterpret_cast<const uint32_t *>(p);
    } else if constexpr (N == 2) {
        const u32x2 v = *reinterpret_cast<const u32x2 *>(p);
        d[0] = v.x, d[1] = v.y;
    } else {
#pragma unroll
        for (int i = 0; i < N / 4; ++i) {
            const u32x4 v = *reinterpret_cast<const u32x4 *>(p + 16 * i);
            d[4 * i] = v.x, d[4 * i + 1] = v.y, d[4 * i + 2] = v.z, d[4 * i + 3] = v.w;
        }
    }
}

// A value into lane `lane` (a constant) of a register: v_writelane_b32, for which this compiler has no builtin.
extern "C" __device__ __attribute__((const)) uint32_t dab_writelane(uint32_t value, uint32_t lane, uint32_t old) __asm("llvm.amdgcn.writelane.i32");

// Cache policies of buffer stores (the builtins' last operand): streaming, and written through the L2 at device scope.
constexpr int kStoreStream = 2, kStoreThrough = 16;

}  // namespace dab
