// bf3.hpp -- FP32 products on the bf16 matrix unit by exact splitting.
//
// An FP32 value is the sum of three bf16 values, x = h + m + l: h the top
// eight significand bits (truncated), m the rest rounded to eight bits, l
// what is left, which eight bits hold exactly (24 = 8 + 8 + 8; values whose
// pieces would fall below 2^-126 lose those bits, an absolute error under
// 2^-133).  A product a.b is then formed as six bf16 MFMAs, each exact into an FP32
// accumulator:
//   main   h.h
//   cross  h.m + m.h + m.m + h.l + l.h
// and the three dropped terms (m.l, l.m, l.l) are below 2^-23 of the product
// with random signs.  v_mfma_f32_32x32x16_bf16 multiplies 16384 pairs in 32
// cycles where v_mfma_f32_16x16x4_f32 takes 512: six of them are 2.7 times
// the FP32 matrix rate.  Against 64 bits, sums of K products of N(0, 1)
// values are off by (2-norm, MI355X): K = 64 5.4e-8, 768 1.6e-7, 6144 4.9e-7,
// with FP32 MFMA 1.4e-7, 4.9e-7, 1.4e-6, the cross terms in an accumulator of
// their own; with both in one accumulator 9.5e-8, 4.1e-7, 1.3e-6.
//
// Infinities and NaN: h keeps them (truncation never overflows), while m and
// l become NaN and meet the cross accumulator only, so a non-finite main sum
// is the result as it stands (bf3_join): the FP32 product's own value.
#pragma once

#include "common.hpp"

namespace cxg {

typedef __bf16 b8 __attribute__((ext_vector_type(8)));
typedef __bf16 b2 __attribute__((ext_vector_type(2)));
typedef float f2 __attribute__((ext_vector_type(2)));
typedef float f16 __attribute__((ext_vector_type(16)));
typedef unsigned u2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ f16 mfma32b(b8 a, b8 b, f16 c)
{
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ f4 mfma16b(b8 a, b8 b, f4 c)
{
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// A finished chain of MFMAs, before vector or memory instructions read it.  The
// compiler's own wait for a 32x32x16 result has been seen four cycles short
// where a branch lies between the MFMA and the reader (the last of the sixteen
// registers came out stale), so the wait is written out: sixteen wait states,
// where the matrix unit needs eleven.
__device__ __forceinline__ void settle(f16& x) { asm volatile("s_nop 15" : "+v"(x)); }

// The pieces of two values, each pair packed (a low, b high): eleven VALU
// instructions.
__device__ __forceinline__ void bf3_split2(float a, float b, unsigned& h, unsigned& m, unsigned& l)
{
    const unsigned ua = __builtin_bit_cast(unsigned, a), ub = __builtin_bit_cast(unsigned, b);
    h = __builtin_amdgcn_perm(ub, ua, 0x07060302u);
    const float ra = a - __builtin_bit_cast(float, ua & 0xffff0000u);
    const float rb = b - __builtin_bit_cast(float, ub & 0xffff0000u);
    m = __builtin_bit_cast(unsigned, __builtin_convertvector((f2){ra, rb}, b2));
    const float sa = ra - __builtin_bit_cast(float, m << 16);
    const float sb = rb - __builtin_bit_cast(float, m & 0xffff0000u);
    l = __builtin_bit_cast(unsigned, __builtin_convertvector((f2){sa, sb}, b2));
}

// The same in four parts of two or three instructions, for a caller that puts
// MFMAs between them: a and b are left as the rests.
__device__ __forceinline__ void bf3_split2_part(int part, float& a, float& b, unsigned& h, unsigned& m,
                                                unsigned& l)
{
    const unsigned ua = __builtin_bit_cast(unsigned, a), ub = __builtin_bit_cast(unsigned, b);
    if (part == 0) {
        h = __builtin_amdgcn_perm(ub, ua, 0x07060302u);
        a -= __builtin_bit_cast(float, ua & 0xffff0000u);
    } else if (part == 1) {
        b -= __builtin_bit_cast(float, ub & 0xffff0000u);
        m = __builtin_bit_cast(unsigned, __builtin_convertvector((f2){a, b}, b2));
    } else if (part == 2) {
        a -= __builtin_bit_cast(float, m << 16);
    } else {
        b -= __builtin_bit_cast(float, m & 0xffff0000u);
        l = __builtin_bit_cast(unsigned, __builtin_convertvector((f2){a, b}, b2));
    }
}

// A sum from its main and cross accumulators.
__device__ __forceinline__ float bf3_join(float main, float cross)
{
    return __builtin_isfinite(main) ? main + cross : main;
}

// LDS planes of bf16 rows, DHP columns a row.  A row's 16-byte chunks are
// exchanged by its number, so that a row operand's ds_read_b128 and a column
// operand's transposing read each cover the 64 banks once: measured, a wave's
// b128 read takes 4.5 cycles so and 8 to 16 otherwise.
template <int DHP>
__device__ __forceinline__ int swz(int row)
{
    if constexpr (DHP == 32 || DHP == 96)
        return (row >> 2) & 3;
    else if constexpr (DHP == 64)
        return 4 * ((row >> 1) & 1) + ((row >> 2) & 3);
    else
        return 4 * (row & 3) + ((row >> 2) & 3);
}

template <int DHP>
__device__ __forceinline__ int chunk_off(int row, int c)
{
    return row * (DHP * 2) + ((c ^ swz<DHP>(row)) << 4);
}

// Column operand of k-step rows r0 .. r0+15 (r0 a multiple of 16), columns
// c0 .. c0+31, from one plane: two transposing reads (ds_read_b64_tr_b16: a
// group of 16 lanes reads four rows' 16 columns, lane i receiving column i).
// Slot (g, e) is row r0 + 8 (e / 4) + 4g + e % 4, an accumulator's order, or
// with NAT row r0 + 8g + e, a row operand's.
template <int DHP, bool NAT = false>
__device__ __forceinline__ b8 read_tr(const char* plane, int r0, int c0, int lane)
{
    typedef short s4v __attribute__((ext_vector_type(4)));
    typedef __attribute__((address_space(3))) s4v* lp;
    const int g = lane >> 5, i = lane & 15;
    const int row = r0 + (NAT ? 8 : 4) * g + (i >> 2);
    const int col = c0 + 16 * ((lane >> 4) & 1) + 4 * (i & 3);
    const char* a = plane + chunk_off<DHP>(row, col >> 3) + 2 * (col & 7);
    const char* b = plane + chunk_off<DHP>(row + (NAT ? 4 : 8), col >> 3) + 2 * (col & 7);
    const s4v x = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lp)a);
    const s4v y = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lp)b);
    return __builtin_bit_cast(b8, __builtin_shufflevector(x, y, 0, 1, 2, 3, 4, 5, 6, 7));
}

template <int DHP>
__device__ __forceinline__ b8 read_row(const char* plane, int row, int c)
{
    return *reinterpret_cast<const b8*>(plane + chunk_off<DHP>(row, c));
}

// eight values to their three pieces
__device__ __forceinline__ void split8(const float* v, b8& h, b8& m, b8& l)
{
    u4 x, y, z;
#pragma unroll
    for (int e = 0; e < 4; e++) {
        unsigned a, b, c;
        bf3_split2(v[2 * e], v[2 * e + 1], a, b, c);
        x[e] = a;
        y[e] = b;
        z[e] = c;
    }
    h = __builtin_bit_cast(b8, x);
    m = __builtin_bit_cast(b8, y);
    l = __builtin_bit_cast(b8, z);
}

// The cross terms of a product: pieces (pa, pb) = h.m, m.h, m.m, h.l, l.h.
constexpr int kPa[5] = {0, 1, 1, 0, 2}, kPb[5] = {1, 0, 1, 2, 0};

__device__ __forceinline__ f16 f16zero()
{
    f16 z;
#pragma unroll
    for (int i = 0; i < 16; i++)
        z[i] = 0.0f;
    return z;
}

} // namespace cxg
