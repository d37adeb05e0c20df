// f32 products on the bf16 matrix cores: every operand value is taken apart into three bf16 pieces whose sum IS the value, and
// a product is put together from the six pairs of pieces that reach f32.
//
// v_mfma_f32_32x32x2_f32 does 64 multiply-adds per lane in 64 cycles, v_mfma_f32_32x32x16_bf16 does 512 in 32: six of the
// latter for eight of the former make 192 cycles against 512, and both accumulate in f32.
//   x = h + m + l:  h = bf16(x), m = bf16(x - h), l = x - h - m.  Both differences are exact (a value has 24 significant bits, a
//   piece holds 8, and a rounding leaves at most half a place of the piece before it), so nothing of the operand is lost
//   down to |x| = 2^-110.
//   x y = hh' + (hm' + mh') + (mm' + hl' + lh') + (ml' + lm' + ll'); the last three are left out: |m| <= 2^-8 |h| and
//   |l| <= 2^-16 |h| make them 2^-23 of the product at most and 2^-26 on average, of either sign, where one f32 addition rounds
//   2^-24 of the running sum -- and a step of 16 along the inner dimension has six such additions here and eight there.
// Against double precision sums (192 x 3072 outputs, inner length 2304, relative error of the 2-norm): 4e-7 here, 8e-7 with
// the f32 matrix instruction.
// Operands without three finite pieces -- infinite, NaN, or so large that the first piece rounds to infinity (kSplitLimit) -- make every
// sum they enter infinite or NaN.  Such a sum is looked for once, when it is finished (split_all_finite), and put in its place comes the
// chain of f32 multiply-adds it stands for, from the operands themselves: an infinity stays one, and a large value is a value.
#pragma once

#include "device_common.h"

namespace mynah {

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

__device__ __forceinline__ unsigned bf16_pair(float a, float b) {   // one instruction (v_cvt_pk_bf16_f32, round to nearest even)
    const f32x2 v = {a, b};
    return __builtin_bit_cast(unsigned, __builtin_convertvector(v, bf16x2));
}
__device__ __forceinline__ float bf16_low(unsigned p) { return __uint_as_float(p << 16); }
__device__ __forceinline__ float bf16_high(unsigned p) { return __uint_as_float(p & 0xffff0000u); }

constexpr float kSplitLimit = 0x1.ffp127f;   // bf16 rounds what is not below it to infinity
// Where pieces are all that is kept of an operand, one from kSplitLimit on is kept as (infinity, upper half, lower half of its bits): it
// makes its products infinite or NaN as it must, and can be had again.  piece: 16 bits each, as they lie in memory.
__device__ __forceinline__ void split_keep_bits(float x, unsigned short &h, unsigned short &m, unsigned short &l) {
    if (fabsf(x) < kSplitLimit) return;
    h = 0x7f80;
    m = (unsigned short)(__float_as_uint(x) >> 16);
    l = (unsigned short)__float_as_uint(x);
}
__device__ __forceinline__ float split_value(unsigned short h, unsigned short m, unsigned short l) {
    if (h == 0x7f80) return __uint_as_float((unsigned)m << 16 | l);
    return __uint_as_float((unsigned)h << 16) + (__uint_as_float((unsigned)m << 16) + __uint_as_float((unsigned)l << 16));   // exact
}

// The three pieces of four neighbouring values, 8 bytes each (22 vector instructions).
struct SplitFour {
    uint2 piece[3];
    __device__ __forceinline__ explicit SplitFour(const float4 v) {
        const unsigned h0 = bf16_pair(v.x, v.y), h1 = bf16_pair(v.z, v.w);
        const float x = v.x - bf16_low(h0), y = v.y - bf16_high(h0), z = v.z - bf16_low(h1), w = v.w - bf16_high(h1);
        const unsigned m0 = bf16_pair(x, y), m1 = bf16_pair(z, w);
        piece[0] = make_uint2(h0, h1);
        piece[1] = make_uint2(m0, m1);
        piece[2] = make_uint2(bf16_pair(x - bf16_low(m0), y - bf16_high(m0)), bf16_pair(z - bf16_low(m1), w - bf16_high(m1)));
    }
    __device__ __forceinline__ void keep_bits(const float4 v) {
        typedef unsigned short ushort4_t __attribute__((ext_vector_type(4)));
        const float x[4] = {v.x, v.y, v.z, v.w};
        ushort4_t at[3];
#pragma unroll
        for (int q = 0; q < 3; ++q) at[q] = __builtin_bit_cast(ushort4_t, piece[q]);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            unsigned short h = at[0][e], m = at[1][e], l = at[2][e];
            split_keep_bits(x[e], h, m, l);
            at[0][e] = h;
            at[1][e] = m;
            at[2][e] = l;
        }
#pragma unroll
        for (int q = 0; q < 3; ++q) piece[q] = __builtin_bit_cast(uint2, at[q]);
    }
};
// ... of eight: one operand of a matrix instruction per piece.
__device__ __forceinline__ void split_eight(const float4 a, const float4 b, bf16x8 (&out)[3]) {
    const SplitFour x(a), y(b);
#pragma unroll
    for (int p = 0; p < 3; ++p) out[p] = __builtin_bit_cast(bf16x8, make_uint4(x.piece[p].x, x.piece[p].y, y.piece[p].x, y.piece[p].y));
}

__device__ __forceinline__ bool split_finite(float x) { return fabsf(x) < __builtin_inff(); }
// Whether all sums of the wavefront are finite (one instruction a value: 0 * x is 0 or NaN).
template <int N>
__device__ __forceinline__ bool split_all_finite(const f32x16 (&acc)[N]) {
    float zero[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int n = 0; n < N; ++n)
#pragma unroll
        for (int r = 0; r < 16; ++r) zero[r & 3] = __builtin_fmaf(acc[n][r], 0.0f, zero[r & 3]);
    return !__any((zero[0] + zero[1]) + (zero[2] + zero[3]) != 0.0f);
}
// One 16-deep step: acc += a * w over the six pairs, the smallest first.
__device__ __forceinline__ f32x16 split_multiply(const bf16x8 (&a)[3], const bf16x8 (&w)[3], f32x16 acc) {
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[2], w[0], acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[0], w[2], acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[1], w[1], acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[1], w[0], acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[0], w[1], acc, 0, 0, 0);
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[0], w[0], acc, 0, 0, 0);
}

// Row of C held in accumulator register r of lane l for a 32x32 tile; the column is l % 32.
__device__ __forceinline__ int split_acc_row(int r, int lane) { return 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3); }

}  // namespace mynah
