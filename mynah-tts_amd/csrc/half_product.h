// f32 products on the f16 matrix cores: every operand value is taken apart into two f16 pieces, and a product is put together from the
// three pairs of pieces that reach f32.
//
// v_mfma_f32_32x32x2_f32 does 64 multiply-adds per lane in 64 cycles, v_mfma_f32_32x32x16_f16 does 512 in 32: three of the latter for
// eight of the former make 96 cycles against 512 (three bf16 pieces a value need six: 192).  All accumulate in f32.
//   s x = h + 2^-11 m + 2^-22 l:  h = f16(s x), m = f16(2^11 (s x - h)), l = f16(2^11 (2^11 (s x - h) - m)), s a power of two.  The
//   differences are exact; two pieces hold 22 bits and the sign between them, three hold the value.
//   x y = (hh' + 2^-11 (hm' + mh') + ...) / s s'.  What is left out is at most 2^-22 of the product and 2^-24.5 of it in the mean, of either
//   sign and independent from term to term, so that a sum of many keeps that share; one f32 addition rounds up to 2^-24 of the running sum.
//   The two small products have sums of their own: the large chain then has one addition per sixteen terms where the three bf16
//   pieces had six, which is why the result is the closer one.
// f16 holds s x in full from 2^-14 to 2^16: that is what the scales are for.
//   A weight has one per output row, so that the row's largest value lies in [2^13, 2^14) (half_row_scale); it is divided out of the finished sum.
//   An input has 1, as long as the largest that a tile reads of it is in [2^-10, 65520): then what the two pieces miss is 2^-37 at most, or
//   2^-27 of that largest.  A tile whose largest input is smaller, or larger up to 2^24, is multiplied once more with a scale of its own
//   (half_rescale): twice the time, in tiles that hold nothing but near silence or values that no trained network has.  (What stands beside a value
//   just below 2^24 loses 2^-26 at most, which is half of f32's last place of 1/2.)
// Operands without two finite pieces (infinite, NaN, or out of those ranges upwards) make every sum they enter infinite or NaN.  Such a sum
// is looked for once, when it is finished, and put in its place comes the chain of f32 multiply-adds it stands for, from the operands
// themselves, which a weight's three pieces are: an infinity stays one, and a large value is a value.
#pragma once

#include "device_common.h"

namespace mynah {

typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
typedef _Float16 half4_t __attribute__((ext_vector_type(4)));
typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef unsigned short ushort4_t __attribute__((ext_vector_type(4)));
typedef unsigned short ushort8_t __attribute__((ext_vector_type(8)));

constexpr float kHalfLimit = 65520.0f;    // f16 rounds what is not below it to infinity
constexpr float kHalfStep = 2048.0f;      // 2^11: from a piece to the next
constexpr unsigned short kHalfMarked = 0x7c00;

__device__ __forceinline__ unsigned half_pair(float a, float b) {   // one instruction (v_cvt_pk_f16_f32, round to nearest even)
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    const f32x2 v = {a, b};
    return __builtin_bit_cast(unsigned, __builtin_convertvector(v, half2_t));
}
// The pieces of two neighbouring values under a scale: h and m (seven vector instructions), and what h leaves.
__device__ __forceinline__ void half_pieces(float a, float b, float scale, unsigned &h, unsigned &m, float (&rest)[2]) {
    a *= scale;
    b *= scale;
    h = half_pair(a, b);
    const half2_t hh = __builtin_bit_cast(half2_t, h);
    rest[0] = __builtin_fmaf((float)hh[0], -1.0f, a);   // exact (v_fma_mix_f32)
    rest[1] = __builtin_fmaf((float)hh[1], -1.0f, b);
    const half2_t mm = {(_Float16)(rest[0] * kHalfStep), (_Float16)(rest[1] * kHalfStep)};
    m = __builtin_bit_cast(unsigned, mm);
}
__device__ __forceinline__ unsigned half_third(unsigned m, const float (&rest)[2]) {
    const half2_t mm = __builtin_bit_cast(half2_t, m);
    return half_pair((rest[0] * kHalfStep - (float)mm[0]) * kHalfStep, (rest[1] * kHalfStep - (float)mm[1]) * kHalfStep);
}
// Where pieces are all that is kept of an operand, one without a finite first piece is kept as (infinity, upper half, lower half of its
// bits): it makes its products infinite or NaN as it must, and can be had again.  One so far below the scale that its first two pieces are
// zero is kept as (-0, 0, its upper half, rounded).
constexpr float kHalfNothing = 0x1p-37f;
__device__ __forceinline__ void half_keep_bits(float x, float scale, unsigned short &h, unsigned short &m, unsigned short &l) {
    if (x != 0.0f && fabsf(x * scale) < kHalfNothing) {
        h = 0x8000;
        m = 0;
        l = (unsigned short)((__float_as_uint(x) + 0x8000u) >> 16);
        return;
    }
    if (fabsf(x * scale) < kHalfLimit) return;
    h = kHalfMarked;
    m = (unsigned short)(__float_as_uint(x) >> 16);
    l = (unsigned short)__float_as_uint(x);
}
__device__ __forceinline__ float half_value(unsigned short h, unsigned short m, unsigned short l, float inverse) {
    if (h == kHalfMarked) return __uint_as_float((unsigned)m << 16 | l);
    if (h == 0x8000 && m == 0) return __uint_as_float((unsigned)l << 16);
    const auto f = [](unsigned short b) { return (float)__builtin_bit_cast(_Float16, b); };
    return (f(h) + (f(m) + f(l) * (1.0f / kHalfStep)) * (1.0f / kHalfStep)) * inverse;   // exact
}

// Two pieces of eight values, an operand of a matrix instruction each.  largest: takes part in the largest size among them.
__device__ __forceinline__ void half_eight(const float (&v)[8], float scale, float &largest, uint4 &h, uint4 &m) {
    unsigned hp[4], mp[4];
    float rest[2];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        half_pieces(v[2 * i], v[2 * i + 1], scale, hp[i], mp[i], rest);
        largest = fmaxf(largest, fmaxf(fabsf(v[2 * i]), fabsf(v[2 * i + 1])));
    }
    h = make_uint4(hp[0], hp[1], hp[2], hp[3]);
    m = make_uint4(mp[0], mp[1], mp[2], mp[3]);
}

__device__ __forceinline__ float power_of_two(int e) { return __uint_as_float((unsigned)(e + 127) << 23); }   // -126 .. 127
__device__ __forceinline__ int exponent_of(float x) { return (int)(__float_as_uint(x) >> 23 & 255) - 127; }     // (-127: zero and the subnormal values)
// The power of two under which a tile's inputs are taken apart again, or 0 where its products hold.
__device__ __forceinline__ int half_rescale(float largest) {
    const bool quiet = largest < 0x1p-10f && largest > 0.0f, loud = largest >= kHalfLimit && largest < 0x1p24f;
    return quiet || loud ? min(13 - exponent_of(largest), 100) : 0;
}

// A value at `bytes` behind an address that is the same for every lane: one instruction with the address in scalar registers, where
// pointer arithmetic by lanes takes 64-bit addresses in vector registers.
// (opaque: what stays the same from request to request is otherwise added up ahead of all loops, 64 bits a lane and request)
template <class T>
__device__ __forceinline__ T load_behind(const T *base, unsigned bytes) { return *reinterpret_cast<const T *>(reinterpret_cast<const char *>(base) + bytes); }
__device__ __forceinline__ unsigned opaque(unsigned v) {
    asm volatile("" : "+v"(v));
    return v;
}
__device__ __forceinline__ int opaque_scalar(int v) {
    asm volatile("" : "+s"(v));
    return v;
}

// The three pieces of eight values, or their bits: where they are all that is kept of an operand.
__device__ __forceinline__ void half_keep_eight(const float (&v)[8], float scale, uint4 (&piece)[3]) {
    ushort8_t at[3];
#pragma unroll
    for (int e = 0; e < 8; e += 2) {
        unsigned h, m;
        float rest[2];
        half_pieces(v[e], v[e + 1], scale, h, m, rest);
        const unsigned l = half_third(m, rest);
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            unsigned short ph = (unsigned short)(h >> 16 * k), pm = (unsigned short)(m >> 16 * k), pl = (unsigned short)(l >> 16 * k);
            half_keep_bits(v[e + k], scale, ph, pm, pl);
            at[0][e + k] = ph;
            at[1][e + k] = pm;
            at[2][e + k] = pl;
        }
    }
#pragma unroll
    for (int q = 0; q < 3; ++q) piece[q] = __builtin_bit_cast(uint4, at[q]);
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
// Row of C held in accumulator register r of lane l for a 32x32 tile; the column is l % 32.
__device__ __forceinline__ int split_acc_row(int r, int lane) { return 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3); }

struct HalfSums {   // a 32 x 32 tile: the products of the first pieces, and the small ones in units of 2^-11
    f32x16 large, small;
    __device__ __forceinline__ void clear() { large = small = f32x16{0}; }
    // One 16-deep step.
    __device__ __forceinline__ void multiply(const half8_t (&a)[2], const half8_t (&b)[2]) {
        small = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[1], b[0], small, 0, 0, 0);
        large = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[0], b[0], large, 0, 0, 0);
        small = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[0], b[1], small, 0, 0, 0);
    }
    __device__ __forceinline__ float sum(int r) const { return __builtin_fmaf(small[r], 1.0f / kHalfStep, large[r]); }
};

}  // namespace mynah
