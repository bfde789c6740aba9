// fp32 products on the bf16 matrix cores.
//
// An fp32 value is the exact sum of three bf16 values: hi = bf16(x), mid =
// bf16(x - hi), lo = bf16(x - hi - mid); 8 significand bits each, and bf16
// has fp32's exponents, so no range is lost.  A product of two values is the
// sum of the nine products of their pieces; the six with weight down to
// 2^-18 (hi hi, hi mid, mid hi, mid mid, hi lo, lo hi) are kept, and what is
// left out (mid lo, lo mid, lo lo) is at most 2^-26 of the product, a quarter
// of the rounding an fp32 product carries by itself.  Every piece product is
// exact in the matrix unit, which adds 16 of them to the fp32 accumulator in
// one step, so a K-long sum is rounded 6 K / 16 times instead of the K / 2 of
// v_mfma_f32_32x32x2_f32.
//
// Measured on MI355X against 64-bit sums, 2-norm of the error over that of the result, this
// against v_mfma_f32_32x32x2_f32: N(0,1) x N(0,0.02) at K 64 / 1,024 / 4,096 / 14,336
// 1.16e-7 / 5.0e-7 / 1.05e-6 / 2.0e-6 against 1.42e-7 / 5.7e-7 / 1.12e-6 / 2.2e-6;
// U[0,1] x U[0,1] 8.6e-8 / 2.9e-7 / 5.3e-7 / 1.1e-6 against 1.1e-7 / 4.3e-7 / 8.3e-7 / 1.7e-6.
//
// Where the split is not exact the caller computes the block with fp32 MFMA
// instead: infinities and NaN (x - hi is NaN), values within bf16's last
// rounding of the largest float (hi overflows), sums that overflow only
// through a rounded-up hi -- all of these leave a non-finite accumulator --
// and non-zero values below kSplitTiny, whose lo would fall under bf16's
// smallest denormal.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace moe {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// 2^-100: lo >= 2^-24 of its value, bf16 holds multiples of 2^-133
constexpr float kSplitTiny = 7.888609052210118e-31f;

// (bf16(a), bf16(b)) in one register, a in the low half (round to nearest even)
__device__ __forceinline__ uint32_t pack_bf16(float a, float b) {
    typedef float f32x2_ __attribute__((ext_vector_type(2)));
    const bf16x2 v = __builtin_convertvector((f32x2_{a, b}), bf16x2);
    return __builtin_bit_cast(uint32_t, v);
}
__device__ __forceinline__ float low_bf16(uint32_t v) { return __uint_as_float(v << 16); }
__device__ __forceinline__ float high_bf16(uint32_t v) {
    return __uint_as_float(v & 0xffff0000u);
}

// The pieces of a and b: p[0] their hi, p[1] their mid, p[2] their lo.
__device__ __forceinline__ void split_pair(float a, float b, uint32_t (&p)[3]) {
    p[0] = pack_bf16(a, b);
    const float ra = a - low_bf16(p[0]), rb = b - high_bf16(p[0]);
    p[1] = pack_bf16(ra, rb);
    p[2] = pack_bf16(ra - low_bf16(p[1]), rb - high_bf16(p[1]));
}

// The piece products kept, smallest first: (A piece, B piece).
constexpr int kSplitTerms = 6;
constexpr int kSplitA[kSplitTerms] = {2, 0, 1, 1, 0, 0};
constexpr int kSplitB[kSplitTerms] = {0, 2, 1, 0, 1, 0};

}  // namespace moe
