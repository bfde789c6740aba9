// fp32 products on the bf16 matrix cores: every fp32 value as three bf16 ones,
// six of the nine products of their pieces (Henry, Tang and Heinecke,
// "Leveraging the bfloat16 Artificial Intelligence Datatype For
// Higher-Precision Computations", ARITH 2019).
//
// With x scaled by 2^23, hi = bf16(x), mid = bf16(x - hi), lo = x - hi - mid:
// 8 significand bits each.  Unscaled, the low pieces of values under 2^-110
// would fall below bf16's smallest value; scaled, the last bit of the smallest
// fp32 denormal is bf16's smallest normal, so the three pieces hold every
// value below 2^105 exactly, zeros and denormals included.  The product of two
// scaled values is scaled by 2^46; the accumulators are brought back at the
// end, which is exact down to fp32's own denormals.
//
// A product is the sum of the nine products of its pieces.  Six are kept (hi
// hi, hi mid, mid hi, mid mid, hi lo, lo hi); mid lo, lo mid and lo lo are left
// out: at most 2^-24 of the product (|mid| <= 2^-8, |lo| <= 2^-17 of it), 2^-27.4
// rms over N(0,1) and U[1,2) pairs.  2^-24 is what an fp32 product's own rounding
// may be, so a sum of a single product is off by up to 2.5 x 2^-24 of it (the
// matrix unit's rounding included) where v_mfma_f32_32x32x2_f32 is by 1.0.
// Sums of several gain it back: every piece product is exact in the matrix
// unit, which adds 16 of them to the fp32 accumulator in one step, so a K-long
// sum is rounded 6 K / 16 times instead of K / 2.
//
// Measured on MI355X against 64-bit sums, 2-norm of the error over that of the result, this
// against v_mfma_f32_32x32x2_f32: N(0,1) x N(0,1) at K 1 / 2 / 3 / 8 3.4e-8 / 3.4e-8 / 3.3e-8 /
// 3.1e-8 against 2.5e-8 / 3.1e-8 / 3.6e-8 / 5.3e-8; N(0,1) x N(0,0.02) at K 64 / 1,024 /
// 4,096 / 14,336 1.16e-7 / 5.0e-7 / 1.05e-6 / 2.0e-6 against 1.42e-7 / 5.7e-7 / 1.12e-6 /
// 2.2e-6; U[0,1] x U[0,1] 8.6e-8 / 2.9e-7 / 5.3e-7 / 1.1e-6 against 1.1e-7 / 4.3e-7 / 8.3e-7 /
// 1.7e-6.
//
// What the pieces do not hold the caller computes with fp32 MFMA instead:
// infinities and NaN (x - hi is NaN), magnitudes from 2^105 on (hi overflows)
// and sums that pass 2^82 -- all of these leave a non-finite accumulator.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace moe {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr float kSplitScale = 8388608.0f;                // 2^23
constexpr float kSplitUnscale = 1.4210854715202004e-14f;  // 2^-46

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

// The pieces of a and b, scaled by 2^23: p[0] their hi, p[1] their mid, p[2] their lo.
__device__ __forceinline__ void split_pair(float a, float b, uint32_t (&p)[3]) {
    a *= kSplitScale;
    b *= kSplitScale;
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
