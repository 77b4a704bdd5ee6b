// fp32 products on the bf16 matrix cores, without giving up fp32 accuracy.
//
// An fp32 value is the exact sum of three bf16 values: h = bf16(x),
// m = bf16(x - h), l = bf16(x - h - m) (round to nearest; the two
// differences are exact in fp32, and 3 x 8 significand bits cover its 24).
// A product x y is then formed from six bf16 products,
//     hh' + (hm' + mh') + (mm' + hl' + lh'),
// each exact in the fp32 accumulator's input.  Of the three products left out
// ml' and lm' reach 2^-25 of x y each (|m| <= 2^-8 |x|, |l| <= 2^-17 |x|): 2^-24
// at most, half an fp32 ulp or one, and 2^-27.4 rms.  A single product is
// then not always the correctly rounded one, so sums of one or two stay with
// the fp32 kernels (kSplitLeast); from three on the fp32 chain's own roundings
// are the larger error (3584 x K x 3584, two-norm, fp32 and split: K = 1 2.53e-8,
// 3.45e-8; 2 3.12e-8, 3.38e-8; 3 3.57e-8, 3.29e-8; 16 7.4e-8, 3.4e-8).  The
// accumulator is fp32 as before, and the six are summed from the smallest
// terms up.  v_mfma_f32_32x32x16_bf16 does 16 times the multiply-adds per
// cycle of v_mfma_f32_32x32x2_f32, so six of them leave a factor of 2.7 in
// matrix-core cycles.
//
// Range: bf16 has fp32's exponents, but parts of x below 2^-110 reach its
// subnormals and end at 2^-133.  So operands are scaled by 2^16 on the way to
// their parts (exact; then every fp32 value, subnormals included, is a
// multiple of 2^-133) and the sums by 2^-32: one more vector instruction a
// value beside 5.5, up to 3% of a call (both builds on one box: 4096^3 571.5 ->
// 572.5 us, 1537 x 1000 x 2999 65.6 -> 67.1, N32 64->128 3x3 56^2 99.2 -> 100.4
// and its two gradients 228 -> 236).  Above, what passes the largest
// bf16 as scaled (2^112) rounds to infinity, and infinities and NaN give NaN
// in the differences; sums of 2^96 overflow.  Every such case makes the
// affected sums non-finite, and the kernels recompute a tile whose sums are
// not all finite with the fp32 matrix instructions, so those inputs give what
// they give in fp32.
#pragma once

#include "kernels.hpp"

namespace lancius {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x8 __attribute__((ext_vector_type(8)));

// One lane's MFMA operand: eight consecutive k of one row, in three parts.
struct SplitOperand {
    bf16x8 h, m, l;
};

// bf16 of two floats in one register, and those two back as floats.
__device__ __forceinline__ unsigned pack_bf16(float a, float b) {
    const f32x2 v = {a, b};
    return __builtin_bit_cast(unsigned, __builtin_convertvector(v, bf16x2));
}

// Products that a sum has at least.
constexpr size_t kSplitLeast = 3;
constexpr float kSplitUp = 0x1p16f, kSplitDown = 0x1p-32f;

// The three parts of x; split8_up: of x as scaled.
__device__ __forceinline__ SplitOperand split8(f32x8 x) {
    u32x4 h, m, l;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        float a = x[2 * i], b = x[2 * i + 1];
        h[i] = pack_bf16(a, b);
        a -= __builtin_bit_cast(float, h[i] << 16);
        b -= __builtin_bit_cast(float, h[i] & 0xffff0000u);
        m[i] = pack_bf16(a, b);
        a -= __builtin_bit_cast(float, m[i] << 16);
        b -= __builtin_bit_cast(float, m[i] & 0xffff0000u);
        l[i] = pack_bf16(a, b);
    }
    return {__builtin_bit_cast(bf16x8, h), __builtin_bit_cast(bf16x8, m), __builtin_bit_cast(bf16x8, l)};
}

__device__ __forceinline__ SplitOperand split8_up(f32x8 x) { return split8(x * kSplitUp); }

__device__ __forceinline__ f32x16 mfma_bf16(bf16x8 a, bf16x8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

// An instruction that reads a matrix instruction's result needs wait states
// that the compiler counts; across a branch it has been seen to count them
// along the longer of two paths only (the reader got registers 14 and 15 of a
// 32 x 32 result from before the last product).  So a result that is read
// behind control flow passes one of these first.
//  settle: the value is complete here, whatever follows (20 wait states).
//  pin: the instruction that computed the value stays in this block, where
//  the count is right; for values that vector instructions have already read
//  out of the matrix result.
__device__ __forceinline__ void pin(f32x16& c) { asm volatile("" : "+v"(c)); }
template <int M, int N>
__device__ __forceinline__ void settle(f32x16 (&c)[M][N]) {
#pragma unroll
    for (int i = 0; i < M; ++i)
#pragma unroll
        for (int j = 0; j < N; ++j) pin(c[i][j]);
    asm volatile("s_nop 15\n\ts_nop 3");
#pragma unroll
    for (int i = 0; i < M; ++i)
#pragma unroll
        for (int j = 0; j < N; ++j) pin(c[i][j]);
}
__device__ __forceinline__ void settle(f32x16& c) {
    pin(c);
    asm volatile("s_nop 15\n\ts_nop 3");
    pin(c);
}

}  // namespace lancius
