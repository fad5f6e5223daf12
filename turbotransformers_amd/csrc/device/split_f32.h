// fp32 products on the 16-bit matrix instructions of gfx950: a value is split in two halves of 11 bits,
//
//   x = hi + lo / 2^16,  hi = fp16(x),  lo = fp16((x - hi) * 2^16),  to within 2^-22 max(|x|, 2^-14)
//   a b = hi_a hi_b + (hi_a lo_b + lo_a hi_b) / 2^16,  to within 3 * 2^-22 max(|a|, 2^-14) max(|b|, 2^-14); a zero stays one
//
// and the sums of the two kinds of products are kept apart (split and scaling as in Ootomo and Yokota, "Recovering single precision
// accuracy from Tensor Cores while surpassing the FP32 theoretical peak performance", 2022).  v_mfma_f32_16x16x4_f32 takes 32 cycles for
// an eighth of the products that v_mfma_f32_16x16x32_f16 does in 16: three of the latter are 5.3 times as fast.
//
// What that means for accuracy.  A quarter of the 24-bit values lose their last bit, and lo_a lo_b is dropped; the sums are rounded
// 32 products at a time instead of four.  Error against 64 bits, relative to the result (2-norms), fp32 instruction / split, activations
// N(0,1), weights N(0, 0.02^2): K = 32 1.02e-7 / 0.92e-7, K = 96 1.8e-7 / 1.0e-7, K = 768 5.0e-7 / 2.0e-7, K = 3072 1.0e-6 / 2.0e-7; GELU of
// N(0,1) or values of one sign the same or better.  It is not nearer where a result hangs on one product (a weight that is a unit matrix gives a
// quarter of its inputs back with another last bit), or on elements below 2^-14 beside larger ones whose products vanish: those are
// held to 2^-36 instead of 24 bits.
#pragma once

#include "common.h"

namespace ttmi {

// The window of a row's largest absolute value in which the halves hold a product to fp32 accuracy.  Above, lo could
// overflow; below, the subnormal step of lo, 2^-24 / 2^16, comes near 2^-24 of the row's largest value.  Rows of a weight that are outside
// (and not all zero) are scaled by a power of two on their way into the halves, which their flag holds; rows with an infinity and rows of
// the other operand that are outside are formed again with the fp32 instruction.
constexpr float kSplitScale = 65536.f, kSplitLargest = 2048.f, kSplitSmallest = 0x1p-13f;
constexpr int kSplitOutside = 1 << 30;  // beside the powers of two that rows of packed weights are scaled by
__device__ __forceinline__ bool split_outside(float largest) { return (largest != 0.f) & !((largest >= kSplitSmallest) & (largest < kSplitLargest)); }

#if defined(__HIP_DEVICE_COMPILE__)
typedef _Float16 halfx2 __attribute__((ext_vector_type(2)));
typedef float floatx2 __attribute__((ext_vector_type(2)));
// two values, rounded to fp16 / what the rounding left of them
__device__ __forceinline__ uint32_t split_hi(float a, float b) { return __builtin_bit_cast(uint32_t, __builtin_convertvector((floatx2{a, b}), halfx2)); }
__device__ __forceinline__ uint32_t split_lo(uint32_t hi, float a, float b) {
  const halfx2 h = __builtin_bit_cast(halfx2, hi);
  halfx2 l;
  l[0] = (_Float16)__builtin_fmaf((float)h[0], -kSplitScale, a * kSplitScale);
  l[1] = (_Float16)__builtin_fmaf((float)h[1], -kSplitScale, b * kSplitScale);
  return __builtin_bit_cast(uint32_t, l);
}
// (an instruction: fmaxf would quiet signalling NaNs first, one more per value)
__device__ __forceinline__ void split_max(float& largest, float a, float b) { asm("v_max3_f32 %0, |%1|, |%2|, %0" : "+v"(largest) : "v"(a), "v"(b)); }
#else
__device__ __forceinline__ uint32_t split_hi(float, float) { return 0; }
__device__ __forceinline__ uint32_t split_lo(uint32_t, float, float) { return 0; }
__device__ __forceinline__ void split_max(float&, float, float) {}
#endif

}  // namespace ttmi
