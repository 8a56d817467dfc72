// FP32 operands as three bfloat16 parts for the BF16 matrix pipe (the identity and its error are
// described at the top of gemm_kernel.hpp).
#pragma once

#include "cta_common.hpp"

namespace cta {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

__device__ __forceinline__ f32x16 mfma_bf16(bf16x8 a, bf16x8 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

// The six products of parts, smallest first: a's part and b's part.
constexpr int kSplitA[6] = {0, 1, 2, 0, 1, 0};
constexpr int kSplitB[6] = {2, 1, 0, 1, 0, 0};

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t pack_bf16(float lo, float hi) {
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  const f32x2 v = {lo, hi};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
}

// A float is a multiple of 2^-149, so three bfloat16 parts of x itself (multiples of 2^-133) would
// lose low bits of |x| < 2^-109.  x 2^24 loses none, whatever x: its last part is zero or at least
// 2^-125, a normal number.  Products of scaled operands are taken back by the factor in FP32, which
// is exact.  Scaled values round to infinity from 2^103 on.
constexpr float kSplitScale = 0x1p24f, kSplitUnscale = 0x1p-24f;

// x 2^24 (SCALE; else x) = p[0] + p[1] + p[2], each part rounded to nearest.  The differences are
// exact; the last part holds what is left, in at most 8 bits.  Eleven instructions a pair (and two
// for the scale), all of which run beside the MFMAs (up to five for each 32-cycle MFMA).
// v_dot2_f32_bf16, which subtracts a packed half without unpacking it (seven instructions a
// pair), shares the matrix pipe: measured, each one held it for about ten cycles.
template <bool SCALE = false>
__device__ __forceinline__ void split_bf16(const float (&x)[8], bf16x8 (&p)[3]) {
#pragma clang fp contract(off)  // fused into the subtraction, the scale keeps x alive beside x 2^24
  u32x4 w[3];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    float lo = SCALE ? x[2 * e] * kSplitScale : x[2 * e];
    float hi = SCALE ? x[2 * e + 1] * kSplitScale : x[2 * e + 1];
    w[0][e] = pack_bf16(lo, hi);
    lo -= __uint_as_float(w[0][e] << 16);
    hi -= __uint_as_float(w[0][e] & 0xffff0000u);
    w[1][e] = pack_bf16(lo, hi);
    lo -= __uint_as_float(w[1][e] << 16);
    hi -= __uint_as_float(w[1][e] & 0xffff0000u);
    w[2][e] = pack_bf16(lo, hi);
  }
#pragma unroll
  for (int q = 0; q < 3; ++q) p[q] = __builtin_bit_cast(bf16x8, w[q]);
}

// Whether any of 16 sums is infinite or NaN: an operand was, or was too large to scale, or the
// scaled sum overflowed.
__device__ __forceinline__ bool not_finite(const f32x16& s) {
  float z = 0.0f;  // 0, or NaN: one instruction a value, no mask to keep
#pragma unroll
  for (int r = 0; r < 16; ++r) z = fmaf(s[r], 0.0f, z);
  return z != 0.0f;
}

// Largest magnitude of the scaled operand of the scores whose other operand goes without the scale
// (q of k in the forward, k of q in the backward): what the other's parts lack, at most 2^-134 an
// element, moves an exponent by less than 128 x 2^-134 x 2^85 x log2(e) / sqrt(32) < 2^-42.
constexpr float kMaxScoreFactor = 0x1p85f;

}  // namespace cta
