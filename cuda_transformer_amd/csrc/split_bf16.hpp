// FP32 operands as three bfloat16 parts for the BF16 matrix pipe (the identity and its error are
// described at the top of gemm_kernel.hpp).
#pragma once

#include "cta_common.hpp"

namespace cta {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x8 __attribute__((ext_vector_type(8)));

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

// x = p[0] + p[1] + p[2], each part rounded to nearest.  The differences are exact; the last
// part holds what is left in at most 8 bits (above 2^-109).  Eleven instructions a pair, all of
// which run beside the MFMAs (up to five for each 32-cycle MFMA).  v_dot2_f32_bf16, which
// subtracts a packed half without unpacking it (seven instructions a pair), shares the matrix
// pipe: measured, each one held it for about ten cycles.
__device__ __forceinline__ void split_bf16(const float (&x)[8], bf16x8 (&p)[3]) {
  u32x4 w[3];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    float lo = x[2 * e], hi = x[2 * e + 1];
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

// Whether a sum of split products may differ from FP32 arithmetic by more than rounding: it is
// infinite or NaN (an operand was, or rounded to infinity), or nonzero below 2^-100 (operands
// may have been too small for their low parts).  With u = 2 |bits| and T = 2^-100's, the fine
// range [T, inf) is one unsigned comparison; exact zeros fail it too and are let off in the
// second look, which ordinary tiles never reach.
__device__ __forceinline__ bool split_suspect(const f32x16& s) {
  constexpr uint32_t T = 27u << 24, kInf = 255u << 24;
  bool any = false;
#pragma unroll
  for (int r = 0; r < 16; ++r) any |= ((__float_as_uint(s[r]) << 1) - T) >= kInf - T;
  if (!__any(any)) return false;
  bool bad = false;
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const uint32_t u = __float_as_uint(s[r]) << 1;
    bad |= u != 0 && u - T >= kInf - T;
  }
  return bad;
}

}  // namespace cta
