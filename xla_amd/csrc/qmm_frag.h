// MFMA operand fragments shared by the weight-only kernels: int8 / packed int4 weights -> 8 elements
// of x's dtype (bf16 or f16), the 16x16x32 MFMA on such fragments, and a fragment of ones.
#pragma once
#include "qmm_common.h"

namespace qmm_frag {

__device__ __forceinline__ uint32_t pack_hi16(float lo, float hi) {
  // {bf16(lo), bf16(hi)} by truncation: exact for integers of magnitude <= 256.
  return __builtin_amdgcn_perm(__float_as_uint(hi), __float_as_uint(lo), 0x07060302u);
}

__device__ __forceinline__ uint32_t pack_f16(float lo, float hi) {
  typedef _Float16 h2 __attribute__((ext_vector_type(2)));
  h2 v = __builtin_bit_cast(h2, __builtin_amdgcn_cvt_pkrtz(lo, hi));  // exact for small integers
  return __builtin_bit_cast(uint32_t, v);
}

// 8 int8 weights (two dwords) -> 8 elements of the x dtype.
template <int XT>
__device__ __forceinline__ i32x4 cvt_w8(uint32_t d0, uint32_t d1) {
  float f[8];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    f[i] = (float)(int8_t)(d0 >> (8 * i));
    f[4 + i] = (float)(int8_t)(d1 >> (8 * i));
  }
  i32x4 o;
  if constexpr (XT == XLA_AMD_DT_BF16) {
    o[0] = pack_hi16(f[0], f[1]); o[1] = pack_hi16(f[2], f[3]);
    o[2] = pack_hi16(f[4], f[5]); o[3] = pack_hi16(f[6], f[7]);
  } else {
    o[0] = pack_f16(f[0], f[1]); o[1] = pack_f16(f[2], f[3]);
    o[2] = pack_f16(f[4], f[5]); o[3] = pack_f16(f[6], f[7]);
  }
  return o;
}

// Two int8 weights (the low or the high half of a dword) -> two elements of the x dtype: a quarter of cvt_w8.
template <int XT, class HiC>
__device__ __forceinline__ uint32_t cvt_w2(uint32_t d, HiC) {
  constexpr int sh = HiC::value ? 16 : 0;
  const float lo = (float)(int8_t)(d >> sh), hi = (float)(int8_t)(d >> (sh + 8));
  if constexpr (XT == XLA_AMD_DT_BF16) return pack_hi16(lo, hi);
  else return pack_f16(lo, hi);
}

// An int4 weight w becomes an element of the x dtype by setting mantissa bits alone, u = w + 8 in 0..15: 1 + u/16 in bf16,
// 16 + u in f16.  The caller undoes the affine map with the exact x sum:
//   sum w x = kInt4Factor (sum a x - kInt4Offset sum x)
// In bf16 the factor may wait until behind the rounding of a dot product, a power of two commutes with it (down to 2^-126).
// Not so in f16: a sixteenth of a dot product below 2^-10 is subnormal and would lose up to four of its bits, and one of
// more than 65504 would not overflow.  (bf16 keeps 1 + u/16: sums of a x sixteen times as large would overflow at
// x = 2^121.)
template <int XT> constexpr float kInt4Factor = XT == XLA_AMD_DT_BF16 ? 16.0f : 1.0f;
template <int XT> constexpr float kInt4Offset = XT == XLA_AMD_DT_BF16 ? 1.5f : 24.0f;
template <int XT> constexpr uint32_t kInt4Bits = XT == XLA_AMD_DT_BF16 ? 0x3F803F80u : 0x4C004C00u;  // two elements of u = 0 ...
template <int XT> constexpr uint32_t kInt4Mask = XT == XLA_AMD_DT_BF16 ? 0x00780078u : 0x03C003C0u;  // ... and the bits u sets

// 8 packed int4 weights (one dword, nibble j = column P[j], biased by 8) -> 8 elements.
template <int XT>
__device__ __forceinline__ i32x4 cvt_w4(uint32_t d) {
  i32x4 o;
  constexpr uint32_t mask = kInt4Mask<XT>, zero = kInt4Bits<XT>;
  if constexpr (XT == XLA_AMD_DT_BF16) {
    o[0] = ((d << 3) & mask) | zero;
    o[1] = ((d >> 1) & mask) | zero;
    o[2] = ((d >> 5) & mask) | zero;
    o[3] = ((d >> 9) & mask) | zero;
  } else {
    o[0] = ((d << 6) & mask) | zero;
    o[1] = ((d << 2) & mask) | zero;
    o[2] = ((d >> 2) & mask) | zero;
    o[3] = ((d >> 6) & mask) | zero;
  }
  return o;
}

template <int XT>
__device__ __forceinline__ f32x4 mfma16(i32x4 a, i32x4 b, f32x4 c) {
  if constexpr (XT == XLA_AMD_DT_BF16)
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                   __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a),
                                                  __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}

template <int XT> __device__ __forceinline__ i32x4 ones_frag() {
  uint32_t one2 = XT == XLA_AMD_DT_BF16 ? 0x3F803F80u : 0x3C003C00u;
  i32x4 o = {(int)one2, (int)one2, (int)one2, (int)one2};
  return o;
}

}  // namespace qmm_frag
