// The linear layer's dynamic activation quantisation of one 128-column group
// (shared by the quantisation kernel and the small-M linear kernel, which
// quantises its own activations).
#pragma once

#include "fp8_common.h"

namespace nvamd {

constexpr int kFp8Block = 128;  // the reference's BLOCK_SIZE (fp8_linear.py:8)

template <bool F16_IN>
__device__ __forceinline__ float in_to_f32(uint32_t bits16) {
  if constexpr (F16_IN) return (float)__builtin_bit_cast(_Float16, (uint16_t)bits16);
  return bf16_bits_to_f32(bits16);
}

// Eight consecutive values of a group held by one of its 16 lanes (a DPP row)
// -> their E4M3FN bytes and the group's scale: amax / 448, 1 when not > 0
// (IEEE division); byte = E4M3FN(clamp(x / scale)) (IEEE division, RNE).
//
// The division is the cost of this step, so x / scale is taken as a product
// with the group's reciprocal r = RN(1 / scale) and one correction,
// q = x r, q - (q scale - x) r (signed so that -0 stays -0).  The remainder is
// exact where q scale has no bits below 2^-149, and the result is then the
// correctly rounded quotient; at the smallest scales the remainder of a
// quotient below 1 loses its last bits, which can move a result that lies
// halfway between two fp32 values, not its E4M3 byte.  The bytes equal those of
// the division for every pair of significands of x and amax, in bf16 and fp16,
// at scales of both ends of the range too (a test).  A group with a non-finite
// value or a scale outside 2^+-100 takes the divisions instead.
template <bool F16_IN>
__device__ __forceinline__ u32x2 quant_group8(u32x4 w, float& scale) {
  const uint32_t d[4] = {w.x, w.y, w.z, w.w};
  float v[8];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    v[2 * i] = in_to_f32<F16_IN>(d[i] & 0xFFFFu);
    v[2 * i + 1] = in_to_f32<F16_IN>(d[i] >> 16);
  }
  float amax = 0.f;
#pragma unroll
  for (int i = 0; i < 8; ++i) amax = fmaxf(amax, __builtin_fabsf(v[i]));  // NaN operands are skipped
  amax = row16_max(amax);  // the group's 16 lanes are one DPP row
  scale = amax / 448.0f;   // correctly rounded fp32 division
  scale = scale > 0.f ? scale : 1.0f;
  bool odd = !(scale >= 0x1p-100f && scale <= 0x1p100f);
#pragma unroll
  for (int i = 0; i < 8; ++i) odd |= v[i] != v[i];
  float y[8];
  if (wave_any(odd)) {
#pragma unroll
    for (int i = 0; i < 8; ++i) y[i] = v[i] / scale;
    return u32x2{f32x4_to_fp8x4(y[0], y[1], y[2], y[3]), f32x4_to_fp8x4(y[4], y[5], y[6], y[7])};
  }
  const float r = 1.0f / scale;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const float q = v[i] * r;
    y[i] = __builtin_fmaf(-__builtin_fmaf(q, scale, -v[i]), r, q);
  }
  // |y| <= 448 (1 + 2^-23): nothing saturates, so no clamp before the conversion
  u32x2 o;
  int b = __builtin_amdgcn_cvt_pk_fp8_f32(y[0], y[1], 0, false);
  o.x = (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(y[2], y[3], b, true);
  b = __builtin_amdgcn_cvt_pk_fp8_f32(y[4], y[5], 0, false);
  o.y = (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(y[6], y[7], b, true);
  return o;
}

// The scale as the GEMM multiplies it: bf16 (RNE).
__device__ __forceinline__ uint32_t scale_bf16_bits(float scale) { return pack_bf16x2(scale, 0.f) & 0xFFFFu; }

}  // namespace nvamd
