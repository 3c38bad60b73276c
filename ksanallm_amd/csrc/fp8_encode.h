// e4m3 codes of a quantization group of 16-bit (or, kF32, fp32) values: scale and codes as every quantizer here forms them.
#pragma once

#include "exact_div.h"
#include "ksq_common.h"

namespace ksq {

__device__ __forceinline__ uint32_t cvt2_e4m3(float a, float b, uint32_t old, bool hi) {
  // v_cvt_pk_fp8_f32 rounds to nearest even; inputs are clamped to +-448 first so the result never leaves the
  // finite range (NaN passes through and encodes as NaN).
  float ca = fminf(fmaxf(a, -448.0f), 448.0f);
  float cb = fminf(fmaxf(b, -448.0f), 448.0f);
  ca = (a != a) ? a : ca;
  cb = (b != b) ? b : cb;
  return hi ? static_cast<uint32_t>(__builtin_amdgcn_cvt_pk_fp8_f32(ca, cb, static_cast<int>(old), true))
            : static_cast<uint32_t>(__builtin_amdgcn_cvt_pk_fp8_f32(ca, cb, static_cast<int>(old), false));
}

// two quotients that are known to lie within +-448 * (1 + 2^-23), or NaN: no clamp in front of the conversion
__device__ __forceinline__ uint32_t cvt2_e4m3_in_range(float a, float b, uint32_t old, bool hi) {
  return hi ? static_cast<uint32_t>(__builtin_amdgcn_cvt_pk_fp8_f32(a, b, static_cast<int>(old), true))
            : static_cast<uint32_t>(__builtin_amdgcn_cvt_pk_fp8_f32(a, b, static_cast<int>(old), false));
}

// max(amax, 1e-10) / 448, correctly rounded, by reciprocal and correction (amax, with its floor applied, has at most 11
// significant bits, or is the floor 1e-10, whose quotient is a constant)
template <bool kF32>
__device__ __forceinline__ float fp8_group_scale(float amax) {
  constexpr float y448 = 1.0f / 448.0f;
  const float q0 = amax * y448;
  const float r = __builtin_fmaf(-q0, 448.0f, amax);
  float scale = __builtin_fmaf(r, y448, q0);
  scale = amax == 1e-10f ? 1e-10f / 448.0f : scale;
  return (!kF32 && amax >= 0x1p-60f && amax <= 0x1p100f) ? scale : amax / 448.0f;
}

// four values of a group whose scale `div` holds -> four codes
template <bool kF32>
__device__ __forceinline__ uint32_t fp8_encode4(const ExactDiv& div, const float* v) {
  uint32_t o = 0;
  if (!kF32 && div.fast) {
    // every |v| <= amax (an infinite v makes amax, hence the scale, infinite: not this branch), so the quotients stay
    // within 448 * (1 + 2^-23), which the conversion rounds to 448 by itself
    o = cvt2_e4m3_in_range(div(v[0]), div(v[1]), o, false);
    return cvt2_e4m3_in_range(div(v[2]), div(v[3]), o, true);
  }
  o = cvt2_e4m3(v[0] / div.s, v[1] / div.s, o, false);
  return cvt2_e4m3(v[2] / div.s, v[3] / div.s, o, true);
}

}  // namespace ksq
