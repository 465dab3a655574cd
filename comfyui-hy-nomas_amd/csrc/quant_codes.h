// The activation quantizer's arithmetic on 8 values of a lane, shared by the quantization kernels and the skinny linear.
#pragma once

#include "hn_common.h"

namespace hn {

// 8 consecutive input values of one lane, loaded as 16 (2-byte types) or 32 (fp32) bytes.
template <int DT>
struct Chunk8 {
  uint4 v[DT == HN_DTYPE_F32 ? 2 : 1];
  __device__ __forceinline__ void load(const char* p) {
    v[0] = ld_nt16(p);
    if constexpr (DT == HN_DTYPE_F32) v[1] = ld_nt16(p + 16);
  }
  __device__ __forceinline__ void widen(float* f) const {
    if constexpr (DT == HN_DTYPE_F32) {
      f[0] = __uint_as_float(v[0].x); f[1] = __uint_as_float(v[0].y);
      f[2] = __uint_as_float(v[0].z); f[3] = __uint_as_float(v[0].w);
      f[4] = __uint_as_float(v[1].x); f[5] = __uint_as_float(v[1].y);
      f[6] = __uint_as_float(v[1].z); f[7] = __uint_as_float(v[1].w);
    } else {
      In<DT>::widen8(v[0], f);
    }
  }
  static constexpr int kElemBytes = DT == HN_DTYPE_F32 ? 4 : 2;
};

// Codes of 8 values with one scale; returns them packed in 8 bytes.  FAST: bf16-valued inputs in a group
// with FastQuot<KIND>::ok(peak) -- the exact fast quotient, and (int8) no clamp since |x| <= peak.  Otherwise an
// IEEE division and the clamped rounding.
template <int KIND, int ROUND, bool FAST>
__device__ __forceinline__ uint2 encode8(const float* f, float scale) {
  int c[8];
  if constexpr (FAST && KIND == HN_KIND_FP8) {
    const typename FastQuot<KIND>::Div div(scale);
    float y[8];
#pragma unroll
    for (int i = 0; i < 8; i++) y[i] = div(f[i]);
    return make_uint2(e4m3_pack4_hw(y[0], y[1], y[2], y[3]), e4m3_pack4_hw(y[4], y[5], y[6], y[7]));
  } else if constexpr (FAST) {
    const typename FastQuot<KIND>::Div div(scale);
#pragma unroll
    for (int i = 0; i < 8; i++) {
      const float y = div(f[i]);
      if constexpr (ROUND == HN_ROUND_HALF_EVEN) c[i] = rne_code_bits(y);  // low byte only: packed below
      else c[i] = round_half_away_i8_inrange(y);
    }
  } else {
#pragma unroll
    for (int i = 0; i < 8; i++) {
      const float y = f[i] / scale;
      if constexpr (KIND == HN_KIND_FP8) c[i] = (int)e4m3_encode(y);
      else c[i] = round_i8<ROUND>(y);
    }
  }
  return make_uint2(pack4_i8(c[0], c[1], c[2], c[3]), pack4_i8(c[4], c[5], c[6], c[7]));
}

// Scale and codes of one group from its absmax `peak` (non-negative, NaN-free).  bf16 inputs in a group
// with FastQuot<KIND>::ok(peak) use the fast exact quotients (hn_common.h); other groups and inputs divide.
template <int DT, int KIND, int ROUND>
__device__ __forceinline__ uint2 encode8_group(const float* f, float peak, float& scale) {
  if constexpr (DT == HN_DTYPE_BF16) {
    if (__builtin_expect(FastQuot<KIND>::ok(peak), 1)) {
      scale = KIND == HN_KIND_INT8 ? int8_scale_fast(peak) : fp8_scale_fast(peak);
      return encode8<KIND, ROUND, true>(f, scale);
    }
  }
  scale = KIND == HN_KIND_INT8 ? int8_scale(peak) : fp8_scale(peak);
  return encode8<KIND, ROUND, false>(f, scale);
}

}  // namespace hn
