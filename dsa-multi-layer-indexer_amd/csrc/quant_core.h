// The fp8 quantisation rule of one 128-element row held by 16 lanes (8
// elements each), shared by the operand-preparation and prefill kernels:
//   scale = max(amax, 1e-6) / 448,  code = e4m3_rne(clamp(x / scale, +-448)),
// the division IEEE fp32 (the reference harness's quantize_e4m3_rowwise,
// K:2969-2974).
#pragma once

#include "dsa_common.h"

namespace dsa {

// Element types of an input: 0 fp32, 1 bf16, 2 fp16.
constexpr int kF32 = 0, kBF16 = 1, kF16 = 2;

template <int DT>
__device__ __forceinline__ float load_elem(const void* p, long i) {
  if constexpr (DT == kF32) return static_cast<const float*>(p)[i];
  const uint16_t v = static_cast<const uint16_t*>(p)[i];
  if constexpr (DT == kBF16) return __uint_as_float((uint32_t)v << 16);
  return (float)__builtin_bit_cast(_Float16, v);
}

// Elements i .. i + 7; WIDE: by 16-byte loads (p 16-byte aligned, i a
// multiple of 8), otherwise one by one.
template <int DT, bool WIDE = true>
__device__ __forceinline__ void load8(const void* p, long i, float* x) {
  if constexpr (!WIDE) {
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] = load_elem<DT>(p, i + e);
  } else if constexpr (DT == kF32) {
    const v4f* f = reinterpret_cast<const v4f*>(static_cast<const float*>(p) + i);
    const v4f a = f[0], b = f[1];
#pragma unroll
    for (int e = 0; e < 4; ++e) x[e] = a[e], x[4 + e] = b[e];
  } else {
    const uint4 v = *reinterpret_cast<const uint4*>(static_cast<const uint16_t*>(p) + i);
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if constexpr (DT == kBF16) {
        x[2 * e] = bf16_lo(w[e]);
        x[2 * e + 1] = bf16_hi(w[e]);
      } else {
        x[2 * e] = (float)__builtin_bit_cast(_Float16, (uint16_t)w[e]);
        x[2 * e + 1] = (float)__builtin_bit_cast(_Float16, (uint16_t)(w[e] >> 16));
      }
    }
  }
}

// Row scale from each lane's 8 elements.  NANS: a NaN among the row's 128
// makes the scale NaN; otherwise it is passed over (its own code is -448's).
template <bool NANS>
__device__ __forceinline__ float row_scale(const float* x) {
  uint32_t am = 0;  // |x| as integer bits: NaN above infinity above every finite value
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const uint32_t a = __float_as_uint(x[e]) & 0x7fffffffu;
    am = max(am, NANS || a <= 0x7f800000u ? a : 0u);
  }
  // max over the 16-lane DPP row: rotations by 1, 2, 4, 8
  am = max(am, dpp_u32<0x121, 0xf>(am, 0u));
  am = max(am, dpp_u32<0x122, 0xf>(am, 0u));
  am = max(am, dpp_u32<0x124, 0xf>(am, 0u));
  am = max(am, dpp_u32<0x128, 0xf>(am, 0u));
  const float amax = __uint_as_float(am);
  return (amax < 1e-6f ? 1e-6f : amax) / 448.f;
}

// The 8 codes (two words, element e in byte e).  The quotients are x times
// the correctly rounded reciprocal, corrected twice by the exact remainder:
// the first correction is within an ulp, the second then rounds correctly
// (Markstein's theorem), at 5 instructions a quotient where the compiler's
// general division takes about 10 and a quarter-rate reciprocal.  A scale
// that is not finite takes the division.
template <bool NANS>
__device__ __forceinline__ v2u_t quant8(const float* x, float scale) {
  float y[8];
  if (scale < INFINITY) {
    const float r = 1.f / scale;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      float q = x[e] * r;
      q = __builtin_fmaf(__builtin_fmaf(-q, scale, x[e]), r, q);
      q = __builtin_fmaf(__builtin_fmaf(-q, scale, x[e]), r, q);
      y[e] = __builtin_copysignf(q, x[e]);  // the corrections turn -0 into +0
    }
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e) y[e] = x[e] / scale;
  }
  int c[4];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    if constexpr (NANS) y[e] = y[e] > 448.f ? 448.f : (y[e] < -448.f ? -448.f : y[e]);  // NaN stays
    else y[e] = fminf(fmaxf(y[e], -448.f), 448.f);
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) c[e] = __builtin_amdgcn_cvt_pk_fp8_f32(y[2 * e], y[2 * e + 1], 0, false);
  v2u_t w;
  w[0] = ((uint32_t)c[0] & 0xffffu) | (uint32_t)c[1] << 16;
  w[1] = ((uint32_t)c[2] & 0xffffu) | (uint32_t)c[3] << 16;
  return w;
}

}  // namespace dsa
