// Pieces of 16-bit rows as floats and as 8-bit codes: what every kernel that quantises activations does alike.
#pragma once

#include "common.h"

namespace mi355q {

// the 8 values of a piece of 16-bit elements
template <int DT>
__device__ __forceinline__ void unpack8(const u4& v, float* f) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    f[2 * i] = Elem<DT>::to_f32((uint16_t)(v[i] & 0xffffu));
    f[2 * i + 1] = Elem<DT>::to_f32((uint16_t)(v[i] >> 16));
  }
}

// 8 floats (already within +-448) -> 8 e4m3fn codes, round to nearest even
__device__ __forceinline__ u2 to_fp8x8(const float* y) {
  u2 r;
  int w0 = 0, w1 = 0;
  w0 = __builtin_amdgcn_cvt_pk_fp8_f32(y[0], y[1], w0, false);
  w0 = __builtin_amdgcn_cvt_pk_fp8_f32(y[2], y[3], w0, true);
  w1 = __builtin_amdgcn_cvt_pk_fp8_f32(y[4], y[5], w1, false);
  w1 = __builtin_amdgcn_cvt_pk_fp8_f32(y[6], y[7], w1, true);
  r.x = (uint32_t)w0;
  r.y = (uint32_t)w1;
  return r;
}

__device__ __forceinline__ int8_t sat_rne_s8(float y) {
  y = __builtin_rintf(y);                       // round half to even
  y = fminf(fmaxf(y, -128.0f), 127.0f);
  return (int8_t)(int)y;
}
__device__ __forceinline__ u2 pack_s8x8(const float* y) {
  uint32_t q[2] = {0u, 0u};
#pragma unroll
  for (int e = 0; e < 8; ++e) q[e >> 2] |= ((uint32_t)(uint8_t)sat_rne_s8(y[e])) << (8 * (e & 3));
  return (u2){q[0], q[1]};
}

// 8 values of a row with the largest magnitude mx -> codes of the per-token int8 quantiser, and the row's scale
struct RowInt8 {
  float scale, inv;
  __device__ __forceinline__ explicit RowInt8(float mx) : scale(mx / 127.0f), inv(127.0f / mx) {}   // (inv: inf for an all-zero row)
  __device__ __forceinline__ u2 codes(float* y) const {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      y[e] *= inv;
      if (y[e] != y[e]) y[e] = 0.f;             // 0 * inf
    }
    return pack_s8x8(y);
  }
};
// ... of the per-token fp8 quantiser
struct RowFp8 {
  float scale;
  SharedDivisor by;
  __device__ __forceinline__ explicit RowFp8(float mx) : scale(fmaxf(mx, 1e-10f) / FP8_MAX), by(scale) {}
  __device__ __forceinline__ u2 codes(float* y) const {
#pragma unroll
    for (int e = 0; e < 8; ++e) y[e] = clamp448(by.div(y[e]));
    return to_fp8x8(y);
  }
};
// ... of the static int8 quantiser with one scale per column: the reciprocals are rounded to the type of the inputs
template <int DT>
__device__ __forceinline__ u2 static_int8_codes(float* y, const float* s) {
#pragma unroll
  for (int e = 0; e < 8; ++e) y[e] *= Elem<DT>::to_f32(Elem<DT>::from_f32(1.0f / s[e]));
  return pack_s8x8(y);
}

}  // namespace mi355q
