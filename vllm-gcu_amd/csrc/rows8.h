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

// Rounded to even and saturated to int8, in the low byte: the sum with 1.5 * 2^23 has no bits for a fraction.  (NaN: -128.)
__device__ __forceinline__ uint32_t rne_s8_byte(float y) { return bitcast<uint32_t>(__builtin_amdgcn_fmed3f(y, -128.0f, 127.0f) + 12582912.0f); }
__device__ __forceinline__ int8_t sat_rne_s8(float y) { return (int8_t)rne_s8_byte(y); }
// the low bytes of four words
__device__ __forceinline__ uint32_t low_bytes(uint32_t a, uint32_t b, uint32_t c, uint32_t d) {
  return __builtin_amdgcn_perm(__builtin_amdgcn_perm(d, c, 0x0c0c0400u), __builtin_amdgcn_perm(b, a, 0x0c0c0400u), 0x05040100u);
}
__device__ __forceinline__ u2 pack_s8x8(const float* y) {
  return (u2){low_bytes(rne_s8_byte(y[0]), rne_s8_byte(y[1]), rne_s8_byte(y[2]), rne_s8_byte(y[3])),
              low_bytes(rne_s8_byte(y[4]), rne_s8_byte(y[5]), rne_s8_byte(y[6]), rne_s8_byte(y[7]))};
}

// 8 values of a row with the largest magnitude mx -> codes of the per-token int8 quantiser, and the row's scale
struct RowInt8 {
  float scale, inv;
  __device__ __forceinline__ explicit RowInt8(float mx) : scale(mx / 127.0f), inv(127.0f / mx) {}   // (inv: inf for an all-zero row)
  // (NaN, also of 0 * inf: 0, which the conversion makes of it by itself; it saturates as well)
  __device__ __forceinline__ uint32_t code(float y) const {
    int i;
    asm("v_cvt_i32_f32 %0, %1" : "=v"(i) : "v"(__builtin_rintf(y * inv)));
    return (uint32_t)min(max(i, -128), 127);
  }
  __device__ __forceinline__ u2 codes(const float* y) const {
    return (u2){low_bytes(code(y[0]), code(y[1]), code(y[2]), code(y[3])), low_bytes(code(y[4]), code(y[5]), code(y[6]), code(y[7]))};
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
