// mx_widen.h - weight codes to f16 MFMA operands, in registers.
#pragma once

#include "mx_device.h"
#include "mx_internal.h"

namespace mx {

// INT8 x8 -> f16 x8 (exact): byte b -> half(1024 + (b ^ 0x80)) - 1152.
__device__ __forceinline__ v8h i8x8_to_f16(uint32_t w0, uint32_t w1) {
  const uint32_t x[2] = {w0 ^ 0x80808080u, w1 ^ 0x80808080u};
  v8h out;
#pragma unroll
  for (int t = 0; t < 2; t++) {
    const uint32_t lo = __builtin_amdgcn_perm(0x64646464u, x[t], 0x04010400u);  // b0, b1
    const uint32_t hi = __builtin_amdgcn_perm(0x64646464u, x[t], 0x04030402u);  // b2, b3
    v2h l = __builtin_bit_cast(v2h, lo) - (v2h){(_Float16)1152.0f, (_Float16)1152.0f};
    v2h h = __builtin_bit_cast(v2h, hi) - (v2h){(_Float16)1152.0f, (_Float16)1152.0f};
    out[4 * t] = l[0]; out[4 * t + 1] = l[1]; out[4 * t + 2] = h[0]; out[4 * t + 3] = h[1];
  }
  return out;
}

// INT4 x8 (one dword, low nibble first) -> f16 x8: ((n ^ 8) - 8) * scale,
// rounded once to f16 (PackedNumericKernels.metal:30-33).  Per nibble pair
// (byte i): one v_perm puts byte i of w and of w >> 4 into the two halves,
// one v_bitop3 keeps their low nibbles, flips the sign bit (two's
// complement -> offset 8) and ORs in the 0x6400 exponent (1024 + u), then
// a packed subtract and the packed scale multiply: 17 VALU per dword.
__device__ __forceinline__ v8h i4x8_to_f16(uint32_t w, _Float16 sc) {
  const uint32_t y = w >> 4;
  const v2h off = {(_Float16)1032.0f, (_Float16)1032.0f};
  const v2h s2 = {sc, sc};
  v8h out;
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const uint32_t t = __builtin_amdgcn_perm(y, w, 0x0c000c00u | (uint32_t)i | ((uint32_t)(4 + i) << 16));
    const uint32_t p = ((t ^ 0x00080008u) & 0x000f000fu) | 0x64006400u;
    const v2h q = (__builtin_bit_cast(v2h, p) - off) * s2;
    out[2 * i] = q[0];
    out[2 * i + 1] = q[1];
  }
  return out;
}

template <int BK>
__device__ __forceinline__ v8h fp8x8_to_f16(uint32_t w0, uint32_t w1) {
  const uint32_t w[2] = {w0, w1};
  v8h h;
#pragma unroll
  for (int t = 0; t < 2; t++) {
    v2h lo, hi;
    if (BK == BK_E4M3) {
      lo = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w[t], 1.0f, false);
      hi = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w[t], 1.0f, true);
    } else {
      lo = __builtin_amdgcn_cvt_scalef32_pk_f16_bf8(w[t], 1.0f, false);
      hi = __builtin_amdgcn_cvt_scalef32_pk_f16_bf8(w[t], 1.0f, true);
    }
    h[4 * t] = lo[0]; h[4 * t + 1] = lo[1]; h[4 * t + 2] = hi[0]; h[4 * t + 3] = hi[1];
  }
  return h;
}

// 8 f32 activations as two f16 terms, x = hi + lo with lo = f16(x - hi) (0
// where hi is infinite): the two products keep x to ~2^-22 of its value.
__device__ __forceinline__ void split_f32(v4f a, v4f b, v8h& hi, v8h& lo) {
#pragma unroll
  for (int t = 0; t < 8; t++) {
    const float x = t < 4 ? a[t & 3] : b[t & 3];
    const _Float16 h = (_Float16)x;
    hi[t] = h;
    lo[t] = __builtin_isinf((float)h) ? (_Float16)0.0f : (_Float16)(x - (float)h);
  }
}

}  // namespace mx
