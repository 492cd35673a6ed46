// MX (OCP Microscaling v1.0) element and scale encoding, shared by the
// quantisation kernel (mx.hip) and the norm that quantises its own output
// rows (norm.hip): blocks of 32 elements share one E8M0 scale X =
// 2^(floor(log2 amax) - emax_elem) (byte = exponent + 127, clamped to
// [0, 254]; an all-zero block gets byte 0); each element is v / X rounded to
// nearest-even in the element format and saturated to its largest finite
// magnitude (E4M3 448, E2M1 6).
#pragma once
#include "common.h"
#include "mkd_internal.h"

namespace mkd {

template <int FMT>
struct MxSpec;
template <>
struct MxSpec<MX_E4M3> {
  static constexpr int EMAX = 8, BPL = 32, HW = 0;
};
template <>
struct MxSpec<MX_E2M1> {
  static constexpr int MB = 1, EB = 2, BIAS = 1, EMIN = 0, EMAX = 2, BPL = 16, HW = 4;
  static constexpr float VMAX = 6.0f;
};

// floor(log2(a)) for finite a > 0, fp32 subnormals included.
MKD_DEV int floor_log2_pos(float a) {
  const uint32_t b = __float_as_uint(a);
  const int e = (int)((b >> 23) & 0xffu);
  if (e) return e - 127;
  return (31 - __clz(b & 0x7fffffu)) - 149;
}

// E2M1 code of v (already divided by the block scale): RNE, saturating (NaN: 6).
MKD_DEV uint32_t mx_encode_e2m1(float v) {
  using S = MxSpec<MX_E2M1>;
  const uint32_t sign = __float_as_uint(v) >> 31;
  const float a = fabsf(v);
  const int e = a > 0.f ? max(floor_log2_pos(a), S::EMIN) : S::EMIN;
  float q = ldexpf(rintf(ldexpf(a, S::MB - e)), e - S::MB);  // exact scalings, RNE
  q = fminf(q, S::VMAX);
  uint32_t mag = 0;
  if (q > 0.f) {
    const int qe = floor_log2_pos(q);
    if (qe >= S::EMIN)
      mag = ((uint32_t)(qe + S::BIAS) << S::MB) |
            ((__float_as_uint(q) >> (23 - S::MB)) & ((1u << S::MB) - 1u));
    else
      mag = (uint32_t)ldexpf(q, S::MB - S::EMIN);            // subnormal: q / 2^(EMIN-MB)
  }
  return (sign << (S::EB + S::MB)) | mag;
}

// Four E4M3 codes (v[0] lowest byte) by gfx950's v_cvt_pk_fp8_f32: round to nearest
// even, subnormals included; the magnitude is clamped to 448 first, so nothing
// overflows and a NaN becomes +-448 (every code, tie and neighbour of a tie against
// the oracle: tests/test_gpu_mx.py).  ~3 instructions per value, ~25 in integer math.
MKD_DEV float mx_clamp448(float v) { return __builtin_copysignf(fminf(fabsf(v), 448.0f), v); }
MKD_DEV uint32_t mx_encode4_e4m3(float a, float b, float c, float d) {
  int o = __builtin_amdgcn_cvt_pk_fp8_f32(mx_clamp448(a), mx_clamp448(b), 0, false);
  o = __builtin_amdgcn_cvt_pk_fp8_f32(mx_clamp448(c), mx_clamp448(d), o, true);
  return (uint32_t)o;
}

template <int FMT>
MKD_DEV uint32_t mx_scale_byte(float amax) {
  if (!(amax > 0.f)) return 0u;
  const int e = floor_log2_pos(amax) - MxSpec<FMT>::EMAX + 127;
  return (uint32_t)min(max(e, 0), 254);
}

// MXFP8 of eight consecutive values by one of the four consecutive lanes holding a
// 32-element block: the eight codes, and the block's scale byte (the same in all four).
MKD_DEV uint2 mx_quant8_e4m3(const float (&v)[8], uint32_t& scale) {
  float amax = 0.f;
#pragma unroll
  for (int j = 0; j < 8; ++j) amax = fmaxf(amax, fabsf(v[j]));
  amax = fmaxf(amax, __shfl_xor(amax, 1, 64));
  amax = fmaxf(amax, __shfl_xor(amax, 2, 64));
  scale = mx_scale_byte<MX_E4M3>(amax);
  const int sh = 127 - (int)scale;
  float q[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) q[j] = ldexpf(v[j], sh);
  return uint2{mx_encode4_e4m3(q[0], q[1], q[2], q[3]), mx_encode4_e4m3(q[4], q[5], q[6], q[7])};
}

// MXFP8 rows: item `it` quantises eight elements of a row (four consecutive items,
// lanes of one wave, per 32-element block; K % 32 == 0); blocks past K are zeros.
template <bool XF32>
MKD_DEV void mx_quant_rows_item(const void* x, long long it, int K, long long ldx, uint8_t* codes, uint8_t* scales,
                                int K_pad) {
  const int per = K_pad / 8;
  const long long r = it / per;
  const int i = (int)(it % per) * 8;
  float v[8];
  if (i >= K) {
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = 0.f;
  } else if (XF32) {
    const float* p = static_cast<const float*>(x) + r * ldx + i;
    const f32x4_t a = *reinterpret_cast<const f32x4_t*>(p), b = *reinterpret_cast<const f32x4_t*>(p + 4);
#pragma unroll
    for (int j = 0; j < 4; ++j) { v[j] = a[j]; v[4 + j] = b[j]; }
  } else {
    const u32x4_t t = ld16(static_cast<const uint16_t*>(x) + r * ldx + i);
#pragma unroll
    for (int j = 0; j < 4; ++j) { v[2 * j] = bf_lo(t[j]); v[2 * j + 1] = bf_hi(t[j]); }
  }
  uint32_t sb;
  const uint2 c = mx_quant8_e4m3(v, sb);
  *reinterpret_cast<uint2*>(codes + r * K_pad + i) = c;
  if ((i & 31) == 0) scales[r * (K_pad / 32) + i / 32] = (uint8_t)sb;
}

}  // namespace mkd
