// Packed codes -> matrix-core operands, shared by the quantised GEMMs.
#pragma once
#include "common.h"

// byte I of v as float.  Written as the instruction: the compiler otherwise extracts
// bytes 1 and 2 with a v_bfe_u32 first.
template <int I>
__device__ __forceinline__ float ubyte_f(uint32_t v) {
  float f;
  if (I == 0) asm("v_cvt_f32_ubyte0 %0, %1" : "=v"(f) : "v"(v));
  if (I == 1) asm("v_cvt_f32_ubyte1 %0, %1" : "=v"(f) : "v"(v));
  if (I == 2) asm("v_cvt_f32_ubyte2 %0, %1" : "=v"(f) : "v"(v));
  if (I == 3) asm("v_cvt_f32_ubyte3 %0, %1" : "=v"(f) : "v"(v));
  return f;
}

// The eight codes in `v0` (4 bits; 8 bits: `v0`, `v1`) as the bf16x8 B operand of one MFMA step:
// bf16(fma(s, q, b))
template <int BITS>
__device__ __forceinline__ bf16x8_t dequant_words8(uint32_t v0, uint32_t v1, float s, float b) {
  uint4 o;
  if (BITS == 4) {
    const uint32_t ev = v0 & 0x0f0f0f0fu, od = (v0 >> 4) & 0x0f0f0f0fu;
    const float e0 = ubyte_f<0>(ev), e1 = ubyte_f<1>(ev), e2 = ubyte_f<2>(ev), e3 = ubyte_f<3>(ev);
    const float o0 = ubyte_f<0>(od), o1 = ubyte_f<1>(od), o2 = ubyte_f<2>(od), o3 = ubyte_f<3>(od);
    o.x = pack_bf2(fmaf(s, e0, b), fmaf(s, o0, b));
    o.y = pack_bf2(fmaf(s, e1, b), fmaf(s, o1, b));
    o.z = pack_bf2(fmaf(s, e2, b), fmaf(s, o2, b));
    o.w = pack_bf2(fmaf(s, e3, b), fmaf(s, o3, b));
  } else {
    o.x = pack_bf2(fmaf(s, ubyte_f<0>(v0), b), fmaf(s, ubyte_f<1>(v0), b));
    o.y = pack_bf2(fmaf(s, ubyte_f<2>(v0), b), fmaf(s, ubyte_f<3>(v0), b));
    o.z = pack_bf2(fmaf(s, ubyte_f<0>(v1), b), fmaf(s, ubyte_f<1>(v1), b));
    o.w = pack_bf2(fmaf(s, ubyte_f<2>(v1), b), fmaf(s, ubyte_f<3>(v1), b));
  }
  return __builtin_bit_cast(bf16x8_t, o);
}
