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

// `a` * (half H of v, a float16) + c, in float32 with one rounding
template <int H>
__device__ __forceinline__ float fma_half(float a, uint32_t v, float c) {
  float f;
  if (H == 0) asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel_hi:[0,1,0]" : "=v"(f) : "v"(a), "v"(v), "v"(c));
  if (H == 1) asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel:[0,1,0] op_sel_hi:[0,1,0]" : "=v"(f) : "v"(a), "v"(v), "v"(c));
  return f;
}

// Scale and bias of a group, as the codes want them.
//  4 bits: a code that is masked where it stands, in the low eight bits of a half-word, IS the float16
// q * 2^-24 (bits 0..3) or q * 2^-20 (bits 4..7), a denormal, so that the mixed-precision FMA takes it without
// a conversion: fma(s * 2^24, q * 2^-24, b) is fma(s, q, b), bit for bit.  Eight codes to
// bf16 are 4 masks, a shift, 8 FMAs and 4 packs instead of 3 + 8 conversions + 8 + 4, and vector issue is what the
// GEMMs' loops have too much of: 4-bit pair of 14336x4096 under 2047 rows 425 -> 414 us, under 100 rows 58 -> 52,
// 6144x4096 under 300 rows 49.7 -> 45.8.
//  Scales from 2^104 on have no s * 2^24: operands made from them are not right until large_scales() has made those of such lanes
// once more, from the scale itself.  (A branch behind each operand costs the short GEMM 0.6 %, the prompt GEMM 2 to 12: their loops only
// note that there are some, and the wave's sums are made once more.)
template <int BITS>
struct GroupScale {
  float s, b;
};
template <>
struct GroupScale<4> {
  float s24, s20, b;
};
template <int BITS>
__device__ __forceinline__ GroupScale<BITS> group_scale(float s, float b) {
  GroupScale<BITS> g;
  if constexpr (BITS == 4)
    g.s24 = s * 0x1p24f, g.s20 = s * 0x1p20f;
  else
    g.s = s;
  g.b = b;
  return g;
}
// the largest magnitude so far: one instruction for two scales
__device__ __forceinline__ void note_scales(float& most, float s0, float s1) {
  asm("v_max3_f32 %0, %0, |%1|, |%2|" : "+v"(most) : "v"(s0), "v"(s1));
}
// whether a lane's scale, or the largest that it has noted, is one of those
__device__ __forceinline__ bool any_large(float s) { return __builtin_amdgcn_ballot_w64(fabsf(s) >= 0x1p104f) != 0; }

// One MFMA step's B operand - eight codes as bf16(fma(s, q, b)) - is made in four pieces of one
// register each, in two parts so that a caller can put products between them: piece_codes() masks or converts the
// two codes, piece_value() scales and packs them.  Piece i makes register piece_reg(i) (4 bits: codes 0 1,
// 4 5, 2 3, 6 7, as the words masked for an even piece serve the odd one behind it too).
template <int BITS>
__device__ __forceinline__ constexpr int piece_reg(int i) {
  return BITS == 4 ? (i >> 1) | (i & 1) << 1 : i;
}
struct PieceCodes {
  uint32_t x, y;
};
// `v0` (8 bits: `v0`, `v1`) holds the eight codes
template <int BITS>
__device__ __forceinline__ void piece_codes(PieceCodes& w, int i, uint32_t v0, uint32_t v1) {
  if (BITS == 4) {
    if (i & 1) return;
    const uint32_t v = i < 2 ? v0 : v0 >> 8;
    w.x = v & 0x000f000fu, w.y = v & 0x00f000f0u;
  } else {
    const uint32_t v = i < 2 ? v0 : v1;
    w.x = __builtin_bit_cast(uint32_t, (i & 1) ? ubyte_f<2>(v) : ubyte_f<0>(v));
    w.y = __builtin_bit_cast(uint32_t, (i & 1) ? ubyte_f<3>(v) : ubyte_f<1>(v));
  }
}
template <int BITS>
__device__ __forceinline__ uint32_t piece_value(int i, const PieceCodes& w, const GroupScale<BITS>& g) {
  if constexpr (BITS == 4) {
    if (i & 1) return pack_bf2(fma_half<1>(g.s24, w.x, g.b), fma_half<1>(g.s20, w.y, g.b));
    return pack_bf2(fma_half<0>(g.s24, w.x, g.b), fma_half<0>(g.s20, w.y, g.b));
  } else {
    return pack_bf2(fmaf(g.s, __builtin_bit_cast(float, w.x), g.b), fmaf(g.s, __builtin_bit_cast(float, w.y), g.b));
  }
}

// The operand of lanes whose scale is large, from its codes (4 bits; 8 have no such scales)
template <int BITS, typename V>
__device__ __forceinline__ void large_scales(V& operand, uint32_t v0, float s, float b) {
  if constexpr (BITS == 4) {
    u32x4 o = __builtin_bit_cast(u32x4, operand);
    const uint32_t ev = v0 & 0x0f0f0f0fu, od = (v0 >> 4) & 0x0f0f0f0fu;
    const u32x4 l = {pack_bf2(fmaf(s, ubyte_f<0>(ev), b), fmaf(s, ubyte_f<0>(od), b)),
                     pack_bf2(fmaf(s, ubyte_f<1>(ev), b), fmaf(s, ubyte_f<1>(od), b)),
                     pack_bf2(fmaf(s, ubyte_f<2>(ev), b), fmaf(s, ubyte_f<2>(od), b)),
                     pack_bf2(fmaf(s, ubyte_f<3>(ev), b), fmaf(s, ubyte_f<3>(od), b))};
#pragma unroll
    for (int i = 0; i < 4; ++i) o[i] = fabsf(s) >= 0x1p104f ? l[i] : o[i];
    operand = __builtin_bit_cast(V, o);
  }
}

// The whole operand at once (but for large scales)
template <int BITS>
__device__ __forceinline__ bf16x8_t dequant_words8(uint32_t v0, uint32_t v1, const GroupScale<BITS>& g) {
  u32x4 o;
  PieceCodes w{};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    piece_codes<BITS>(w, i, v0, v1);
    o[piece_reg<BITS>(i)] = piece_value<BITS>(i, w, g);
  }
  return __builtin_bit_cast(bf16x8_t, o);
}
