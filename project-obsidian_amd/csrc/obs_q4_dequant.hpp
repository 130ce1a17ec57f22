// obs_q4_dequant.hpp — the grouped and dense GEMMs' dequantization of 4-bit
// weights to bf16 MFMA fragments (device code).
#pragma once

#include "obs_internal.hpp"

namespace obsd {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8_t;
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float f32x16_t;
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));  // register-friendly 16-byte word

// Two fp32 values -> one packed bf16 pair (RNE, v_cvt_pk_bf16_f32).
__device__ __forceinline__ uint32_t pack_bf16_rne(float lo, float hi) { return pack_bf16_pair_rne(lo, hi); }

// fp32 fma(h, s, b) where h is the low (HI = 0) or high (HI = 1) f16 half of v
// (v_fma_mix_f32: the f16 operand converts exactly to fp32 inside the fma).
template <int HI>
__device__ __forceinline__ float fma_mix_f16(uint32_t v, float s, float b) {
  float r;
  if (HI)
    asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(r) : "v"(v), "v"(s), "v"(b));
  else
    asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel_hi:[1,0,0]" : "=v"(r) : "v"(v), "v"(s), "v"(b));
  return r;
}

// Scale operands of dequant_word_mix for one (row, group): s * 2^24, s * 2^20.
struct MixScale {
  float s24, s20, b;
};
__device__ __forceinline__ MixScale mix_scale(uint32_t packed_sb) {
  const float s = bf16lo(packed_sb);
  return MixScale{s * 0x1p24f, s * 0x1p20f, bf16hi(packed_sb)};
}

// One 32-bit word = 8 nibbles of a weight row -> one bf16x8 MFMA fragment,
// bf16 = RNE(fp32(q*s + b)), with 17 VALU instructions. A nibble masked in
// place at bits 3:0 (or 7:4) of a 16-bit half is the f16 subnormal q * 2^-24
// (or q * 2^-20), exactly; fma_mix multiplies it by s * 2^24 (or s * 2^20),
// which is exact (a power-of-two scaling of the bf16 s, then a 4 x 8-bit
// significand product), and adds b with the single fp32 rounding of
// fmaf(q, s, b). Valid for |s| <= 2^100 (so s * 2^24 cannot overflow); tiles
// holding larger scales use dequant_word. Checked bit for bit against
// fmaf(q, s, b) for every finite bf16 s in that range, on the target GPU.
__device__ __forceinline__ bf16x8_t dequant_word_mix(uint32_t w, const MixScale& m) {
  const uint32_t w8 = w >> 8;
  const uint32_t p04 = w & 0x000F000Fu;   // (q0, q4) * 2^-24
  const uint32_t p15 = w & 0x00F000F0u;   // (q1, q5) * 2^-20
  const uint32_t p26 = w8 & 0x000F000Fu;  // (q2, q6) * 2^-24
  const uint32_t p37 = w8 & 0x00F000F0u;  // (q3, q7) * 2^-20
  u32x4_t r;
  r.x = pack_bf16_rne(fma_mix_f16<0>(p04, m.s24, m.b), fma_mix_f16<0>(p15, m.s20, m.b));
  r.y = pack_bf16_rne(fma_mix_f16<0>(p26, m.s24, m.b), fma_mix_f16<0>(p37, m.s20, m.b));
  r.z = pack_bf16_rne(fma_mix_f16<1>(p04, m.s24, m.b), fma_mix_f16<1>(p15, m.s20, m.b));
  r.w = pack_bf16_rne(fma_mix_f16<1>(p26, m.s24, m.b), fma_mix_f16<1>(p37, m.s20, m.b));
  return __builtin_bit_cast(bf16x8_t, r);
}

// A staged scale|bias word whose scale is beyond dequant_word_mix's range
// (|s| > 2^100, inf, NaN): bf16 exponent field above 127 + 100.
__device__ __forceinline__ bool scale_out_of_mix_range(uint32_t packed_sb) {
  return (packed_sb & 0x7f80u) > (227u << 7);
}

// Reference-form dequant of one word (convert, fma, round), for any scale.
__device__ __forceinline__ bf16x8_t dequant_word(uint32_t w, float s, float b) {
  uint32_t lo = w & 0x0f0f0f0fu, hi = (w >> 4) & 0x0f0f0f0fu;
  // opaque to the optimizer, so each byte converts with one v_cvt_f32_ubyteN
  // instead of being re-derived from w with a shift and a mask
  asm("" : "+v"(lo), "+v"(hi));
  float v[8];
  v[0] = __builtin_fmaf(static_cast<float>(lo & 0xffu), s, b);
  v[1] = __builtin_fmaf(static_cast<float>(hi & 0xffu), s, b);
  v[2] = __builtin_fmaf(static_cast<float>((lo >> 8) & 0xffu), s, b);
  v[3] = __builtin_fmaf(static_cast<float>((hi >> 8) & 0xffu), s, b);
  v[4] = __builtin_fmaf(static_cast<float>((lo >> 16) & 0xffu), s, b);
  v[5] = __builtin_fmaf(static_cast<float>((hi >> 16) & 0xffu), s, b);
  v[6] = __builtin_fmaf(static_cast<float>(lo >> 24), s, b);
  v[7] = __builtin_fmaf(static_cast<float>(hi >> 24), s, b);
  u32x4_t r;
  r.x = pack_bf16_rne(v[0], v[1]);
  r.y = pack_bf16_rne(v[2], v[3]);
  r.z = pack_bf16_rne(v[4], v[5]);
  r.w = pack_bf16_rne(v[6], v[7]);
  return __builtin_bit_cast(bf16x8_t, r);
}

}  // namespace obsd
