// Helpers of the prefill GEMMs (gemm.hip, gemm_mid.hip): fp16 operands from
// packed codes and activations.
#pragma once

#include "common.h"
#include "internal.h"

namespace nvm {

typedef _Float16 h2_t __attribute__((ext_vector_type(2)));

__device__ __forceinline__ uint32_t pk_fma_h(uint32_t a, uint32_t b, uint32_t c) {  // v_pk_fma_f16
  return __builtin_bit_cast(uint32_t,
                            __builtin_elementwise_fma(__builtin_bit_cast(h2_t, a),
                                                      __builtin_bit_cast(h2_t, b),
                                                      __builtin_bit_cast(h2_t, c)));
}
__device__ __forceinline__ uint32_t pk_add_h(uint32_t a, uint32_t b) {  // v_pk_add_f16
  return __builtin_bit_cast(uint32_t, __builtin_bit_cast(h2_t, a) + __builtin_bit_cast(h2_t, b));
}

// One packed word (codes q0..q7, q_i at bits 4i) -> the 8 weights q_i*s + b
// as fp16, each the correctly rounded value of the exact q*s + b (one
// v_pk_fma_f16 per pair, single rounding), in the pair order
// (q0,q4)(q1,q5)(q2,q6)(q3,q7).  The codes become exact fp16 values by OR-ing
// them into the mantissa of a constant that is then taken off exactly: codes
// in bits 0-3 into 1024.0 (ulp 1), codes in bits 4-7 into 64.0 (bit 4 is
// worth 1), so a word needs one shift where one constant would need three.
// s2, b2: (s, s) and (b, b) as fp16 pairs.
struct DeqConst {
  uint32_t mask0, mask4;      // SGPRs: a v_and_or_b32 reads one
  uint32_t magic0, magic4;    // VGPRs
};
__device__ __forceinline__ DeqConst deq_const() {
  return DeqConst{sgpr_const(0x000F000Fu), sgpr_const(0x00F000F0u), vgpr_const(0x64006400u),
                  vgpr_const(0x54005400u)};
}
__device__ __forceinline__ u32x4 dequant8_h(uint32_t w, uint32_t s2, uint32_t b2,
                                            const DeqConst &k) {
  const uint32_t v = w >> 8;
  const uint32_t d0 = pk_add_h((w & k.mask0) | k.magic0, 0xE400E400u);  // - 1024
  const uint32_t d1 = pk_add_h((w & k.mask4) | k.magic4, 0xD400D400u);  // - 64
  const uint32_t d2 = pk_add_h((v & k.mask0) | k.magic0, 0xE400E400u);
  const uint32_t d3 = pk_add_h((v & k.mask4) | k.magic4, 0xD400D400u);
  return u32x4{pk_fma_h(d0, s2, b2), pk_fma_h(d1, s2, b2), pk_fma_h(d2, s2, b2),
               pk_fma_h(d3, s2, b2)};
}

// Eight consecutive activations x0..x7 (one 16-byte chunk of a row) -> fp16
// in the pair order (x0,x4)(x1,x5)(x2,x6)(x3,x7) of dequant8_h.  (Activations
// that arrive in fp16, GroupedArgs::act_h, are in that order already.)  bf16 values
// convert exactly (fp16 carries more significand bits) within fp16's range;
// v_cvt_pkrtz_f16_f32 only rounds below it (|x| < 2^-14, with a contribution
// far under the product's rounding) and saturates above 65504.
template <int DT>
__device__ __forceinline__ u32x4 act_to_h(u32x4 v) {
  if constexpr (DT == DT_F16) {
    return pair_order(v);
  } else {
    u32x4 o;
    const float x0 = __uint_as_float(v.x << 16), x1 = __uint_as_float(v.x & 0xFFFF0000u);
    const float x2 = __uint_as_float(v.y << 16), x3 = __uint_as_float(v.y & 0xFFFF0000u);
    const float x4 = __uint_as_float(v.z << 16), x5 = __uint_as_float(v.z & 0xFFFF0000u);
    const float x6 = __uint_as_float(v.w << 16), x7 = __uint_as_float(v.w & 0xFFFF0000u);
    o.x = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(x0, x4));
    o.y = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(x1, x5));
    o.z = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(x2, x6));
    o.w = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(x3, x7));
    return o;
  }
}

// A scale or bias (act bits) as fp16 bits; bf16 values convert with round to
// nearest even (exactly, inside fp16's normal range).
template <int DT>
__device__ __forceinline__ uint32_t sb_h(uint32_t bits) {
  if constexpr (DT == DT_F16)
    return bits & 0xFFFFu;
  else
    return __builtin_bit_cast(uint16_t, (_Float16)__uint_as_float(bits << 16));
}

__device__ __forceinline__ f32x16 mfma32_h(u32x4 a, u32x4 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a),
                                                __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}

}  // namespace nvm
