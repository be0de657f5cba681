// The residual sum as an epilogue step: int8 + int8 -> int8 over a calibrated range,
// optionally followed by the int8 relu of _contrib_quantized_act
// (quantized_activation.cc:84-120).  It mirrors add_kernel in mxq_eltwise.hip and the CPU
// oracle bit for bit.  The scales come from the reference's own files
// (src/operator/quantization/quantized_elemwise_add.cc:30-134,
// dnnl/dnnl_quantized_elemwise_add.cc:134-257); the element arithmetic itself (two float
// products, one sum, nearest-even, saturation, NaN -> 0) happens inside oneDNN in the
// reference and is not pinned by anything in its tree: parity unpinned, as for add_kernel.  A kernel that holds the
// left operand in registers applies it to 16-byte pieces on their way out.
//
// A graph whose sum is calibrated behind the operator (the sum in int32 over its own range, then
// _contrib_requantize over the calibrated one: what QuantizeGraph makes of an elemwise_add) has
// the second form, RequantRule: add32 and requantize element by element, the int32 between them
// in a register.
#ifndef MXQ_SUM_H_
#define MXQ_SUM_H_

#include <hip/hip_runtime.h>

#include <cstdint>

namespace mxq {

// Four floats of at most 127 truncated to bytes, negative ones to 0, a in byte 0.
// v_cvt_pk_u8_f32 saturates at 0, writes byte k of its destination, and rounds as the wave's
// float rounding mode says.  The mode is switched to round-toward-zero for exactly the four
// converts (one asm statement, so that no multiply or add of a requantization can be scheduled
// into the stretch) and back: the operands are computed in round-to-nearest as before.
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ uint32_t pack4_truncated(float a, float b, float c, float d) {
  uint32_t w;
  asm volatile(
      "s_setreg_imm32_b32 hwreg(HW_REG_MODE, 0, 2), 3\n\t"
      "v_cvt_pk_u8_f32 %0, %1, 0, 0\n\t"
      "v_cvt_pk_u8_f32 %0, %2, 1, %0\n\t"
      "v_cvt_pk_u8_f32 %0, %3, 2, %0\n\t"
      "v_cvt_pk_u8_f32 %0, %4, 3, %0\n\t"
      "s_setreg_imm32_b32 hwreg(HW_REG_MODE, 0, 2), 0"
      : "=&v"(w)
      : "v"(a), "v"(b), "v"(c), "v"(d));
  return w;
}
#pragma clang diagnostic pop

struct SumRule {
  float s0, s1;  // output levels per level of the left / right operand
  int fast;      // neither product can overflow: no NaN, the one-instruction clamp applies
};

// dnnl_quantized_elemwise_add.cc:143-210 for two int8 operands and a calibrated int8 output:
// every scale is the type's range (127.5) over the tensor's largest magnitude.
__device__ __forceinline__ SumRule sum_rule(float a_absmax, float b_absmax, float min_calib,
                                            float max_calib) {
  SumRule r;
  const float a_scale = 127.5f / a_absmax;
  const float b_scale = 127.5f / b_absmax;
  const float x = fabsf(min_calib), y = fabsf(max_calib);
  const float out_scale = static_cast<float>(127.5 / static_cast<double>((x < y) ? y : x));
  r.s0 = out_scale / a_scale;
  r.s1 = out_scale / b_scale;
  r.fast = fabsf(r.s0) < 1e30f && fabsf(r.s1) < 1e30f;  // false for NaN as well
  return r;
}

// The sum's int32 form followed by the requantization (quantized_elemwise_add.cc:110-134,
// requantize-inl.h:89-125): s0 / s1 are int32 levels per operand level.
struct RequantRule {
  float s0, s1;
  float in_scale;  // float per int32 level
  float qscale;    // int8 levels per float
  int fast;        // no product overflows and nothing is NaN: the sum needs no saturation
  float ta, tb;    // the short form, where `pairs` says that it holds (SumPairs): the scales
                   // above are then left out
  int pairs;
};

// The short form of a RequantRule with the relu behind it: nearest-even(a * ta + b * tb) clamped
// to [0, 127], one rounding per product and one for the sum instead of seven.  Both operands are
// int8, so it either gives the definition's result for all 255 x 256 pairs or it does not, and
// that is found out by trying them: sum_pairs_kernel (mxq_fc.hip) does so once for ranges that
// stay (a plan's constants).  What it may be off by is a last place of a value near a tie, so the
// products of the rule's scales hold as they are for most ranges and within three last places of
// them for nearly all others.
struct SumPairs {
  float ta, tb;
  int ok;
};

__device__ __forceinline__ RequantRule sum_requant_rule(float a_absmax, float b_absmax,
                                                        float min_calib, float max_calib) {
  RequantRule r;
  const float a_scale = 127.5f / a_absmax;
  const float b_scale = 127.5f / b_absmax;
  const float range = a_absmax + b_absmax;
  const float out_scale = static_cast<float>(2147483647.0 / static_cast<double>(range));
  r.s0 = out_scale / a_scale;
  r.s1 = out_scale / b_scale;
  r.in_scale = range / 2147483648.0f;
  const float x = fabsf(min_calib), y = fabsf(max_calib);
  r.qscale = 127.0f / ((x < y) ? y : x);
  r.fast = fabsf(r.s0) < 1e30f && fabsf(r.s1) < 1e30f && fabsf(r.qscale) < 1e30f &&
           r.in_scale > 0.0f;
  r.ta = r.tb = 0.0f;
  r.pairs = 0;
  return r;
}

// Four pairs under the short form: 6 instructions a pair instead of 11.5.
__device__ __forceinline__ uint32_t sum_pairs4(uint32_t x, uint32_t y, const RequantRule& r) {
  uint32_t w = 0;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int a = static_cast<int>(static_cast<int8_t>((x >> (8 * k)) & 0xffu));
    const int b = static_cast<int>(static_cast<int8_t>((y >> (8 * k)) & 0xffu));
    const float u = __builtin_fmaf(static_cast<float>(a), r.ta, static_cast<float>(b) * r.tb);
    // rounds to nearest even, what is below zero becomes 0
    w = __builtin_amdgcn_cvt_pk_u8_f32(u < 127.0f ? u : 127.0f, k, w);
  }
  return w;
}

// One element, as the two operators compute it one after the other.
template <bool RELU>
__device__ __forceinline__ int sum_requant_one(int a, int b, const RequantRule& r) {
  const float p = static_cast<float>(a) * r.s0;
  const float q = static_cast<float>(b) * r.s1;
  float f = p + q;
  int acc = 0;  // NaN
  if (f == f) {
    f = f < -2147483648.0f ? -2147483648.0f : f;
    f = f > 2147483520.0f ? 2147483520.0f : f;
    acc = static_cast<int>(rintf(f));
  }
  f = static_cast<float>(acc) * r.in_scale;
  float u = fabsf(f) * r.qscale + 0.5f;
  u = 127.0f < u ? 127.0f : u;
  const int v = static_cast<int>(u);
  const int s = f < 0.0f ? -v : (f > 0.0f ? v : 0);
  return RELU && s < 0 ? 0 : s;
}

// One element under whatever form the rule has.
__device__ __forceinline__ int sum_requant_any(int a, int b, bool relu, const RequantRule& r) {
  if (r.pairs)
    return static_cast<int>(sum_pairs4(static_cast<uint32_t>(a) & 0xffu,
                                       static_cast<uint32_t>(b) & 0xffu, r) & 0xffu);
  return relu ? sum_requant_one<true>(a, b, r) : sum_requant_one<false>(a, b, r);
}

// One element: saturate, round to nearest even, NaN -> 0; with RELU the negative results
// become 0 (clamping at 0 before the rounding gives the same integer).
template <bool RELU, bool FAST>
__device__ __forceinline__ uint32_t sum_one(int a, int b, const SumRule& r) {
  const float p = static_cast<float>(a) * r.s0;
  const float q = static_cast<float>(b) * r.s1;
  float f = p + q;
  constexpr float lo = RELU ? 0.0f : -128.0f;
  if (FAST)  // nearest-even(f) in the low mantissa byte of f + 1.5 * 2^23
    return __float_as_uint(__builtin_amdgcn_fmed3f(f, lo, 127.0f) + 12582912.0f);
  if (f != f) return 0u;
  f = f < lo ? lo : f;
  f = f > 127.0f ? 127.0f : f;
  return static_cast<uint32_t>(static_cast<int>(rintf(f)));
}

// Four pairs under a fast RequantRule.  The int32 of the definition stays a float: a rounded
// sum of that size is an integer whether it is converted or not, and the way back to float is
// exact.  With the relu no saturation is left: the sum of two int8 values of at most 127 cannot
// pass int32's upper end (127 / 127.5 of the range), and what is below zero becomes 0 anyway;
// without it the lower end is reached by -128 with -128.  The requantization is that of
// epi_requant_pack.
template <bool RELU>
__device__ __forceinline__ uint32_t sum_requant4(uint32_t x, uint32_t y, const RequantRule& r) {
  float u[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int a = static_cast<int>(static_cast<int8_t>((x >> (8 * k)) & 0xffu));
    const int b = static_cast<int>(static_cast<int8_t>((y >> (8 * k)) & 0xffu));
    const float p = static_cast<float>(a) * r.s0;
    const float q = static_cast<float>(b) * r.s1;
    float f = p + q;
    if (!RELU) f = __builtin_amdgcn_fmed3f(f, -2147483648.0f, 2147483520.0f);
    f = rintf(f) * r.in_scale;
    if (RELU) {
      u[k] = f * r.qscale + 0.5f;
      u[k] = u[k] < 127.0f ? u[k] : 127.0f;
    } else {
      u[k] = __builtin_amdgcn_fmed3f(copysignf(fabsf(f) * r.qscale + 0.5f, f), -127.0f, 127.0f);
    }
  }
  if (RELU) return pack4_truncated(u[0], u[1], u[2], u[3]);
  uint32_t q[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) q[k] = static_cast<uint32_t>(static_cast<int>(u[k]));
  const uint32_t lo = __builtin_amdgcn_perm(q[1], q[0], 0x0c0c0400u);
  const uint32_t hi = __builtin_amdgcn_perm(q[3], q[2], 0x04000c0cu);
  return lo | hi;
}

// Four pairs under any RequantRule.
template <bool RELU>
__device__ __forceinline__ uint32_t sum_requant4_general(uint32_t x, uint32_t y,
                                                         const RequantRule& r) {
  uint32_t w = 0;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int a = static_cast<int>(static_cast<int8_t>((x >> (8 * k)) & 0xffu));
    const int b = static_cast<int>(static_cast<int8_t>((y >> (8 * k)) & 0xffu));
    w |= (static_cast<uint32_t>(sum_requant_one<RELU>(a, b, r)) & 0xffu) << (8 * k);
  }
  return w;
}

// Four int8 pairs (x: left operand, y: right operand, byte k of each) -> four int8 results.
template <bool RELU, bool FAST>
__device__ __forceinline__ uint32_t sum4(uint32_t x, uint32_t y, const SumRule& r) {
  if (RELU && FAST) {
    // results in [0, 127]: v_cvt_pk_u8_f32 rounds to nearest even, saturates and places the
    // byte in one instruction (instead of the 1.5 * 2^23 add and three quarters of a pack)
    uint32_t w = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int a = static_cast<int>(static_cast<int8_t>((x >> (8 * k)) & 0xffu));
      const int b = static_cast<int>(static_cast<int8_t>((y >> (8 * k)) & 0xffu));
      const float p = static_cast<float>(a) * r.s0;
      const float q = static_cast<float>(b) * r.s1;
      w = __builtin_amdgcn_cvt_pk_u8_f32(__builtin_amdgcn_fmed3f(p + q, 0.0f, 127.0f), k, w);
    }
    return w;
  }
  uint32_t q[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int a = static_cast<int>(static_cast<int8_t>((x >> (8 * k)) & 0xffu));
    const int b = static_cast<int>(static_cast<int8_t>((y >> (8 * k)) & 0xffu));
    q[k] = sum_one<RELU, FAST>(a, b, r);
  }
  const uint32_t lo = __builtin_amdgcn_perm(q[1], q[0], 0x0c0c0400u);
  const uint32_t hi = __builtin_amdgcn_perm(q[3], q[2], 0x04000c0cu);
  return lo | hi;
}

}  // namespace mxq
#endif  // MXQ_SUM_H_
