// Short forms of a requantize whose scales stay.
#ifndef MXQ_FORMS_H_
#define MXQ_FORMS_H_

#include <hip/hip_runtime.h>

#include <cstdint>

#include "mxq_gemm.h"

namespace mxq {

// Short forms.  The definition of a requantize is four float operations with a rounding each, then
// a clamp, a truncation and a relu: 6.5 vector instructions per output with the packing, 7.75
// without the relu, and 6 more for the sum, together several times what the matrix cores take for
// a 1 x 1 layer.  Each of them is a function with few steps of an integer: a requantize has 127
// thresholds (its negative half mirrors the positive one), the sum is defined on 255 x 256 pairs.
// So whether one multiplication and one addition give the same int8 everywhere is found out by
// looking at every threshold from both sides, or at every pair; the factor may move by some last
// places until they do (it holds for nearly all ranges, the others keep the definition).
//   with the relu   cvt_pk_u8(fma(acc, 2t, c)) / 2 with c = 0.5, or some 2^-18 beside it: twice the
//                   level, rounded, in [0, 255]; the halving drops what the rounding of twice the
//                   level and a half is off by
//   without         fma(acc, t, 2^23 + 128) clamped to 2^23 + [1, 255]: its rounding is the
//                   level's, and the low byte is the level + 128
// 3.25 instructions per output of a layer with a relu, 4 without.
constexpr float kRound = 8388608.0f + 128.0f;
__device__ __forceinline__ uint32_t halve4(uint32_t w) { return __builtin_amdgcn_lerp(w, 0u, 0u); }
__device__ __forceinline__ uint32_t short_relu4(int a0, int a1, int a2, int a3, float t, float c) {
  uint32_t w = 0;
  w = __builtin_amdgcn_cvt_pk_u8_f32(__builtin_fmaf(static_cast<float>(a0), t, c), 0, w);
  w = __builtin_amdgcn_cvt_pk_u8_f32(__builtin_fmaf(static_cast<float>(a1), t, c), 1, w);
  w = __builtin_amdgcn_cvt_pk_u8_f32(__builtin_fmaf(static_cast<float>(a2), t, c), 2, w);
  w = __builtin_amdgcn_cvt_pk_u8_f32(__builtin_fmaf(static_cast<float>(a3), t, c), 3, w);
  return halve4(w);
}
// the level + 128, in the low 16 bits
__device__ __forceinline__ uint32_t short_level(int a, float t) {
  return __float_as_uint(
      __builtin_amdgcn_fmed3f(__builtin_fmaf(static_cast<float>(a), t, kRound), kRound - 127.0f,
                              kRound + 127.0f));
}
// Four levels as bytes, a0 in byte 0.
__device__ __forceinline__ uint32_t short_plain4(int a0, int a1, int a2, int a3, float t) {
  return pack_bytes(static_cast<int>(short_level(a0, t)), static_cast<int>(short_level(a1, t)),
                    static_cast<int>(short_level(a2, t)), static_cast<int>(short_level(a3, t))) ^
         0x80808080u;
}

// What a prepared layer holds of them behind its scalars, kFormsAt bytes in: with the relu and
// without.
struct LayerForms {
  int has;  // bit 0: with the relu, bit 1: without
  float t_relu, c_relu, t_plain;
};
constexpr int kFormsAt = 32;
static_assert(sizeof(EpiScalars) <= kFormsAt && kFormsAt + sizeof(LayerForms) <= kPreparedBias,
              "room in front of the bias");

struct LayerForm {
  bool has;
  float t, c;
};
constexpr int kFactors = 64, kConstants = 16;  // tried, one pair a thread
__device__ __forceinline__ float moved(float v, int c) {  // 0, +1, -1, +2, ... last places away
  return __int_as_float(__float_as_int(v) + ((c & 1) ? (c + 1) / 2 : -(c / 2)));
}
__device__ __forceinline__ float constant(int k) {  // likewise around 0.5, in steps of 2^-18
  return 0.5f + static_cast<float>((k & 1) ? (k + 1) / 2 : -(k / 2)) * (1.0f / 262144.0f);
}
// Room in LDS for find_form.
struct FormSearch {
  int threshold[128];
  unsigned long long left[kFactors * kConstants / 64];
};
// Looked for by a work-group of 1024, every thread has the result.  Each thread tries its factor and
// constant at every eighth threshold; those that are left are few, and go one by one through all of
// them, a threshold and a side per thread (all thresholds by one thread each: 28 us, this way 8).
__device__ __forceinline__ LayerForm find_form(const EpiScalars& s, bool relu, FormSearch* m) {
  const int tid = threadIdx.x;
  // the smallest accumulator of level tid, or the largest int where none reaches it
  if (tid < 128) {
    int lo = 0, hi = 0x7fffffff;  // level(lo) < tid, unless tid is 0
    while (tid > 0 && hi - lo > 1) {
      const int at = lo + (hi - lo) / 2;
      (epi_requant(at, s, -127.0f) >= tid ? hi : lo) = at;
    }
    m->threshold[tid] = hi;
  }
  __syncthreads();
  const float unit = s.in_scale * s.qscale * (relu ? 2.0f : 1.0f);
  if (!(unit > 1e-30f && unit < 1e30f)) return {false, unit, 0.5f};
  // d = 0: the definition gives v at its threshold (unless that is the end), d = 1: not before
  auto same = [&](float t, float c, int v, int d) {
    const int a = m->threshold[v] - d;
    const bool reached = d == 0 && epi_requant(a, s, -127.0f) >= v;
    const int level = relu ? static_cast<int>(short_relu4(a, 0, 0, 0, t, c) & 0xffu)
                           : static_cast<int>(short_level(a, t) & 0xffu) - 128;
    return (level >= v) == reached;
  };
  {
    const float t = moved(unit, tid / kConstants), c = constant(tid % kConstants);
    bool ok = true;
    for (int v = 7; v < 128; v += 8) ok = ok && same(t, c, v, 0) && same(t, c, v, 1);
    const unsigned long long left = __ballot(ok);
    if ((tid & 63) == 0) m->left[tid >> 6] = left;
  }
  __syncthreads();
  for (int w = 0; w < kFactors * kConstants / 64; ++w) {
    for (unsigned long long left = m->left[w]; left != 0; left &= left - 1) {
      const int at = 64 * w + __builtin_ctzll(left);
      const float t = moved(unit, at / kConstants), c = constant(at % kConstants);
      const int v = tid >> 1;
      const bool differs = v >= 1 && v < 128 && !same(t, c, v, tid & 1);
      if (__syncthreads_or(differs) == 0) return {true, t, c};
    }
  }
  return {false, unit, 0.5f};
}

}  // namespace mxq
#endif  // MXQ_FORMS_H_
