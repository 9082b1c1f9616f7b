// The seam of a MoE layer on tiles (tile_expert_core.h, tile_wide_core.h): what a wave does with the first product's sums -- rounded as the operator stores
// them, activated, quantized, and left as the second product's kernel takes its rows.
#pragma once
#include "mmq_formats.h"
#include "q8_1_device.h"

namespace gguf {

__device__ __forceinline__ float seam_rounded(float v, int dtype) {   // to the result's type and back
  return dtype == GGUF_DTYPE_F32 ? v : dtype == GGUF_DTYPE_F16 ? (float)(_Float16)v : (float)(__bf16)v;
}
// gate1 in the result's type (which the branches around it are on, not its values)
__device__ __forceinline__ float seam_gate(float g, float u, int act, int dtype) {
  const float a = act == ACT_SILU ? g / (1.0f + expf(-g)) : g * 0.5f * (1.0f + erff(g * 0.70710678118654752440f));
  return seam_rounded(seam_rounded(a, dtype) * u, dtype);
}
// The quants of h as q8_1_quantize8 rounds them: by the reciprocal, by the quotient where a value lies close to a tie.  What is not a
// number is 0, as the conversion to an integer leaves it there.
template <int N> __device__ __forceinline__ void seam_quants(const float (&h)[N], float d, bool none, float (&q)[N]) {
  const float dd = none ? 1.0f : d, rd = __builtin_amdgcn_rcpf(dd);
  bool exact = !(rd < 3.0e38f);
#pragma unroll
  for (int i = 0; i < N; ++i) {
    q[i] = h[i] * rd;
    exact = exact || fabsf(__builtin_amdgcn_fractf(fabsf(q[i])) - 0.5f) < 6.1035156e-5f;
  }
  if (exact) {
#pragma unroll
    for (int i = 0; i < N; ++i) q[i] = roundf(h[i] / dd);
  } else {
#pragma unroll
    for (int i = 0; i < N; ++i) q[i] = truncf(q[i] + copysignf(0.5f, q[i]));
  }
#pragma unroll
  for (int i = 0; i < N; ++i) q[i] = q[i] == q[i] ? q[i] : 0.0f;
}

// Four neighbouring quants of h, in the record that the second product's kernel takes (gate.kp: 1 tile_wide.h's, 0 tile_expert.h's), features `at` .. of
// block blk of the record's four; the block's scale and sum.
__device__ __forceinline__ char* seam_h_record(const Gate16& gate, int n0, int pair, int pairs) {
  return gate.rows + ((int64_t)(n0 >> 7) * pairs + pair) * (gate.kp ? WIDE_REC : EXPERT_REC);
}
__device__ __forceinline__ void seam_h_store(char* rec, const Gate16& gate, int blk, int at, const float* q) {
  if (gate.kp) {
    union { _Float16 v[4]; uint2 u; } o;
#pragma unroll
    for (int e = 0; e < 4; ++e) o.v[(e & 1) * 2 + (e >> 1)] = (_Float16)q[e];
    *(uint2*)(rec + 64 * blk + 2 * at) = o.u;
  } else {
    uint32_t o = 0;
#pragma unroll
    for (int e = 0; e < 4; ++e) o |= ((uint32_t)(int)q[e] & 0xFFu) << (8 * e);
    *(uint32_t*)(rec + 32 * blk + at) = o;
  }
}
__device__ __forceinline__ void seam_h_scales(char* rec, const Gate16& gate, int blk, float d, float sum) {
  *(_Float16*)(rec + (gate.kp ? WIDE_D_AT : EXPERT_D_AT) + 2 * blk) = (_Float16)d;
  *(_Float16*)(rec + (gate.kp ? WIDE_S_AT : EXPERT_S_AT) + 2 * blk) = (_Float16)sum;
}

}  // namespace gguf
