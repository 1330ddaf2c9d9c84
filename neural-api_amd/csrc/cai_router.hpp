// Selection among up to 64 experts by one wave, a lane an expert (TNNetPointwiseSoftMax + TNNetTopKGate, neural/neural.cl:1594-1647): shared by the router's
// launches and the gathered products that choose their experts themselves.
#pragma once
#include "cai_gemv_common.hpp"

namespace cai {

__device__ __forceinline__ float last_lane(float v) { return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 63)); }
// maximum of the wave, valid in lane 63 (wave_sum's steps; a lane without a partner keeps its own)
__device__ __forceinline__ float wave_max(float v)
{
#define STEP(ctrl, rows) { const int t = __builtin_bit_cast(int, v); v = fmaxf(v, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(t, t, ctrl, rows, 0xf, false))); }
  STEP(0x111, 0xf) STEP(0x112, 0xf) STEP(0x114, 0xf) STEP(0x118, 0xf) STEP(0x142, 0xa) STEP(0x143, 0xc)
#undef STEP
  return v;
}
__device__ __forceinline__ uint32_t wave_max_bits(uint32_t v)
{
#define STEP(ctrl, rows) v = max(v, (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, ctrl, rows, 0xf, false));
  STEP(0x111, 0xf) STEP(0x112, 0xf) STEP(0x114, 0xf) STEP(0x118, 0xf) STEP(0x142, 0xa) STEP(0x143, 0xc)
#undef STEP
  return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}

// Selection key of a probability: larger key = selected earlier.  A total order whatever the value: lanes that hold no expert
// get 0, a NaN (a poisoned activation row reaches the router as NaN logits) ranks below every number, and probabilities are
// non-negative, so their bit patterns order like their values.  With a total order the k selected experts are always k
// distinct ids inside [0, n); the gates still carry the NaN to the outputs.
__device__ __forceinline__ uint32_t router_key(float p, bool candidate)
{
  if (!candidate) return 0u;
  if (!(p == p)) return 1u;
  return __builtin_bit_cast(uint32_t, fmaxf(p, 0.0f)) + 2u;
}
// Soft-max over n <= 64 logits by one wave, lane i holding logit i: the lane's probability (0 past the last)
__device__ __forceinline__ float router_softmax64(float logit, int n, int lane)
{
  float v = lane < n ? logit : -3.0e38f;
  const float mx = last_lane(wave_max(v));
  float a = v - mx; a = a > 4000.0f ? 4000.0f : (a < -4000.0f ? -4000.0f : a);
  v = lane < n ? expf(a) : 0.0f;
  const float tot = last_lane(wave_sum(v));
  const float inv = tot > 0.0f ? 1.0f / tot : 1.0f;
  return v * inv;
}
// The experts of places 0 .. last of such a soft-max, by one wave, one after another (larger probability first, lower index between equals): returns the
// expert of place `last`; lane j <= last holds that of place j, and its probability.  (Ranking all 64 against each other takes as long as twenty of these.)
__device__ __forceinline__ int router_pick64(float prob, int n, int last, int lane, int& expert_j, float& prob_j)
{
  uint32_t key = router_key(prob, lane < n);
  int e = 0;
  expert_j = 0; prob_j = 0.0f;
  for (int j = 0; j <= last; j++) {
    const uint32_t top = wave_max_bits(key);
    e = __ffsll((unsigned long long)__ballot(key == top)) - 1;
    if (lane == e) key = 0u;
    const float pe = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, prob), e));
    if (lane == j) { expert_j = e; prob_j = pe; }
  }
  return e;
}

}  // namespace cai
