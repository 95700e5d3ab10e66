// Top-k gating of one token by one wavefront, shared by the router kernels
// of router.hip (the chunk fold with and without the fused dispatch, and the
// standalone topk), which must pick the same ids and gates bit for bit.
//
// Reference: src/core/kernels/reduce/topkSelect.ts:21-92 (selection) and
// :142-156 (softmax over the selected logits). Each lane owns experts lane,
// lane + 64, …; k rounds of a butterfly arg-max (ties → lower id) pick the
// winners: the reference's bubble insertion restated for a wavefront. A
// logit is a candidate only if it is strictly above the reference's
// −3.4e38 start value (so NaN never enters), and a slot no candidate fills
// keeps (−3.4e38, id 0), as the reference's does. Both including files are
// compiled with -ffp-contract=off.
#pragma once
#include "dispatch_dev.h"

namespace moe_dev {

constexpr float NEG_START = -3.4e38f;

// A logit as an unsigned key in the same order (0 below every one); −0 as +0,
// which compares equal to it.
__device__ __forceinline__ uint32_t order_key(float v) {
  const int32_t b = __builtin_bit_cast(int32_t, v + 0.f);
  return (uint32_t)(b ^ ((b >> 31) | INT32_MIN));
}
__device__ __forceinline__ float key_value(uint32_t key) {
  const int32_t b = (int32_t)key;
  return __builtin_bit_cast(float, b < 0 ? b ^ INT32_MIN : ~b);
}

// The largest key of the wavefront: six max steps whose partners come through
// DPP (rows of 16 by shifts, then the row broadcasts), no LDS trip; lane 63
// ends with it. A lane without a source takes 0, below every key.
template <int CTRL>
__device__ __forceinline__ uint32_t max_dpp(uint32_t v) {
  const uint32_t o = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xf, 0xf, false);
  return v > o ? v : o;
}
__device__ __forceinline__ uint32_t wave_max_key(uint32_t v) {
  v = max_dpp<0x111>(v);  // row_shr 1
  v = max_dpp<0x112>(v);  // row_shr 2
  v = max_dpp<0x114>(v);  // row_shr 4
  v = max_dpp<0x118>(v);  // row_shr 8
  v = max_dpp<0x142>(v);  // row_bcast 15
  v = max_dpp<0x143>(v);  // row_bcast 31
  return (uint32_t)__builtin_amdgcn_readlane((int)v, WAVE - 1);
}

// Selects the top k of the wavefront's logits and writes the route row.
// vals[i] is expert lane + 64·i (i < NI). Each round takes the largest key
// and, of the experts that hold it, the lowest (i first, then the lane, from
// a ballot): a serial chain of about ten dependent register operations and a
// few scalar ones, where comparing (value, id) pairs through six exchanges
// took two LDS trips and some forty. Round r's winner is kept by lane r.
// Then w_i = exp(v_i − v_0) / Σ_j exp(v_j − v_0), the sum taken left to right
// (topkSelect.ts:142-156); lane i < k writes slot i.
template <int NI>
__device__ __forceinline__ int wave_topk_route(const float (&vals)[NI], int E, int k, int lane,
                                               float *row) {
  uint32_t key[NI];
#pragma unroll
  for (int i = 0; i < NI; i++)
    key[i] = lane + WAVE * i < E && vals[i] > NEG_START ? order_key(vals[i]) : 0;
  float my_v = NEG_START;
  int my_id = 0;
#pragma unroll 1
  for (int r = 0; r < k; r++) {
    uint32_t best = key[0];
#pragma unroll
    for (int i = 1; i < NI; i++) best = key[i] > best ? key[i] : best;
    best = wave_max_key(best);
    if (best == 0) break;  // no candidate left: the reference's untouched slots
    int id = 0;
#pragma unroll
    for (int i = NI - 1; i >= 0; i--) {
      const uint64_t at = __ballot(key[i] == best);
      if (at) id = WAVE * i + __builtin_ctzll(at);
    }
#pragma unroll
    for (int i = 0; i < NI; i++) key[i] = lane + WAVE * i == id ? 0 : key[i];
    if (lane == r) {
      my_v = key_value(best);
      my_id = id;
    }
  }
  // Lane reads go through readlane (a register read, no LDS trip).
  auto lane_f = [](float v, int l) {
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), l));
  };
  float m = lane_f(my_v, 0);
  float ex = expf(my_v - m);
  float z = lane_f(ex, 0);
#pragma unroll 1
  for (int i = 1; i < k; i++) z = z + lane_f(ex, i);
  if (lane < k) {
    row[lane] = (float)my_id;
    row[k + lane] = ex / z;
  }
  return my_id;
}

}  // namespace moe_dev
