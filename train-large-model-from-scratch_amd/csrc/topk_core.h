// Wave-level top-k + softmax over the k winners, shared by the router kernel and the fused
// norm + router kernel.  One 64-lane wavefront owns one token; expert e lives in lane e % 64,
// slot e / 64.
#pragma once
#include "common.h"

__device__ __forceinline__ uint32_t moe_orderable(float v) {
  v += 0.0f;  // -0.0 -> +0.0 so that the two compare equal, as they do for torch.topk
  uint32_t u = __builtin_bit_cast(uint32_t, v);
  // a NaN of either sign ranks above every number, as it does for torch.topk (and maps back
  // to a NaN, so the token's gates are NaN as the reference's are)
  return (v != v) ? 0xffffffffu : u ^ ((u >> 31) ? 0xffffffffu : 0x80000000u);
}
__device__ __forceinline__ float moe_from_orderable(uint32_t u) {
  u ^= ((u >> 31) ? 0x80000000u : 0xffffffffu);
  return __builtin_bit_cast(float, u);
}
// Wave-wide maximum, the same value in every lane: a running maximum inside the rows of 16 lanes and then across them
// on the DPP data path of the vector ALU (no LDS, no waits), read from the last lane.
__device__ __forceinline__ uint32_t moe_wave_max_u32(uint32_t v) {
#define MOE_MAX_STEP(ctrl, rows)                                                                            \
  {                                                                                                         \
    const uint32_t o = (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, ctrl, rows, 0xf, false);       \
    v = o > v ? o : v;                                                                                      \
  }
  MOE_MAX_STEP(0x111, 0xf)  // row_shr:1, 2, 4, 8
  MOE_MAX_STEP(0x112, 0xf)
  MOE_MAX_STEP(0x114, 0xf)
  MOE_MAX_STEP(0x118, 0xf)
  MOE_MAX_STEP(0x142, 0xa)  // row_bcast:15 to rows 1 and 3
  MOE_MAX_STEP(0x143, 0xc)  // row_bcast:31 to rows 2 and 3
#undef MOE_MAX_STEP
  return (uint32_t)__builtin_amdgcn_readlane((int)v, MOE_WAVE - 1);
}
__device__ __forceinline__ float moe_wave_sum_f32(float v) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off, MOE_WAVE);
  return v;
}

// The same where only the first 16 lanes have something other than zero, for them: the same pairs in the same order, on the vector
// ALU's own data path.
__device__ __forceinline__ float moe_row_sum_f32(float v) {
#define MOE_SUM_STEP(n) \
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x120 + n, 0xf, 0xf, false));
  MOE_SUM_STEP(8)  // row_ror
  MOE_SUM_STEP(4)
  MOE_SUM_STEP(2)
  MOE_SUM_STEP(1)
#undef MOE_SUM_STEP
  return v;
}

// The keys of one token's E logits, plus the experts' biases unless NULL: the larger the logit, the larger the key; 0
// (which no logit maps to) marks what is taken or absent.
template <int VPL, typename LT>
__device__ __forceinline__ void moe_topk_keys(const LT* __restrict__ logits, const float* __restrict__ bias, int E, int lane,
                                              uint32_t (&key)[VPL]) {
#pragma unroll
  for (int i = 0; i < VPL; ++i) {
    const int e = i * MOE_WAVE + lane;
    key[i] = 0;
    if (e < E) {
      float v;
      if constexpr (sizeof(LT) == 2) v = bf16_to_f32(((const uint16_t*)logits)[e]);
      else v = ((const float*)logits)[e];
      if (bias) v += bias[e];
      key[i] = moe_orderable(v);
    }
  }
}

// k rounds of a wave-wide maximum over the keys (consumed), each won by the first expert that has it, then the
// softmax over the k selected logits in fp32.  On return lane j < k holds slot j: expert id and gate.
// What bounds it is the chain of k rounds: a 32-bit key, and the winner from a ballot, make a round a dozen
// instructions.  (64-bit keys that held the expert too: 4096 tokens, 8 of 128 experts
// 7.5 -> 5.6 us; norm, router and selection of 8192 tokens 52.1 -> 49.4; a single token, whose gate/up waits for it, 15.8 -> 15.1.)
template <int VPL>
__device__ __forceinline__ void moe_topk_softmax_wave(uint32_t (&key)[VPL], int k, int lane, int& my_id,
                                                      float& my_gate) {
  my_id = 0;
  float my_val = 0.f, vmax = 0.f;
  for (int j = 0; j < k; ++j) {
    uint32_t best = key[0];
#pragma unroll
    for (int i = 1; i < VPL; ++i) best = key[i] > best ? key[i] : best;
    best = moe_wave_max_u32(best);
    int e = 0;
#pragma unroll
    for (int i = VPL - 1; i >= 0; --i) {  // (the first slot that has it, and there the first lane)
      const unsigned long long here = __ballot(key[i] == best);
      if (here) e = i * MOE_WAVE + __builtin_ctzll(here);
    }
#pragma unroll
    for (int i = 0; i < VPL; ++i)
      if (e == i * MOE_WAVE + lane) key[i] = 0;
    const float val = moe_from_orderable(best);
    if (j == 0) vmax = val;
    if (lane == j) {
      my_id = e;
      my_val = val;
    }
  }
  const float p = lane < k ? expf(my_val - vmax) : 0.f;
  const float s = k <= 16 ? moe_row_sum_f32(p) : moe_wave_sum_f32(p);
  my_gate = p / s;
}
