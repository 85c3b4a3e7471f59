// A token's k rows added up, by a wave, and the router path's share of its input gradient with them: what combine and its counterpart in the backward
// pass (dispatch.hip) and the norm's backward (norm.hip) have in common.
#pragma once
#include <type_traits>

#include "common.h"

namespace {

struct RouterGrad {
  const float* part;   // [P][T*k], by position
  int P;
  const float* gates;
  const int32_t* ids;
  const uint16_t* wr;  // [E, H]
  void* dlogits;       // [T, ld]
  int ld;
};

// A token's row of dlogits (LT: bf16 or fp32), written if `write`, and the k entries that are not zero: lane j < k gets slot j's, and its expert.
template <typename LT>
__device__ __forceinline__ float router_dsel(const RouterGrad& rg, const int32_t* __restrict__ row_to_pos, int T, int k, int t,
                                             bool write, int& id) {
  const int lane = lane_id(), r0 = t * k;
  id = -1;
  float s = 0.f, g = 0.f;
  if (lane < k) {
    const float* src = rg.part + row_to_pos[r0 + lane];
    id = rg.ids[r0 + lane];
    g = rg.gates[r0 + lane];
    const size_t R = (size_t)T * k;
    int b = 0;
    for (; b + 8 <= rg.P; b += 8) {  // (eight gathers in flight, added in ascending order)
      float v[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) v[i] = src[(size_t)(b + i) * R];
#pragma unroll
      for (int i = 0; i < 8; ++i) s += v[i];
    }
    for (; b + 4 <= rg.P; b += 4) {
      const float v0 = src[(size_t)b * R], v1 = src[(size_t)(b + 1) * R], v2 = src[(size_t)(b + 2) * R], v3 = src[(size_t)(b + 3) * R];
      s = (((s + v0) + v1) + v2) + v3;
    }
    for (; b < rg.P; ++b) s += src[(size_t)b * R];
  }
  const float dg = g != 0.f ? s / g : 0.f;
  float dot = 0.f;
  for (int j = 0; j < k; ++j) dot += read_lane_f(g, j) * read_lane_f(dg, j);
  float dsel = g * (dg - dot);
  if constexpr (sizeof(LT) == 2) dsel = bf16_to_f32(f32_to_bf16(dsel));
  if (write)
    for (int e = lane; e < rg.ld; e += MOE_WAVE) {
      float v = 0.f;
      for (int j = 0; j < k; ++j) v = read_lane(id, j) == e ? read_lane_f(dsel, j) : v;
      if constexpr (sizeof(LT) == 2) ((uint16_t*)rg.dlogits)[(size_t)t * rg.ld + e] = f32_to_bf16(v);
      else ((float*)rg.dlogits)[(size_t)t * rg.ld + e] = v;
    }
  return dsel;
}

// Eight columns from `col` on: acc the rows' sum (times their gates, if any), in slot order, and with ROUTER d2 that of the k rows of the router
// weight times dsel.
template <bool ROUTER, bool IN_ORDER>
__device__ __forceinline__ void sum_rows(const uint16_t* __restrict__ y, const float* __restrict__ gates,
                                         const int32_t* __restrict__ row_to_pos, const RouterGrad& rg, int id, float dsel, int r0,
                                         int k, int H, int col, Row8& acc, Row8& d2) {
#pragma unroll
  for (int i = 0; i < 8; ++i) acc.v[i] = 0.f, d2.v[i] = 0.f;
  // the next N rows, all in flight; summed in slot order
  const auto add = [&](int j, auto n) {
    constexpr int N = decltype(n)::value;
    u32x4 v[N], w[ROUTER ? N : 1];
#pragma unroll
    for (int q = 0; q < N; ++q) {
      const int pos = IN_ORDER ? r0 + j + q : row_to_pos[r0 + j + q];
      v[q] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(y + (size_t)pos * H + col));
    }
    if constexpr (ROUTER) {
#pragma unroll
      for (int q = 0; q < N; ++q) w[q] = *reinterpret_cast<const u32x4*>(rg.wr + (size_t)read_lane(id, j + q) * H + col);
    }
#pragma unroll
    for (int q = 0; q < N; ++q) {
      const float gt = gates ? gates[r0 + j + q] : 1.f;
      const Row8 row = row8_from_bits(v[q]);
#pragma unroll
      for (int i = 0; i < 8; ++i) acc.v[i] += gt * row.v[i];
    }
    if constexpr (ROUTER) {
#pragma unroll
      for (int q = 0; q < N; ++q) {
        const float ds = read_lane_f(dsel, j + q);
        const Row8 row = row8_from_bits(w[q]);
#pragma unroll
        for (int i = 0; i < 8; ++i) d2.v[i] += ds * row.v[i];
      }
    }
  };
  int j = 0;
  for (; j + 8 <= k; j += 8) add(j, std::integral_constant<int, 8>{});
  if (j + 4 <= k) add(j, std::integral_constant<int, 4>{}), j += 4;
  if (j + 2 <= k) add(j, std::integral_constant<int, 2>{}), j += 2;
  if (j < k) add(j, std::integral_constant<int, 1>{});
}

}  // namespace
