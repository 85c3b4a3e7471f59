// What the kernels of the grouped bf16 products share: the modes, a launch's arguments, the gate's sigmoid.
#pragma once
#include "internal.h"

enum Mode { GATEUP = 0, DOWN = 1, DGRAD_DOWN = 2, DGRAD_GATEUP = 3, WGRAD = 4 };

// Division of 0 <= n < 2^31 by a divisor that the host knows, n * m >> s: m = floor(2^s / d) + 1 with s = 31 + ceil(log2 d) is exact there
// (Granlund and Montgomery), as n * (m * d - 2^s) < 2^s.  A dozen cycles where the general one takes a few hundred.
struct Divisor {
  uint32_t m;
  int s;
  void set(uint32_t d) {
    s = 31;
    while ((1ull << (s - 31)) < d) ++s;
    m = (uint32_t)((1ull << s) / d + 1);
  }
  __device__ __forceinline__ int operator()(int n) const { return (int)(((unsigned long long)(uint32_t)n * m) >> s); }
};

struct GemmArgs {
  const uint16_t* A0;
  const uint16_t* A1;
  const uint16_t* B0;
  const uint16_t* B1;
  void* C0;
  void* C1;
  void* C2;
  const uint16_t* X0;
  const uint16_t* X1;
  const int32_t* offs;
  int E;        // experts
  int R;        // total rows of the row-ragged operand(s)
  int M;        // WGRAD only: rows of dw[e]
  int N;        // output columns
  int K;        // contraction length per segment (not used by WGRAD)
  int n_tiles;  // tiles along N
  int m_slots;  // row-tile slots (ragged modes) or tiles along M (WGRAD)
  Divisor by_n_tiles, by_m_slots;  // (gemm.hip; m_slots: WGRAD only)
  int accumulate;
  int ld_a;     // row stride of A0/A1 in elements when it is not the contraction length (0: K)
  int ld_c;     // row stride of the outputs C0/C1 in elements when it is not N (0: N)
  int m_split;  // WGRAD: rows m >= m_split of an expert's result go to C1 (as its rows m - m_split); 0: all to C0
  int whole_only;  // row-ragged modes: no half tiles (test hook)
  const int32_t* row_map;  // row-ragged modes, DOWN and DGRAD_GATEUP: where a row of the result goes (NULL: rows stay in order)
  // GATEUP and DGRAD_DOWN: row r of A0, WGRAD: of A0 or B0, is row by_k(row_from[r]) of it, which has from_bytes bytes (NULL: row r)
  const int32_t* row_from;
  bool from_a;
  Divisor by_k;
  long long from_bytes;  // < 2^31
  int streaming;   // WGRAD: results that replace what is there leave with streaming stores
};

// sigmoid from the two hardware transcendentals (v_exp_f32, v_rcp_f32; about 1 ulp each):
// the epilogues are VALU-bound, and an IEEE division would triple their cost.
__device__ __forceinline__ float sigmoidf_(float x) {
  return __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(x * -1.4426950408889634f));
}

// What the fused epilogues do with an element, the same operations whatever the tile, so that the bits do not depend on it:
// silu(g) * u, and backwards, with `dot` summing up dact * act.
__device__ __forceinline__ float swiglu(float g, float u) { return g * sigmoidf_(g) * u; }
__device__ __forceinline__ void swiglu_bwd(float dact, float g, float u, float& dg, float& du, float& dot) {
  const float sg = sigmoidf_(g), gs = g * sg;  // gs: silu(g)
  du = dact * gs;
  dg = (dact * u) * (sg + (gs - gs * sg));     // silu'(g) = s + g*s*(1-s)
  dot += du * u;
}

// Takes a row-ragged launch of few tiles (csrc/row_ring.hip): false where it does not.  `forced`: any launch, in tiles of 64 or
// 128 rows (0: its own choice).
bool moe_ring_rows(Mode mode, bool blocked, const GemmArgs& a, int forced, hipStream_t s, int* rc);
