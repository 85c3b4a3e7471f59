// A tile of the grouped products over an expert's rows, its k-tiles straight into a ring of LDS stages: for the launches of few
// tiles (row_ring.hip) and for what is left after the whole rounds of the larger tiles (gemm.hip).
#pragma once
#include <type_traits>

#include "gemm_args.h"
#include "ring.h"

namespace {

// A tile of WAVES waves, 2 x WAVES / 2, each 32 FM rows x 64 columns (gate and up: 32 of each), over k-tiles of 64.
template <int MODE, int FM, int WAVES>
struct RingTile {
  static constexpr int BM = 64 * FM, BN = 32 * WAVES, BK = 64, KS = BK / 16, STAGES = FM == 1 ? 3 : 2;
  static constexpr bool DUAL = MODE == GATEUP, B_OUTER = MODE == DGRAD_DOWN || MODE == DGRAD_GATEUP;
  static constexpr int BNC = DUAL ? BN / 2 : BN;  // output columns of a tile
  using OpA = RingInner<BM, BK, WAVES>;
  using OpB = typename std::conditional<B_OUTER, RingOuter<BN, BK, WAVES>, RingInner<BNC, BK, WAVES>>::type;  // (DUAL: two of them)
  static constexpr int NB = DUAL ? 2 : 1, LOADS = OpA::PER_WAVE + NB * OpB::PER_WAVE;
  static constexpr int STAGE = OpA::BYTES + NB * OpB::BYTES, LDS = STAGES * STAGE;
  static_assert(LDS <= 20 * 1024 * WAVES && STAGE >= WAVES * 4096, "eight waves to a compute unit; their strips in a stage");
};

// The tile of expert e, whose rows are first .. row_end, at its row `row` and column n0.  By the whole workgroup; `ring`: LDS bytes
// of LDS that nobody else uses.  BLK: g and u are kept in blocks, as the kernels of larger tiles keep them; TO: the result's rows
// go where p.row_map says, FROM: A's come from where p.row_from says (see there).
template <int MODE, bool BLK, int FM, int WAVES, bool TO = false, bool FROM = false>
__device__ __forceinline__ void ring_tile(const GemmArgs& p, char* ring, int e, int first, int row_end, int row, int n0) {
  using O = RingTile<MODE, FM, WAVES>;
  using OpA = typename O::OpA;
  using OpB = typename O::OpB;
  constexpr int BK = O::BK, KS = O::KS, STAGES = O::STAGES, NSEG = MODE == DGRAD_GATEUP ? 2 : 1;
  constexpr bool DUAL = O::DUAL, B_OUTER = O::B_OUTER;
  const int lane = lane_id(), wv = uniform((int)(threadIdx.x / MOE_WAVE)), wm = wv / (WAVES / 2), wn = wv % (WAVES / 2);
  const int row0 = first + row;
  const int lda = MODE == GATEUP || MODE == DOWN || !p.ld_a ? p.K : p.ld_a, ldb = B_OUTER ? p.N : p.K;
  View vA[2], vB[2];  // of the two segments, or gate and up
  const long long a_at = (long long)row0 * lda, a_valid = (long long)(row_end - row0) * lda;
  const long long b_at = (long long)e * p.K * p.N + (long long)n0 * (B_OUTER ? 1 : p.K);
  const long long b_valid = (long long)p.K * p.N - (long long)n0 * (B_OUTER ? 1 : p.K);
  vA[0] = FROM ? View{p.A0, p.from_bytes} : make_view(p.A0 + a_at, a_valid);
  vB[0] = make_view(p.B0 + b_at, b_valid);
  if constexpr (NSEG == 2) vA[1] = make_view(p.A1 + a_at, a_valid);
  if constexpr (NSEG == 2 || DUAL) vB[1] = make_view(p.B1 + b_at, b_valid);
  // (tiles past the last column: dgrad-down has them for its sums, which are zero there)
  const int steps = n0 < p.N ? (p.K + BK - 1) / BK * NSEG : 0;

  // ---- the contraction
  OpA opA;
  OpB opB;
  opA.init(lda, wv);
  if constexpr (FROM)
    opA.set_rows(wv, [&](int r) { return row0 + r < row_end ? (uint32_t)p.by_k(p.row_from[row0 + r]) * (uint32_t)(lda * 2) : NO_ROW; });
  opB.init(ldb, wv);
  const uint32_t ring0 = lds_address(ring);
  int ask_seg = 0, ask_k = 0;
  if constexpr (MODE == GATEUP || MODE == DOWN) {  // (the start that the other kernels take, for the same reason)
    if (p.K % 2048 == 0) ask_k = ((e * 13) & 31) * BK;
  }
  uint32_t ask_at = 0, at = 0;
  // (TO) a lane a row of the wave's; asked for before the k-tiles, so that it has arrived when the first of them have
  static_assert(!TO || FM <= 2, "a lane a row");
  int row_to = 0;
  if constexpr (TO) {
    const int r = row0 + wm * 32 * FM + lane;
    if (lane < 32 * FM && r < row_end) row_to = p.row_map[r];
  }
  const auto ask = [&](bool live) {
    const int seg = NSEG == 2 && ask_seg, left = p.K - ask_k;
    opA.load(ring0 + ask_at, wv, ring_rsrc(vA[seg], (long long)ask_k * 2, live), left);
    const uint32_t to = ring0 + ask_at + OpA::BYTES;
    if constexpr (B_OUTER) {
      opB.load(to, wv, ring_rsrc(vB[seg], (long long)ask_k * ldb * 2, live));
    } else {
      opB.load(to, wv, ring_rsrc(vB[0], (long long)ask_k * 2, live), left);
      if constexpr (DUAL) opB.load(to + OpB::BYTES, wv, ring_rsrc(vB[1], (long long)ask_k * 2, live), left);
    }
    ask_k += BK;
    if (ask_k >= p.K) ask_k = 0, ++ask_seg;
    ask_at = ask_at == (STAGES - 1) * O::STAGE ? 0 : ask_at + O::STAGE;
  };
#pragma unroll
  for (int i = 0; i < STAGES - 1; ++i) ask(i < steps);
  const auto placeA = OpA::place(wm * 32 * FM);
  const auto placeB = OpB::place(wn * (DUAL ? 32 : 64));
  f32x16 acc[FM][2];  // 32 rows x 32 columns each: two neighbours, or of gate and up
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][c][v] = 0.f;
  const bool idle = wm * 32 * FM >= row_end - row0;  // (such a wave only moves its share of the operands)
  for (int s = 0; s < steps; ++s) {
    ring_wait<(STAGES - 2) * O::LOADS>();
    const char *sa = ring + at, *sb = sa + OpA::BYTES;
    at = at == (STAGES - 1) * O::STAGE ? 0 : at + O::STAGE;
    if (idle) {
      ask(s + STAGES - 1 < steps);
      continue;
    }
    bf16x8 fa[2][FM], fb[2][2];
    const auto read = [&](int u, int ks) {
      if (u >= 2) fa[ks & 1][u - 2] = OpA::frag(sa, placeA, (u - 2) * 32, ks);
      else if (DUAL) fb[ks & 1][u] = OpB::frag(sb + u * OpB::BYTES, placeB, 0, ks);
      else fb[ks & 1][u] = OpB::frag(sb, placeB, u * 32, ks);
    };
#pragma unroll
    for (int u = 0; u < 2 + FM; ++u) read(u, 0);
    __builtin_amdgcn_sched_barrier(0);
    ask(s + STAGES - 1 < steps);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int n = 0; n < 2 * FM; ++n) {
        const int i = n / 2, c = (i & 1) ? 1 - n % 2 : n % 2;
        acc[i][c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fb[ks & 1][c], fa[ks & 1][i], acc[i][c], 0, 0, 0);
        if (ks + 1 < KS) {
          read(n, ks + 1);
          if (FM == 1 && n == 1) read(2, ks + 1);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
  }

  // ---- the epilogue, as in the other kernels: through a strip of the wave's own LDS
  constexpr int WTNC = DUAL ? 32 : 64;
  const int col_w0 = n0 + wn * WTNC, n_cb = (p.N + 31) / 32;
  const int row_w0 = row0 + wm * 32 * FM, rows = row_end - row_w0;
  const auto gu_block = [&](const void* base, int i, int cb) {
    return (char*)base + ((long long)(first / 32 + e + row / 32 + wm * FM + i) * n_cb + cb) * 4096 + lane * 16;
  };
  u32x4 gu[2][4];
  const auto load_gu = [&](int i) {
#pragma unroll
    for (int c = 0; c < 2; ++c) {
#pragma unroll
      for (int v = 0; v < 4; ++v) gu[c][v] = u32x4{0, 0, 0, 0};
      if (rows > i * 32 && col_w0 / 32 + c < n_cb) {
        const u32x4* rec = reinterpret_cast<const u32x4*>(gu_block(p.X0, i, col_w0 / 32 + c));
#pragma unroll
        for (int v = 0; v < 4; ++v) gu[c][v] = __builtin_nontemporal_load(rec + 64 * v);
      }
    }
  };
  if constexpr (MODE == DGRAD_DOWN) load_gu(0);
  ring_wait<0>();  // the strips lie in the stages
  if (idle) return;
  constexpr int STRIDE = WTNC * 2, CPS = STRIDE / 16, RPS = 64 / CPS;
  char* strip = ring + wv * 4096;
  const int ldc = p.ld_c ? p.ld_c : p.N, l32 = lane & 31, lh = lane >> 5;
  const auto perm = [&](int rr, int ch) { return CPS == 8 ? ch ^ ((rr >> 1) & 7) : ch ^ ((rr >> 2) & 3); };
  const auto put4 = [&](int c, int g4, u32x2 v) {
    *reinterpret_cast<u32x2*>(strip + l32 * STRIDE + perm(l32, c * 4 + g4) * 16 + lh * 8) = v;
  };
  const auto pack4 = [](float v0, float v1, float v2, float v3) { return u32x2{pack_bf16x2(v0, v1), pack_bf16x2(v2, v3)}; };
  const auto store_rows = [&](void* base, int strip_row) {
#pragma unroll
    for (int it = 0; it < 32 / RPS; ++it) {
      const int rr = it * RPS + lane / CPS, ch = lane % CPS, col = col_w0 + ch * 8;
      const u32x4 v = *reinterpret_cast<const u32x4*>(strip + rr * STRIDE + perm(rr, ch) * 16);
      const int to = TO ? __shfl(row_to, strip_row + rr, MOE_WAVE) : row_w0 + strip_row + rr;
      if (strip_row + rr < rows && col < p.N) *reinterpret_cast<u32x4*>((char*)base + ((long long)to * ldc + col) * 2) = v;
    }
  };
  if constexpr (MODE == GATEUP) {
#pragma unroll
    for (int i = 0; i < FM; ++i) {
      const bool keep = BLK && col_w0 / 32 < n_cb && rows > i * 32;
      u32x4* rec = keep ? reinterpret_cast<u32x4*>(gu_block(p.C0, i, col_w0 / 32)) : nullptr;
      u32x2 gq[2], uq[2];
#pragma unroll
      for (int g4 = 0; g4 < 4; ++g4) {
        float g[4], u[4], a[4];
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          g[v] = acc[i][0][4 * g4 + v];
          u[v] = acc[i][1][4 * g4 + v];
          a[v] = swiglu(g[v], u[v]);
        }
        put4(0, g4, pack4(a[0], a[1], a[2], a[3]));
        gq[g4 & 1] = pack4(g[0], g[1], g[2], g[3]);
        uq[g4 & 1] = pack4(u[0], u[1], u[2], u[3]);
        if (keep && (g4 & 1)) {
          __builtin_nontemporal_store(u32x4{gq[0][0], gq[0][1], gq[1][0], gq[1][1]}, rec + 64 * (g4 >> 1));
          __builtin_nontemporal_store(u32x4{uq[0][0], uq[0][1], uq[1][0], uq[1][1]}, rec + 128 + 64 * (g4 >> 1));
        }
      }
      store_rows(p.C2, i * 32);
    }
  } else if constexpr (MODE == DGRAD_DOWN) {
#pragma unroll
    for (int i = 0; i < FM; ++i) {
      float rowdot = 0.f;  // this lane's share of <dact[row,:], act[row,:]>
      u32x2 du4[2][4];
#pragma unroll
      for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int g4 = 0; g4 < 4; ++g4) {
          const u32x4 gv = gu[c][g4 >> 1], uv = gu[c][2 + (g4 >> 1)];
          const uint32_t g01 = gv[2 * (g4 & 1)], g23 = gv[2 * (g4 & 1) + 1], u01 = uv[2 * (g4 & 1)], u23 = uv[2 * (g4 & 1) + 1];
          const float g[4] = {bf16lo(g01), bf16hi(g01), bf16lo(g23), bf16hi(g23)};
          const float u[4] = {bf16lo(u01), bf16hi(u01), bf16lo(u23), bf16hi(u23)};
          float dg[4], du[4];
#pragma unroll
          for (int v = 0; v < 4; ++v) swiglu_bwd(acc[i][c][4 * g4 + v], g[v], u[v], dg[v], du[v], rowdot);
          put4(c, g4, pack4(dg[0], dg[1], dg[2], dg[3]));
          du4[c][g4] = pack4(du[0], du[1], du[2], du[3]);
        }
      if (i + 1 < FM) load_gu(i + 1);
      // one partial per 64 columns and row, every one of them written
      rowdot += __shfl_xor(rowdot, 32, MOE_WAVE);
      if (lh == 0 && i * 32 + l32 < rows && p.C2)
        reinterpret_cast<float*>(p.C2)[(long long)(col_w0 / 64) * p.R + row_w0 + i * 32 + l32] = rowdot;
      store_rows(p.C0, i * 32);
#pragma unroll
      for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int g4 = 0; g4 < 4; ++g4) put4(c, g4, du4[c][g4]);
      store_rows(p.C1, i * 32);
    }
  } else {
#pragma unroll
    for (int i = 0; i < FM; ++i) {
      const f32x16* r = acc[i];
#pragma unroll
      for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int g4 = 0; g4 < 4; ++g4) put4(c, g4, pack4(r[c][4 * g4], r[c][4 * g4 + 1], r[c][4 * g4 + 2], r[c][4 * g4 + 3]));
      store_rows(p.C0, i * 32);
    }
  }
}

}  // namespace
