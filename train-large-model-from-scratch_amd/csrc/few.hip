// Few tokens: the router with its selection, and the whole layer body for at most 64 tokens (moe_few_ok
// below has the line).
//
// Generation asks for the experts of one token, or of one token from each sequence of a batch.  What
// such a call cannot do without is one pass over the weights of the experts it asks for (one token of
// the 64-expert layer: 100 MB; 48 tokens: 800 MB, nearly all of them), and next to that a kernel's
// start and end are what costs.  So no kernel waits for another launch to sort rows: every workgroup finds
// the rows of its expert in the expert ids itself, rows stay in routed order, and for one token the selection
// is part of the gate/up kernel and the combine part of the down kernel.  The products run on
// v_mfma_f32_16x16x32_bf16, whose 16 rows are the tokens of an expert: weights go from memory straight to
// the operand registers, every byte once, with a wave's whole share of the contraction requested before
// the first product where it fits.
#include "common.h"
#include "gemm_args.h"
#include "topk_core.h"

namespace {

constexpr int DOWN_ONE_MAX_K = 32;
constexpr unsigned OUTSIDE = 0xfffffff0u;  // a byte offset past every resource: reads as zero

__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc(const void* base, long long bytes) {
  if (bytes > 0xffffffe0ll) bytes = 0xffffffe0ll;
  return __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, (int)(unsigned)bytes, 0x00020000);
}
__device__ __forceinline__ bf16x8 load_frag(__amdgpu_buffer_rsrc_t rs, unsigned off) {
  return __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(rs, (int)off, 0, 0));
}

// ---- router product ---------------------------------------------------------------------------------
// logits[t][e] = bf16(sum_h x[t][h] wr[e][h]) for 16 tokens and 16 experts a block; its 16 waves share the
// contraction (a contiguous sixteenth each, requested at once) and their sums are added in order.  What
// bounds it is one trip to memory; the library's product took 8-11 us and 18 us on the host.
constexpr int RT_WAVES = 16;
__global__ __launch_bounds__(RT_WAVES* MOE_WAVE) void router_few_kernel(const uint16_t* __restrict__ x,
                                                                       const uint16_t* __restrict__ wr, int T, int H,
                                                                       int E, uint16_t* __restrict__ logits) {
  constexpr int KC = 8;
  __shared__ float part[RT_WAVES][16][17];
  const int lane = lane_id(), wv = threadIdx.x / MOE_WAVE, l16 = lane & 15, lq = lane >> 4;
  const int e0 = blockIdx.x * 16, t0 = blockIdx.y * 16;
  const int steps = (H + 31) / 32, per = (steps + RT_WAVES - 1) / RT_WAVES;
  const int s_lo = wv * per, s_hi = s_lo + per < steps ? s_lo + per : steps;
  const __amdgpu_buffer_rsrc_t rx = rsrc(x + (size_t)t0 * H, (long long)(T - t0) * H * 2);
  const __amdgpu_buffer_rsrc_t rw = rsrc(wr + (size_t)e0 * H, (long long)(E - e0) * H * 2);
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  for (int s = s_lo; s < s_hi; s += KC) {
    bf16x8 a[KC], b[KC];
#pragma unroll
    for (int d = 0; d < KC; ++d) {
      const int kk = (s + d) * 32 + lq * 8;
      const unsigned off = s + d < s_hi && kk < H ? (unsigned)(l16 * H + kk) * 2 : OUTSIDE;
      a[d] = load_frag(rx, off);  // (rows past T, experts past E: past the resource's end)
      b[d] = load_frag(rw, off);
    }
#pragma unroll
    for (int d = 0; d < KC; ++d) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[d], b[d], acc, 0, 0, 0);
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) part[wv][lq * 4 + i][l16] = acc[i];
  __syncthreads();
  if (threadIdx.x < 256) {
    const int m = threadIdx.x >> 4, e = threadIdx.x & 15;
    float v = 0.f;
#pragma unroll
    for (int q = 0; q < RT_WAVES; ++q) v += part[q][m][e];
    if (t0 + m < T && e0 + e < E) logits[(size_t)(t0 + m) * E + e0 + e] = f32_to_bf16(v);
  }
}

// One token: a wave an expert, all of its 16-byte pieces requested before the first product where the row is at most
// 4096 wide.  As one column of 16 the matrix kernel above fills four workgroups of sixteen waves, whose start and sums
// cost more than the trip to memory: 64 experts, 2048 wide 5.4 -> 3.7 us (a token 30.5 -> 28.1).
constexpr int RO_WAVES = 4;
__global__ __launch_bounds__(RO_WAVES* MOE_WAVE) void router_one_kernel(const uint16_t* __restrict__ x,
                                                                       const uint16_t* __restrict__ wr, int H, int E,
                                                                       uint16_t* __restrict__ logits) {
  constexpr int KC = 8;
  const int lane = lane_id(), e = blockIdx.x * RO_WAVES + uniform((int)(threadIdx.x / MOE_WAVE));
  if (e >= E) return;
  const __amdgpu_buffer_rsrc_t rx = rsrc(x, (long long)H * 2), rw = rsrc(wr + (size_t)e * H, (long long)H * 2);
  float acc = 0.f;
  for (int h = 0; h < H; h += KC * MOE_WAVE * 8) {
    bf16x8 a[KC], b[KC];
#pragma unroll
    for (int d = 0; d < KC; ++d) {  // (past the row: zeros)
      const unsigned off = (unsigned)(h + (d * MOE_WAVE + lane) * 8) * 2;
      a[d] = load_frag(rx, off);
      b[d] = load_frag(rw, off);
    }
#pragma unroll
    for (int d = 0; d < KC; ++d) {
      const Row8 u = row8_from_bits(__builtin_bit_cast(u32x4, a[d])), v = row8_from_bits(__builtin_bit_cast(u32x4, b[d]));
#pragma unroll
      for (int i = 0; i < 8; ++i) acc += u.v[i] * v.v[i];
    }
  }
  acc = moe_wave_sum_f32(acc);
  if (lane == 0) logits[e] = f32_to_bf16(acc);
}

// ---- rows of one expert times its weights' columns ----------------------------------------------------
// Columns: KC 32-deep k-steps of 16 columns of NB weight stacks; rows: the same steps of MF blocks of 16 rows.
template <int NB, int KC>
struct Columns {
  bf16x8 v[NB][KC];
};
template <int MF, int KC>
struct Rows {
  bf16x8 v[MF][KC];
};
// Request steps s .. s + KC - 1 (those below s_end; the rest reads as zero).
template <int NB, int KC>
__device__ __forceinline__ void request(Columns<NB, KC>& c, const __amdgpu_buffer_rsrc_t (&w)[NB], bool live_col, int K,
                                        int s, int s_end) {
  const int lane = lane_id(), l16 = lane & 15, lq = lane >> 4;
#pragma unroll
  for (int d = 0; d < KC; ++d) {
    const int kk = (s + d) * 32 + lq * 8;
    const unsigned off = s + d < s_end && kk < K && live_col ? (unsigned)(l16 * K + kk) * 2 : OUTSIDE;
#pragma unroll
    for (int n = 0; n < NB; ++n) c.v[n][d] = load_frag(w[n], off);
  }
}
template <typename AT, int MF, int KC>
__device__ __forceinline__ void request(Rows<MF, KC>& r, const AT* const (&row)[MF] /* NULL: no such row */, int K, int s,
                                        int s_end) {
  const int lq = lane_id() >> 4;
#pragma unroll
  for (int d = 0; d < KC; ++d) {
    const int kk = (s + d) * 32 + lq * 8;
    const bool in = s + d < s_end && kk < K;
#pragma unroll
    for (int m = 0; m < MF; ++m) {
      u32x4 v = {0, 0, 0, 0};
      if (in && row[m]) {
        if constexpr (sizeof(AT) == 2) {
          v = *reinterpret_cast<const u32x4*>(row[m] + kk);
        } else {
          const Row8 f = load8(row[m] + kk);
#pragma unroll
          for (int i = 0; i < 4; ++i) v[i] = pack_bf16x2(f.v[2 * i], f.v[2 * i + 1]);
        }
      }
      r.v[m][d] = __builtin_bit_cast(bf16x8, v);
    }
  }
}
template <int NB, int MF, int KC>
__device__ __forceinline__ void multiply(const Rows<MF, KC>& r, const Columns<NB, KC>& c, f32x4 (&acc)[NB][MF]) {
#pragma unroll
  for (int d = 0; d < KC; ++d)
#pragma unroll
    for (int m = 0; m < MF; ++m)
#pragma unroll
      for (int n = 0; n < NB; ++n)
        acc[n][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(r.v[m][d], c.v[n][d], acc[n][m], 0, 0, 0);
}

// The routed rows of expert e, listed in LDS by the whole workgroup (the order is left to chance: a row's
// result does not depend on its place in the list); their number comes back.
__device__ __forceinline__ int list_rows(const int32_t* __restrict__ ids, int R, int E, int e, int* rows, int* count) {
  if (threadIdx.x == 0) *count = 0;
  __syncthreads();
  for (int r = threadIdx.x; r < R; r += blockDim.x) {
    int id = ids[r];
    id = id < 0 ? 0 : (id >= E ? E - 1 : id);
    if (id == e) {
      const int at = atomicAdd(count, 1);
      if (at < FEW_MAX_TOKENS) rows[at] = r;
    }
  }
  __syncthreads();
  return *count < FEW_MAX_TOKENS ? *count : FEW_MAX_TOKENS;
}

// One expert's rows times `nblk` blocks of 16 columns of NB weight stacks [E,N,K], the four waves a contiguous
// quarter of the contraction each.  NB = 2: gate and up, C = silu(g) u; NB = 1: down, C = y.  Rows of A are
// tokens (a routed row's token is row / div) or routed rows (div = 1); rows of C are routed rows.
// The blocks' chunks (KC k-steps) are one stream: while a chunk is multiplied (or a block's partial sums are
// added through LDS) the next one is on its way, so that a workgroup never stops asking for weights.
// KEEP > 0: a wave's share of the contraction is KEEP chunks, and its rows stay in registers for all blocks
// (asked for again with every block they cost an eighth of the time: 48 tokens of the 64-expert layer,
// gate and up 0.54 GB, 109 -> 97 us, 5.5 TB/s; a plain read loop over as much runs at 6.2-6.9).
template <typename AT, int NB, int MF, int KC, int KEEP>
__device__ __forceinline__ void few_columns(const AT* __restrict__ A, int div, const uint16_t* const (&w)[NB], int e,
                                            int n0, int nblk, int N, int K, const int* rows, int n, float* part,
                                            uint16_t* __restrict__ C) {
  const int lane = lane_id(), wv = threadIdx.x / MOE_WAVE, l16 = lane & 15, lq = lane >> 4;
  const int steps = (K + 31) / 32, per = ((steps + 3) / 4 + 1) & ~1;
  const int s_lo = wv * per, s_hi = s_lo + per < steps ? s_lo + per : steps;
  const int chunks = KEEP ? KEEP : (per + KC - 1) / KC;  // per block, the same for every wave
  const AT* row[MF];
#pragma unroll
  for (int m = 0; m < MF; ++m) row[m] = m * 16 + l16 < n ? A + (size_t)(rows[m * 16 + l16] / div) * K : nullptr;
  f32x4 acc[NB][MF];
  const auto clear = [&]() {
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int m = 0; m < MF; ++m) acc[b][m] = f32x4{0.f, 0.f, 0.f, 0.f};
  };
  int rb = 0, rc = 0;  // block and chunk of the next request
  const auto ask = [&](Columns<NB, KC>& c) {
    const int col = n0 + rb * 16;
    __amdgpu_buffer_rsrc_t rs[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) rs[b] = rsrc(w[b] + ((size_t)e * N + col) * K, (long long)(N - col) * K * 2);
    request<NB, KC>(c, rs, col + l16 < N, K, s_lo + rc * KC, s_hi);
    if (++rc == chunks) rc = 0, ++rb;
  };
  int mb = 0;  // block of the current product
  const auto finish = [&]() {
    // part [2][4][NB][MF][4][64]: the four waves' sums of this block (two buffers: a wave that runs ahead
    // writes the other one)
    float* buf = part + (mb & 1) * (4 * NB * MF * 256);
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int m = 0; m < MF; ++m)
#pragma unroll
        for (int q = 0; q < 4; ++q) buf[((wv * NB + b) * MF + m) * 256 + q * MOE_WAVE + lane] = acc[b][m][q];
    clear();
    __syncthreads();
    const int col = n0 + mb * 16 + l16;
#pragma unroll
    for (int m = 0; m < MF; ++m) {  // wave q: rows 16 m + 4 lq + q
      float v[NB];
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        v[b] = 0.f;
#pragma unroll
        for (int i = 0; i < 4; ++i) v[b] += buf[((i * NB + b) * MF + m) * 256 + wv * MOE_WAVE + lane];
      }
      const int at = m * 16 + lq * 4 + wv;
      if (at < n && col < N) C[(size_t)rows[at] * N + col] = f32_to_bf16(NB == 2 ? swiglu(v[0], v[NB - 1]) : v[0]);
    }
    ++mb;
  };
  Columns<NB, KC> c0, c1;
  clear();
  ask(c0);
  const int total = nblk * chunks;
  if constexpr (KEEP > 0) {
    Rows<MF, KC> r[KEEP];
#pragma unroll
    for (int i = 0; i < KEEP; ++i) request<AT, MF, KC>(r[i], row, K, s_lo + i * KC, s_hi);
    for (int i = 0; i < total; i += 2) {
      if (i + 1 < total) ask(c1);
      multiply<NB, MF, KC>(r[0], c0, acc);
      if (KEEP == 1) finish();
      if (i + 1 >= total) break;
      if (i + 2 < total) ask(c0);
      multiply<NB, MF, KC>(r[KEEP - 1], c1, acc);
      finish();
    }
  } else {
    Rows<MF, KC> r0, r1;
    int mc = 0;
    request<AT, MF, KC>(r0, row, K, s_lo, s_hi);
    const auto next_rows = [&](Rows<MF, KC>& r, int i) { request<AT, MF, KC>(r, row, K, s_lo + i % chunks * KC, s_hi); };
    for (int i = 0; i < total; i += 2) {
      if (i + 1 < total) ask(c1), next_rows(r1, i + 1);
      multiply<NB, MF, KC>(r0, c0, acc);
      if (++mc == chunks) mc = 0, finish();
      if (i + 1 >= total) break;
      if (i + 2 < total) ask(c0), next_rows(r0, i + 2);
      multiply<NB, MF, KC>(r1, c1, acc);
      if (++mc == chunks) mc = 0, finish();
    }
  }
}

// At most 16 rows: they stay in registers where a wave's share of the contraction is at most 16 steps.
template <typename AT, int NB>
__device__ __forceinline__ void few_columns_16(const AT* __restrict__ A, int div, const uint16_t* const (&w)[NB], int e,
                                               int n0, int nblk, int N, int K, const int* rows, int n, float* part,
                                               uint16_t* __restrict__ C) {
  const int per = ((((K + 31) / 32) + 3) / 4 + 1) & ~1;
  if (per <= 8) few_columns<AT, NB, 1, 8, 1>(A, div, w, e, n0, nblk, N, K, rows, n, part, C);
  else if (per <= 16) few_columns<AT, NB, 1, 8, 2>(A, div, w, e, n0, nblk, N, K, rows, n, part, C);
  else few_columns<AT, NB, 1, 8, 0>(A, div, w, e, n0, nblk, N, K, rows, n, part, C);
}

// The selection, made where it is needed.  A single token's by every wave for itself (128 experts: in about the time its ids would take to
// arrive, where a launch of its own costs more: 64 experts, 2048 <-> 1024, 33.5 -> 32.1 us a
// token; 128 experts, 1024 <-> 256, 28.2 -> 25.0).
struct Selection {
  const void* logits;
  const float* bias;
  int32_t* ids;  // results, written by the first workgroup
  float* gates;
  int logits_f32, k;
};
template <int VPL>
__device__ __forceinline__ void token_keys(const Selection& sel, int t, int E, uint32_t (&key)[VPL]) {
  if (sel.logits_f32) moe_topk_keys<VPL>((const float*)sel.logits + (size_t)t * E, sel.bias, E, lane_id(), key);
  else moe_topk_keys<VPL>((const uint16_t*)sel.logits + (size_t)t * E, sel.bias, E, lane_id(), key);
}
// The rows of expert e from the logits of T tokens, as list_rows makes them from the ids: a token asks for it if fewer than k of its
// experts come before e, and that many is the slot.  A wave a token, a comparison and a ballot each, so that
// the selection of a few tokens is no launch of its own (moe_gateup_few_selects has the line).
template <int VPL>
__device__ __forceinline__ int list_selected_rows(const Selection& sel, int T, int E, int e, int* rows, int* count) {
  constexpr int AHEAD = 4;
  const int lane = lane_id(), wv = uniform((int)(threadIdx.x / MOE_WAVE)), waves = blockDim.x / MOE_WAVE;
  if (threadIdx.x == 0) *count = 0;
  __syncthreads();
  for (int t0 = wv; t0 < T; t0 += AHEAD * waves) {
    uint32_t key[AHEAD][VPL];
#pragma unroll
    for (int i = 0; i < AHEAD; ++i)
      if (t0 + i * waves < T) token_keys<VPL>(sel, t0 + i * waves, E, key[i]);
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) {
      const int t = t0 + i * waves;
      if (t >= T) break;
      const uint32_t own = e < MOE_WAVE ? read_lane(key[i][0], e) : read_lane(key[i][VPL - 1], e - MOE_WAVE);
      int before = 0;
#pragma unroll
      for (int v = 0; v < VPL; ++v)
        before += __popcll(__ballot(key[i][v] > own || (key[i][v] == own && v * MOE_WAVE + lane < e)));
      if (before < sel.k && lane == 0) rows[atomicAdd(count, 1)] = t * sel.k + before;
    }
  }
  __syncthreads();
  return *count;
}

// ONE: a single token; block row j takes its j-th expert and no list is needed.  VPL > 0: which one that is, and else which rows
// an expert has, comes from the logits of at most 64 * VPL experts, not from ids.
template <typename AT, int NB, bool ONE, int VPL = 0>
__global__ __launch_bounds__(256, 2) void few_kernel(const AT* __restrict__ A, int div, const int32_t* __restrict__ ids,
                                                    int R, const uint16_t* __restrict__ w0,
                                                    const uint16_t* __restrict__ w1, int E, int N, int K, int nblk,
                                                    uint16_t* __restrict__ C, const Selection sel) {
  __shared__ int rows[FEW_MAX_TOKENS], count;
  __shared__ float part[2 * 4 * NB * (ONE ? 1 : 4) * 256];
  const uint16_t* w[NB];
  w[0] = w0;
  if constexpr (NB == 2) w[1] = w1;
  const int n0 = blockIdx.x * nblk * 16, left = (N - n0 + 15) / 16;
  const int nb = left < nblk ? left : nblk;
  if constexpr (ONE) {
    const int j = blockIdx.y;
    int e;
    if constexpr (VPL > 0) {
      const int lane = lane_id();
      uint32_t key[VPL];
      if (sel.logits_f32) moe_topk_keys<VPL>((const float*)sel.logits, sel.bias, E, lane, key);
      else moe_topk_keys<VPL>((const uint16_t*)sel.logits, sel.bias, E, lane, key);
      int id;
      float gate;
      moe_topk_softmax_wave<VPL>(key, sel.k, lane, id, gate);
      if (blockIdx.x == 0 && j == 0 && threadIdx.x < sel.k) {
        sel.ids[lane] = id;
        sel.gates[lane] = gate;
      }
      e = __builtin_amdgcn_readlane(id, j);
    } else {
      e = ids[j];
    }
    e = e < 0 ? 0 : (e >= E ? E - 1 : e);
    if (threadIdx.x == 0) rows[0] = j;
    __syncthreads();
    few_columns_16<AT, NB>(A, div, w, e, n0, nb, N, K, rows, 1, part, C);
  } else {
    const int e = blockIdx.y;
    int n;
    if constexpr (VPL > 0) {
      const int T = R / sel.k;
      n = list_selected_rows<VPL>(sel, T, E, e, rows, &count);
    } else {
      n = list_rows(ids, R, E, e, rows, &count);
    }
    if (n > 0) {
      if (n <= 16) few_columns_16<AT, NB>(A, div, w, e, n0, nb, N, K, rows, n, part, C);
      else if (n <= 32) few_columns<AT, NB, 2, 4, 0>(A, div, w, e, n0, nb, N, K, rows, n, part, C);
      else few_columns<AT, NB, 4, 2, 0>(A, div, w, e, n0, nb, N, K, rows, n, part, C);
    }
    if constexpr (VPL > 0) {  // the launches that follow read ids and gates: the first workgroups leave a token's each, at their end
      const int T = R / sel.k;
      if (threadIdx.x < MOE_WAVE) {
        const int lane = lane_id();
        for (int t = blockIdx.y * gridDim.x + blockIdx.x; t < T; t += gridDim.x * gridDim.y) {
          uint32_t key[VPL];
          token_keys<VPL>(sel, t, E, key);
          int id;
          float gate;
          moe_topk_softmax_wave<VPL>(key, sel.k, lane, id, gate);
          if (lane < sel.k) {
            sel.ids[(size_t)t * sel.k + lane] = id;
            sel.gates[(size_t)t * sel.k + lane] = gate;
          }
        }
      }
    }
  }
}

// ---- down projection and combine of one token -----------------------------------------------------------------
// out[h] = sum_j gate[j] bf16(y[j][h]) for the COLS columns h of this block: the block's eight waves take the
// token's experts in turn (or shares of their contractions, where fewer than eight are asked for) and leave
// their sums in LDS, where they are added up in slot order, as the combine kernel does.
// COLS = 8: the product's 16 columns are 8 columns twice, once for each half of the share (row 0 of the other operand is the
// first half of the token's row, row 1 the second), so that twice the workgroups ask for weights.
// (One token, 64 experts, 2048 <-> 1024, k = 8, the whole layer: 32.7 -> 31.0 us; k = 2 and 4: no difference.)
constexpr int DOWN_WAVES = 8;
template <typename OT, int COLS>
__global__ __launch_bounds__(DOWN_WAVES* MOE_WAVE) void down_one_kernel(const uint16_t* __restrict__ act,
                                                                       const int32_t* __restrict__ ids,
                                                                       const float* __restrict__ gates, int k,
                                                                       const uint16_t* __restrict__ w2, int E, int H,
                                                                       int I, OT* __restrict__ out) {
  constexpr int PARTS = 16 / COLS;                                   // of a share
  constexpr int KC = 32 / PARTS;                                     // k-steps of a part requested at once
  __shared__ float y[DOWN_WAVES + DOWN_ONE_MAX_K][16];               // [splits][k]
  __shared__ __align__(16) uint16_t arow[DOWN_WAVES][32 * 32];       // a wave's pieces of its row of act
  const int lane = lane_id(), wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / MOE_WAVE)), l16 = lane & 15,
            lq = lane >> 4;
  const int h0 = blockIdx.x * COLS;
  const int col = l16 % COLS, part = l16 / COLS;
  const int splits = k >= DOWN_WAVES ? 1 : DOWN_WAVES / k;
  const int steps = (I + 31) / 32, per = ((steps + splits * PARTS - 1) / (splits * PARTS) + 1) & ~1;  // of a part
  for (int item = wv; item < k * splits; item += DOWN_WAVES) {
    const int j = item / splits, sp = item - j * splits;
    int e = __builtin_amdgcn_readfirstlane(ids[j]);
    e = e < 0 ? 0 : (e >= E ? E - 1 : e);
    const int s_lo = sp * PARTS * per;                               // of the first part
    const auto end_of = [&](int p) { return s_lo + (p + 1) * per < steps ? s_lo + (p + 1) * per : steps; };
    const __amdgpu_buffer_rsrc_t rw = rsrc(w2 + ((size_t)e * H + h0) * I, (long long)(H - h0) * I * 2);
    // (an undivided share's activations end where the share does: past it they must not count, not even times a weight
    // of zero, since they may be infinite.  The resource's end costs nothing; a test a lane took 1-2 % of the call.)
    const int a_end = PARTS == 1 && end_of(0) * 32 < I ? end_of(0) * 32 : I;
    const __amdgpu_buffer_rsrc_t ra = rsrc(act + (size_t)j * I, (long long)a_end * 2);
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    for (int s = 0; s < per; s += KC) {
      const int first = s_lo + part * per + s, end = end_of(part);
      bf16x8 w[KC];
#pragma unroll
      for (int d = 0; d < KC; ++d) {
        const int kk = (first + d) * 32 + lq * 8;
        const bool in = (PARTS == 1 || s + d < per) && first + d < end && kk < I && h0 + col < H;
        w[d] = load_frag(rw, in ? (unsigned)(col * I + kk) * 2 : OUTSIDE);
      }
      // (a single row: in operand layout 15 of 16 lanes would carry zeros, so it comes through LDS)
#pragma unroll
      for (int i = 0; i < 32 * 32 / (MOE_WAVE * 8); ++i) {
        const int at = (i * MOE_WAVE + lane) * 8, p = at / (KC * 32), in_p = at % (KC * 32);
        const int step = s + in_p / 32;
        const bool in = PARTS == 1 || (step < per && s_lo + p * per + step < end_of(p));  // (the next part's must not count)
        *reinterpret_cast<bf16x8*>(&arow[wv][at]) =
            load_frag(ra, in ? (unsigned)((s_lo + p * per + s) * 32 + in_p) * 2 : OUTSIDE);
      }
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int d = 0; d < KC; ++d) {  // operand row p: part p
        bf16x8 a = *reinterpret_cast<const bf16x8*>(&arow[wv][(l16 % PARTS) * KC * 32 + d * 32 + lq * 8]);
        if (l16 >= PARTS) a = __builtin_bit_cast(bf16x8, u32x4{0, 0, 0, 0});
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, w[d], acc, 0, 0, 0);
      }
      __builtin_amdgcn_wave_barrier();
    }
    if (lq == 0) y[sp * k + j][l16] = part == 0 ? acc[0] : acc[1];  // row `part` of the product
  }
  __syncthreads();
  if (threadIdx.x < COLS && h0 + threadIdx.x < H) {
    const int c = threadIdx.x;
    float sum = 0.f;
    for (int j = 0; j < k; ++j) {
      float v = y[j][c];
      if constexpr (PARTS == 2) v += y[j][COLS + c];
      for (int sp = 1; sp < splits; ++sp) {
        v += y[sp * k + j][c];
        if constexpr (PARTS == 2) v += y[sp * k + j][COLS + c];
      }
      sum += gates[j] * bf16_to_f32(f32_to_bf16(v));
    }
    if constexpr (sizeof(OT) == 2) out[h0 + c] = f32_to_bf16(sum);
    else out[h0 + c] = sum;
  }
}

}  // namespace

bool moe_router_few_ok(int64_t T, int64_t H, int64_t E, int64_t k) {
  // (a large batch takes the library's product: there the few logits that round the other way would now
  // and then select another expert than a caller's own product of the same tensors)
  return T > 0 && T <= FEW_MAX_TOKENS && H <= 65536 && E <= FEW_MAX_EXPERTS && k <= E && k <= MOE_MAX_TOPK;
}

int moe_router_few(const uint16_t* x, const uint16_t* wr, int64_t T, int64_t H, int64_t E, uint16_t* logits,
                   hipStream_t s) {
  if (T == 1) {
    hipLaunchKernelGGL(router_one_kernel, dim3((unsigned)((E + RO_WAVES - 1) / RO_WAVES)), dim3(RO_WAVES * MOE_WAVE), 0, s, x,
                       wr, (int)H, (int)E, logits);
    return moe_launch_status();
  }
  const dim3 grid((unsigned)((E + 15) / 16), (unsigned)((T + 15) / 16));
  hipLaunchKernelGGL(router_few_kernel, grid, dim3(RT_WAVES * MOE_WAVE), 0, s, x, wr, (int)T, (int)H, (int)E, logits);
  return moe_launch_status();
}

// At most 64 tokens: an expert's rows then fit four blocks of 16, and all of them the lists.  (The tiled
// kernels take 256 rows at a time, of which 1 to 64 are there.)
// Where the experts have more than 8 rows each, those rows are what an expert's workgroups load again with every block of
// columns, while the tiled kernels' time stays as it is.  The line: rows past 8 an expert times an expert's weights,
// 2.5 GB (fp32 rows count twice); at most 8 experts leave compute units without a tile, so 5 GB there.  Whole layer, us,
// these kernels against the tiled ones: 16 experts, 2048 <-> 1024, at 8 / 16 / 24 / 32 rows each (0 / 1.6 / 3.2 /
// 4.8 GB) 49 / 62 / 72 / 84 against 67 / 69 / 69 / 70; 12 experts, 4096 <-> 2048, at 8 / 12 / 20 / 32 (0 / 2.4 / 7.2 / 14)
// 131 / 153 / 180 / 240 against 135 / 145 / 147 / 149; 8 experts, 4096 <-> 2048, at 16 / 24 / 32 (3.2 / 6.4 / 9.7) 109 / 126 /
// 148 against 123 / 124 / 126, and 4096 <-> 1024 at 32 (4.8) 78 against 92; 8 experts, 4096 <-> 2048, fp32 rows, at 12 / 16
// (3.2 / 6.4) 115 / 144 against 124.  At up to 8 rows each these kernels take from a third of the time (few or
// small experts) to 1.08 times (64 experts of 50 MB).
bool moe_few_ok(int64_t T, int64_t H, int64_t E, int64_t I, int64_t k, int x_dtype) {
  if (T <= 0 || T > FEW_MAX_TOKENS || E > 65535 || H > 65536 || I > 65536) return false;
  const double again = (double)(T * k - 8 * E) * 6.0 * (double)H * (double)I * (x_dtype == MOE_DT_F32 ? 2 : 1);
  return again <= (E <= 8 ? 5e9 : 2.5e9);
}

namespace {
// 16-column blocks per workgroup: as many as leave two workgroups for every compute unit (two are resident)
// if `busy` experts are asked for.
int few_blocks(int64_t N, int64_t busy) {
  const int64_t blocks = (N + 15) / 16, fit = blocks * busy / (4 * (int64_t)moe_compute_units());
  return (int)(fit < 1 ? 1 : (fit > 8 ? 8 : fit));
}
}  // namespace

int moe_gateup_few(const void* x, int x_dtype, const int32_t* ids, const uint16_t* w1, const uint16_t* w3, int64_t T,
                   int64_t H, int64_t E, int64_t I, int64_t k, uint16_t* act, hipStream_t s) {
  const int nblk = few_blocks(I, T * k < E ? T * k : E);
  const dim3 grid((unsigned)(((I + 15) / 16 + nblk - 1) / nblk), (unsigned)(T == 1 ? k : E)), block(256);
  const auto go = [&](auto one, auto xt) {
    using XT = decltype(xt);
    hipLaunchKernelGGL((few_kernel<XT, 2, decltype(one)::value>), grid, block, 0, s, (const XT*)x, (int)k, ids, (int)(T * k),
                       w1, w3, (int)E, (int)I, (int)H, nblk, act, Selection{});
    return moe_launch_status();
  };
  if (x_dtype == MOE_DT_BF16) return T == 1 ? go(std::true_type{}, uint16_t{}) : go(std::false_type{}, uint16_t{});
  return T == 1 ? go(std::true_type{}, float{}) : go(std::false_type{}, float{});
}

// Every workgroup of gate/up goes through all tokens, four at a time: up to 2048 such turns in all they cost less than the
// launch they save.  A whole call, us, with the launch and without: 2 tokens, 6 of 24 experts, 448 <-> 192 (288 turns) 32 -> 29; 5, 3
// of 64, 320 <-> 192 (1536) 33 -> 29; 13, 1 of 4, 832 <-> 448 (448) 34 -> 30; 11, 8 of 64, 1088 <-> 192 (2304, not taken) 37 -> 37; 27, 6 of 64,
// 896 <-> 384 (10752) 43 -> 47; 48, 8 of 64, 2048 <-> 1024 (12288) 164 -> 165.5.
bool moe_gateup_few_selects(int64_t T, int64_t E, int64_t I, int64_t k) {
  const int64_t nblk = few_blocks(I, T * k < E ? T * k : E);
  return T > 1 && E <= 2 * MOE_WAVE && ((I + 15) / 16 + nblk - 1) / nblk * E * ((T + 3) / 4) <= 2048;
}

int moe_gateup_few_select(const void* x, int x_dtype, const void* logits, int logits_dtype, const float* bias, const uint16_t* w1,
                          const uint16_t* w3, int64_t T, int64_t H, int64_t E, int64_t I, int64_t k, int32_t* ids, float* gates,
                          uint16_t* act, hipStream_t s) {
  const int nblk = few_blocks(I, T * k < E ? T * k : E);
  const dim3 grid((unsigned)(((I + 15) / 16 + nblk - 1) / nblk), (unsigned)E), block(256);
  const Selection sel{logits, bias, ids, gates, logits_dtype == MOE_DT_F32, (int)k};
  const auto go = [&](auto vpl, auto xt) {
    using XT = decltype(xt);
    hipLaunchKernelGGL((few_kernel<XT, 2, false, decltype(vpl)::value>), grid, block, 0, s, (const XT*)x, (int)k, nullptr,
                       (int)(T * k), w1, w3, (int)E, (int)I, (int)H, nblk, act, sel);
    return moe_launch_status();
  };
  using One = std::integral_constant<int, 1>;
  using Two = std::integral_constant<int, 2>;
  if (x_dtype == MOE_DT_BF16) return E <= MOE_WAVE ? go(One{}, uint16_t{}) : go(Two{}, uint16_t{});
  return E <= MOE_WAVE ? go(One{}, float{}) : go(Two{}, float{});
}

int moe_down_few(const uint16_t* act, const int32_t* ids, const uint16_t* w2, int64_t T, int64_t H, int64_t E, int64_t I,
                 int64_t k, uint16_t* y, hipStream_t s) {
  const int nblk = few_blocks(H, T * k < E ? T * k : E);
  const dim3 grid((unsigned)(((H + 15) / 16 + nblk - 1) / nblk), (unsigned)E), block(256);
  hipLaunchKernelGGL((few_kernel<uint16_t, 1, false>), grid, block, 0, s, act, 1, ids, (int)(T * k), w2, nullptr, (int)E,
                     (int)H, (int)I, nblk, y, Selection{});
  return moe_launch_status();
}

// (64 threads of the first workgroup write the results)
bool moe_gateup_one_ok(int64_t T, int64_t E, int64_t k) { return moe_down_one_ok(T, k) && E <= 2 * MOE_WAVE; }

int moe_gateup_one(const void* x, int x_dtype, const void* logits, int logits_dtype, const float* bias, const uint16_t* w1,
                   const uint16_t* w3, int64_t H, int64_t E, int64_t I, int64_t k, int32_t* ids, float* gates,
                   uint16_t* act, hipStream_t s) {
  const int nblk = few_blocks(I, k);
  const dim3 grid((unsigned)(((I + 15) / 16 + nblk - 1) / nblk), (unsigned)k), block(256);
  const Selection sel{logits, bias, ids, gates, logits_dtype == MOE_DT_F32, (int)k};
  const auto go = [&](auto vpl, auto xt) {
    using XT = decltype(xt);
    hipLaunchKernelGGL((few_kernel<XT, 2, true, decltype(vpl)::value>), grid, block, 0, s, (const XT*)x, (int)k, nullptr,
                       (int)k, w1, w3, (int)E, (int)I, (int)H, nblk, act, sel);
    return moe_launch_status();
  };
  using One = std::integral_constant<int, 1>;
  using Two = std::integral_constant<int, 2>;
  if (x_dtype == MOE_DT_BF16) return E <= MOE_WAVE ? go(One{}, uint16_t{}) : go(Two{}, uint16_t{});
  return E <= MOE_WAVE ? go(One{}, float{}) : go(Two{}, float{});
}

bool moe_down_one_ok(int64_t T, int64_t k) { return T == 1 && k <= DOWN_ONE_MAX_K; }

int moe_down_one(const uint16_t* act, const int32_t* ids, const float* gates, const uint16_t* w2, int64_t H, int64_t E,
                 int64_t I, int64_t k, void* out, int out_dtype, hipStream_t s) {
  // (more workgroups than compute units of the narrow kind: 2880 columns, 32.3 -> 34.0 us a token)
  const bool wide = (H + 7) / 8 > moe_compute_units();
  const auto go = [&](auto cols, auto ot) {
    using OT = decltype(ot);
    constexpr int COLS = decltype(cols)::value;
    hipLaunchKernelGGL((down_one_kernel<OT, COLS>), dim3((unsigned)((H + COLS - 1) / COLS)), dim3(DOWN_WAVES * MOE_WAVE), 0,
                       s, act, ids, gates, (int)k, w2, (int)E, (int)H, (int)I, (OT*)out);
    return moe_launch_status();
  };
  using Narrow = std::integral_constant<int, 8>;
  using Wide = std::integral_constant<int, 16>;
  if (out_dtype == MOE_DT_BF16) return wide ? go(Wide{}, uint16_t{}) : go(Narrow{}, uint16_t{});
  return wide ? go(Wide{}, float{}) : go(Narrow{}, float{});
}
