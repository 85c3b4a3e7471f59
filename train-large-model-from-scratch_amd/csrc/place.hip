// From logits to rows in expert order in two launches: selection with counts, then places and rows.
//
// The general path (route.hip, dispatch.hip) takes four or five: selection, histograms, their scan, positions, rows.
// Each of the middle ones moves a few KB and lasts as long as a launch does, 4 to 7 us.  Here the selection's
// workgroups count their own 16 tokens, a byte an expert, and every workgroup of the second launch adds up the
// bytes in front of it for itself, while its rows are on their way from memory.  The permutation is the same one: a
// token asks for an expert at most once, so rows of an expert in the order of their tokens is the stable order.
// From the selection's start to the rows' end, us, the general path and here: 2048 tokens, 8 experts, 1024 wide 16.9, 10.6;
// 1531 tokens, 64 experts, 8 a token, 2048 wide 35.9, 17.4; 8192 tokens, 8 experts 32.9, 17.2; 512 tokens 15.6, 9.6.
#include "common.h"
#include "internal.h"
#include "topk_core.h"

namespace {

constexpr int PLACE_EXPERTS = 2 * MOE_WAVE;
constexpr int CHUNK = MOE_PLACE_CHUNK;  // tokens counted together, one a wave of a selection's workgroup

// Bytes of counts, all of which every placing workgroup reads: their number times the tokens is what makes the two launches
// the slower ones in the end.  General path -> these, from the selection's start to the rows' end, us: 128 experts, 8 a
// token, 1024 wide, 4096 tokens (32 KB) 37 -> 23, 8192 (64 KB) 55 -> 42, 16384 (128 KB) 93 -> 81; 1 a token, where there is least
// else to do, 8192 28 -> 19, 12000 (94 KB) 31 -> 30, 16384 36 -> 39; 64 experts, 8 a token, 512 wide, 24000 (94 KB) 77 -> 69; 8
// experts, 2 a token, 1024 wide, 60000 (30 KB) 113 -> 105.  (Chunks of 8 tokens, a table of twice the size: 30 of the first;
// 1531 tokens of 64 experts, 2048 wide, 18.3 where 16 take 17.4; 256 tokens of 128 experts 10.0 and 10.3.)
constexpr int64_t PLACE_TABLE = 96 * 1024;

int words_of(int64_t E) { return (int)((E + 3) / 4); }

// One wave a token, as router_topk_fwd_kernel; table[chunk][e] = how many of the chunk's tokens ask for e.
template <int VPL, typename LT>
__global__ __launch_bounds__(CHUNK* MOE_WAVE) void select_count_kernel(const LT* __restrict__ logits,
                                                                      const float* __restrict__ bias, int T, int E, int k,
                                                                      int32_t* __restrict__ ids, float* __restrict__ gates,
                                                                      uint32_t* __restrict__ table) {
  __shared__ uint32_t asked[PLACE_EXPERTS];  // bit t: token t of the chunk asks for the expert
  const int lane = lane_id(), wv = uniform((int)(threadIdx.x / MOE_WAVE));
  if (threadIdx.x < PLACE_EXPERTS) asked[threadIdx.x] = 0;
  __syncthreads();
  const int t = blockIdx.x * CHUNK + wv;
  if (t < T) {
    uint32_t key[VPL];
    moe_topk_keys<VPL>(logits + (size_t)t * E, bias, E, lane, key);
    int id;
    float gate;
    moe_topk_softmax_wave<VPL>(key, k, lane, id, gate);
    if (lane < k) {
      ids[(size_t)t * k + lane] = id;
      gates[(size_t)t * k + lane] = gate;
      atomicOr(&asked[id], 1u << wv);
    }
  }
  __syncthreads();
  const int words = (E + 3) / 4;
  if (threadIdx.x < words) {
    uint32_t w = 0;
#pragma unroll
    for (int b = 0; b < 4; ++b) w |= (uint32_t)__popc(asked[threadIdx.x * 4 + b]) << (8 * b);
    table[(size_t)blockIdx.x * words + threadIdx.x] = w;
  }
}

// The table where the experts are given, one a row: an id outside [0, E) counts for the nearest expert, as in dispatch.hip, and
// bad[chunk] is how many of the chunk's are.  With `narrowed` the ids are also left there in 32 bits.
template <typename IT>
__global__ __launch_bounds__(256) void count_ids_kernel(const IT* __restrict__ ids, int T, int E, int32_t* __restrict__ narrowed,
                                                        uint32_t* __restrict__ table, uint32_t* __restrict__ bad) {
  constexpr int CHUNKS = 256 / CHUNK;
  __shared__ uint32_t counts[CHUNKS][PLACE_EXPERTS / 4];  // a byte an expert: a chunk has 16 rows
  const int t = blockIdx.x * 256 + threadIdx.x, lane = lane_id(), words = (E + 3) / 4;
  for (int i = threadIdx.x; i < CHUNKS * PLACE_EXPERTS / 4; i += 256) counts[0][i] = 0;
  __syncthreads();
  bool outside = false;
  if (t < T) {
    const IT v = ids[t];
    const int id = v < 0 || (int64_t)v > 0x7fffffffll ? -1 : (int)v;
    if (narrowed) narrowed[t] = id;
    const int e = id < 0 ? 0 : id >= E ? E - 1 : id;
    outside = e != id;
    atomicAdd(&counts[threadIdx.x / CHUNK][e >> 2], 1u << (8 * (e & 3)));
  }
  const unsigned long long who = __ballot(outside);
  if (t < T && lane % CHUNK == 0) bad[t / CHUNK] = __popcll((who >> lane) & ((1ull << CHUNK) - 1));
  __syncthreads();
  const int chunks = (T + CHUNK - 1) / CHUNK - blockIdx.x * CHUNKS, n = (chunks < CHUNKS ? chunks : CHUNKS) * words;
  for (int i = threadIdx.x; i < n; i += 256) table[(size_t)blockIdx.x * CHUNKS * words + i] = counts[i / words][i % words];
}

// The experts of E that a token asks for as bits, worked out by one lane from its logits: what moe_topk_softmax_wave selects.
template <int E, typename LT>
struct LaneLogits {
  u32x2 w[E * sizeof(LT) / 8];
  __device__ __forceinline__ void request(const LT* __restrict__ logits) {
#pragma unroll
    for (int i = 0; i < (int)(E * sizeof(LT) / 8); ++i) w[i] = reinterpret_cast<const u32x2*>(logits)[i];
  }
  __device__ __forceinline__ uint32_t selected(const float* __restrict__ bias, int k) const {
    uint32_t key[E], bits = 0;
#pragma unroll
    for (int e = 0; e < E; ++e) {
      constexpr int PER = 4 / sizeof(LT);
      const uint32_t word = w[e / PER / 2][e / PER % 2];
      float v = sizeof(LT) == 4 ? __builtin_bit_cast(float, word) : e & 1 ? bf16hi(word) : bf16lo(word);
      if (bias) v += bias[e];
      key[e] = moe_orderable(v);
    }
    for (int j = 0; j < k; ++j) {
      uint32_t best = key[0], has = 0;
#pragma unroll
      for (int e = 1; e < E; ++e) best = key[e] > best ? key[e] : best;
#pragma unroll
      for (int e = 0; e < E; ++e) has |= key[e] == best ? 1u << e : 0;
      has &= -has;  // the first that has it
      bits |= has;
#pragma unroll
      for (int e = 0; e < E; ++e) key[e] = has & (1u << e) ? 0 : key[e];  // (which no logit maps to)
    }
    return bits;
  }
};

// Where a token's experts come from: a selection's table, the caller (they may lie outside [0, E)), or the logits.
enum Experts { TABLE, GIVEN_IDS, LOGITS };
template <typename LT>
struct Selection {  // LOGITS
  const LT* logits;
  const float* bias;
  int32_t* ids;
  float* gates;
};

// WAVES tokens of a chunk, one a wave.  `shift`: 2^shift words hold a chunk's counts.
// From the logits (of NE experts) every workgroup selects for all tokens, a lane a token, to count them, and leaves ids and gates of
// its own.
template <typename XT, typename OT, int WAVES, Experts FROM, int NE = 8, typename LT = float>
__global__ __launch_bounds__(WAVES* MOE_WAVE) void place_rows_kernel(
    const XT* __restrict__ x, const int32_t* __restrict__ ids, const uint32_t* __restrict__ table, int T, int E, int k,
    int H, int shift, int32_t* __restrict__ counts, int32_t* __restrict__ offs, int32_t* __restrict__ pos_to_row,
    int32_t* __restrict__ row_to_pos, int32_t* __restrict__ bad_ids, OT* __restrict__ xp, const uint32_t* __restrict__ bad,
    const Selection<LT> sel) {
  constexpr bool GIVEN = FROM == GIVEN_IDS;
  __shared__ int below[PLACE_EXPERTS], total[PLACE_EXPERTS];  // of earlier chunks, of all
  __shared__ uint32_t asked[PLACE_EXPERTS];
  constexpr int AHEAD = 4;  // 8-element pieces of the row requested at once
  const int lane = lane_id(), wv = uniform((int)(threadIdx.x / MOE_WAVE));
  const int chunk = blockIdx.x / (CHUNK / WAVES), chunks = (T + CHUNK - 1) / CHUNK, words = (E + 3) / 4;
  const int t = blockIdx.x * WAVES + wv;
  const bool live = t < T, with_rows = xp != nullptr;
  typename std::conditional<sizeof(XT) == 2, u32x4, Row8>::type row[AHEAD];
  const auto request = [&](int base) {
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) {
      const int col = base + (i * MOE_WAVE + lane) * 8;
      if (live && with_rows && col < H) {
        if constexpr (sizeof(XT) == 2) row[i] = *reinterpret_cast<const u32x4*>(x + (size_t)t * H + col);
        else row[i] = load8(x + (size_t)t * H + col);
      }
    }
  };
  request(0);
  const auto expert_of = [&](int r) {
    const int e = ids[r];
    return !GIVEN ? e : e < 0 ? 0 : e >= E ? E - 1 : e;
  };
  int my_id = 0;
  if constexpr (FROM == LOGITS) {
    if (live) {
      uint32_t key[1];
      float gate;
      moe_topk_keys<1>(sel.logits + (size_t)t * E, sel.bias, E, lane, key);
      moe_topk_softmax_wave<1>(key, k, lane, my_id, gate);
      if (lane < k) {
        sel.ids[(size_t)t * k + lane] = my_id;
        sel.gates[(size_t)t * k + lane] = gate;
      }
    }
  } else {
    my_id = live && lane < k ? expert_of(t * k + lane) : 0;
  }
  __shared__ int outside;
  if (GIVEN && threadIdx.x == 0) outside = 0;
  static_assert(WAVES * MOE_WAVE >= PLACE_EXPERTS && CHUNK % WAVES == 0, "a thread an expert");
  if (threadIdx.x < PLACE_EXPERTS) below[threadIdx.x] = total[threadIdx.x] = 0, asked[threadIdx.x] = 0;
  __syncthreads();
  if constexpr (FROM == LOGITS) {
    if (live && lane < k) atomicOr(&asked[my_id], 1u << wv);
    const int t0 = blockIdx.x * WAVES;
    int all = 0, low = 0;  // of expert `lane`
    for (int base = wv * MOE_WAVE; base < T; base += WAVES * MOE_WAVE) {
      uint32_t bits = 0;
      if (base + lane < T) {
        LaneLogits<NE, LT> row;
        row.request(sel.logits + (size_t)(base + lane) * NE);
        bits = row.selected(sel.bias, k);
      }
      const unsigned long long before = t0 <= base ? 0 : t0 - base >= MOE_WAVE ? ~0ull : (1ull << (t0 - base)) - 1;
#pragma unroll
      for (int e = 0; e < NE; ++e) {
        const unsigned long long who = __ballot(bits >> e & 1);
        all += lane == e ? __popcll(who) : 0;
        low += lane == e ? __popcll(who & before) : 0;
      }
    }
    if (lane < E) {
      atomicAdd(&total[lane], all);
      atomicAdd(&below[lane], low);
    }
  } else {
    for (int i = threadIdx.x; i < CHUNK * k; i += blockDim.x) {
      const int r = chunk * CHUNK * k + i;
      if (r < T * k) atomicOr(&asked[expert_of(r)], 1u << (i / k));
    }
    if (GIVEN && blockIdx.x == 0) {
      int n = 0;
      for (int c = threadIdx.x; c < chunks; c += blockDim.x) n += bad[c];
      if (n) atomicAdd(&outside, n);
    }
    // two 16-bit sums a register: no expert has more rows than there are tokens
    const int w = threadIdx.x & ((1 << shift) - 1), step = blockDim.x >> shift;
    uint32_t all02 = 0, all13 = 0, low02 = 0, low13 = 0;
    if (w < words) {
  #pragma unroll 4
      for (int c = threadIdx.x >> shift; c < chunks; c += step) {
        const uint32_t v = table[(size_t)c * words + w];
        const uint32_t v02 = v & 0x00ff00ffu, v13 = (v >> 8) & 0x00ff00ffu;
        all02 += v02;
        all13 += v13;
        low02 += c < chunk ? v02 : 0;
        low13 += c < chunk ? v13 : 0;
      }
    }
    for (int off = MOE_WAVE / 2; off >= 1 << shift; off >>= 1) {
      all02 += __shfl_xor(all02, off, MOE_WAVE);
      all13 += __shfl_xor(all13, off, MOE_WAVE);
      low02 += __shfl_xor(low02, off, MOE_WAVE);
      low13 += __shfl_xor(low13, off, MOE_WAVE);
    }
    if (w < words && lane < (1 << shift)) {
      atomicAdd(&total[4 * w + 0], (int)(all02 & 0xffff));
      atomicAdd(&total[4 * w + 1], (int)(all13 & 0xffff));
      atomicAdd(&total[4 * w + 2], (int)(all02 >> 16));
      atomicAdd(&total[4 * w + 3], (int)(all13 >> 16));
      atomicAdd(&below[4 * w + 0], (int)(low02 & 0xffff));
      atomicAdd(&below[4 * w + 1], (int)(low13 & 0xffff));
      atomicAdd(&below[4 * w + 2], (int)(low02 >> 16));
      atomicAdd(&below[4 * w + 3], (int)(low13 >> 16));
    }
  }
  __syncthreads();
  const int n0 = total[lane], n1 = total[MOE_WAVE + lane];
  const int upto0 = wave_inclusive(n0), half = read_lane(upto0, MOE_WAVE - 1), upto1 = half + wave_inclusive(n1);
  if (blockIdx.x == 0 && wv == 0) {
    if (lane < E) counts[lane] = n0, offs[lane] = upto0 - n0;
    if (MOE_WAVE + lane < E) counts[MOE_WAVE + lane] = n1, offs[MOE_WAVE + lane] = upto1 - n1;
    if (lane == 0) offs[E] = T * k;
    if (lane == 0 && bad_ids) *bad_ids = GIVEN ? outside : 0;  // (a selection asks for no other experts)
  }
  const int first0 = __shfl(upto0 - n0, my_id & 63, MOE_WAVE), first1 = __shfl(upto1 - n1, my_id & 63, MOE_WAVE);
  int pos = 0;
  if (live && lane < k) {
    const uint32_t earlier = asked[my_id] & ((1u << (FROM == LOGITS ? wv : t % CHUNK)) - 1);
    pos = (my_id < MOE_WAVE ? first0 : first1) + below[my_id] + __popc(earlier);
    const int r = t * k + lane;
    row_to_pos[r] = pos;
    pos_to_row[pos] = r;
  }
  if (!live || !with_rows) return;
  for (int base = 0; base < H; base += AHEAD * MOE_WAVE * 8) {
    if (base > 0) request(base);
    for (int j = 0; j < k; ++j) {
      OT* dst = xp + (size_t)read_lane(pos, j) * H;
#pragma unroll
      for (int i = 0; i < AHEAD; ++i) {
        const int col = base + (i * MOE_WAVE + lane) * 8;
        if (col < H) {
          if constexpr (sizeof(XT) == 2) store_bits_nt(dst + col, row[i]);
          else if constexpr (sizeof(OT) == 2) store8_nt(dst + col, row[i]);
          else store8(dst + col, row[i]);
        }
      }
    }
  }
}

}  // namespace

bool moe_place_ok(int64_t T, int64_t E, int64_t k) {
  return T > 0 && T < 65536 && E <= PLACE_EXPERTS && k <= E && k <= MOE_MAX_TOPK && moe_place_bytes(T, E) <= PLACE_TABLE;
}
int64_t moe_place_bytes(int64_t T, int64_t E) { return (T + CHUNK - 1) / CHUNK * words_of(E) * 4; }

int moe_select_count(const void* logits, int logits_dtype, const float* bias, int64_t T, int64_t E, int64_t k,
                     int32_t* ids, float* gates, void* table, void* stream) {
  hipStream_t s = (hipStream_t)stream;
  const auto go = [&](auto vpl, auto lt) {
    using LT = decltype(lt);
    hipLaunchKernelGGL((select_count_kernel<decltype(vpl)::value, LT>), dim3((unsigned)((T + CHUNK - 1) / CHUNK)),
                       dim3(CHUNK * MOE_WAVE), 0, s, (const LT*)logits, bias, (int)T, (int)E, (int)k, ids, gates,
                       (uint32_t*)table);
    return moe_launch_status();
  };
  using One = std::integral_constant<int, 1>;
  using Two = std::integral_constant<int, 2>;
  if (logits_dtype == MOE_DT_BF16) return E <= MOE_WAVE ? go(One{}, uint16_t{}) : go(Two{}, uint16_t{});
  return E <= MOE_WAVE ? go(One{}, float{}) : go(Two{}, float{});
}

// Row by row there is least else to do, and what the general path launches more is soon less than a table read by every workgroup: whole
// training passes of rows, us, there and here: 1123 rows of 24 experts, 272 <-> 176, 69 -> 65; 4392 of 64, 264 <-> 264, 89 -> 81; 9085 of
// 16, 512 <-> 448, 137 -> 129; 18747 of 32, 1280 <-> 192, 287 -> 290; 32768 of 16, 4096 <-> 1536, 3682 -> 3708.
bool moe_count_ok(int64_t T, int64_t E, int64_t k) { return k == 1 && T <= 16384 && moe_place_ok(T, E, k); }
int64_t moe_count_bytes(int64_t T, int64_t E) { return moe_place_bytes(T, E) + (T + CHUNK - 1) / CHUNK * 4; }

int moe_count_ids(const int64_t* ids64, int32_t* ids, int64_t T, int64_t E, void* table, void* stream) {
  uint32_t* bad = (uint32_t*)((char*)table + moe_place_bytes(T, E));
  const dim3 grid((unsigned)((T + 255) / 256)), block(256);
  if (ids64)
    hipLaunchKernelGGL(count_ids_kernel<int64_t>, grid, block, 0, (hipStream_t)stream, ids64, (int)T, (int)E, ids,
                       (uint32_t*)table, bad);
  else
    hipLaunchKernelGGL(count_ids_kernel<int32_t>, grid, block, 0, (hipStream_t)stream, ids, (int)T, (int)E, nullptr,
                       (uint32_t*)table, bad);
  return moe_launch_status();
}

int moe_place_rows(const void* x, int x_dtype, const int32_t* ids, const void* table, int64_t T, int64_t H, int64_t E,
                   int64_t k, int32_t* counts, int32_t* offs, int32_t* pos_to_row, int32_t* row_to_pos, int32_t* bad_ids,
                   void* xp, int xp_dtype, bool counted, void* stream) {
  if (H <= 0 || H % 8 != 0) return MOE_ERR_SHAPE;
  if (H > 65536) return MOE_ERR_LIMIT;
  if (x_dtype == MOE_DT_BF16 && xp_dtype != MOE_DT_BF16) return MOE_ERR_DTYPE;
  hipStream_t s = (hipStream_t)stream;
  const uint32_t* bad = counted ? (const uint32_t*)((const char*)table + moe_place_bytes(T, E)) : nullptr;
  int shift = 0;
  while ((1 << shift) < words_of(E)) ++shift;
  const auto go = [&](auto xt, auto ot, auto waves) {
    using XT = decltype(xt);
    using OT = decltype(ot);
    constexpr int WAVES = decltype(waves)::value;
    const auto launch = [&](auto kern) {
      hipLaunchKernelGGL(kern, dim3((unsigned)((T + WAVES - 1) / WAVES)), dim3(WAVES * MOE_WAVE), 0, s, (const XT*)x, ids,
                         (const uint32_t*)table, (int)T, (int)E, (int)k, (int)H, shift, counts, offs, pos_to_row, row_to_pos,
                         bad_ids, (OT*)xp, bad, Selection<float>{});
    };
    if (counted) launch(place_rows_kernel<XT, OT, WAVES, GIVEN_IDS>);
    else launch(place_rows_kernel<XT, OT, WAVES, TABLE>);
    return moe_launch_status();
  };
  const auto of = [&](auto waves) {
    if (x_dtype == MOE_DT_BF16) return go(uint16_t{}, uint16_t{}, waves);
    return xp_dtype == MOE_DT_BF16 ? go(float{}, uint16_t{}, waves) : go(float{}, float{}, waves);
  };
  // (fewer workgroups to read a large table: 4096 tokens, 128 experts 18.1 us, with 8 waves 20.0; 8192 tokens, 8 experts,
  // 4 KB 11.1 and 10.7)
  return moe_place_bytes(T, E) > 16 * 1024 ? of(std::integral_constant<int, 16>{}) : of(std::integral_constant<int, 8>{});
}

// A launch fewer, as long as the selection of all tokens costs a workgroup less than that: 128 / 512 / 1024 tokens, bf16, 1024 wide, us, two
// launches' own times and here: 2 of 8 experts 7.3, 4.7 / 7.5, 5.2 / 8.6, 7.2 (2048: 9.6, 11.4); 1 of 4 7.1, 4.0 / 7.3, 4.2 / 7.4, 5.1; 512
// tokens, 4 of 8 9.0, 6.8, 4 of 4 9.0, 6.1; 256, 8 of 8 9.9, 8.0.  (2 of 16 7.0, 6.4 / 7.7, 7.0 / 8.6, 10.3, 8 of 16 from the first on slower: not
// taken.  A lane holds a token's logits in registers, their number is the kernel's own: 4 and 8 are what the kernel is made for; counts
// that are not multiples of 4 have bf16 rows that do not come in whole words of 8 bytes, and 12 lies next to 16.)
bool moe_select_place_ok(const void* logits, int64_t T, int64_t E, int64_t k) {
  return moe_place_ok(T, E, k) && (E == 4 || E == 8) && T <= 1024 && T * k <= 2048 && (reinterpret_cast<uintptr_t>(logits) & 7) == 0;
}

int moe_select_place(const void* x, int x_dtype, const void* logits, int logits_dtype, const float* bias, int64_t T, int64_t H,
                     int64_t E, int64_t k, int32_t* ids, float* gates, int32_t* counts, int32_t* offs, int32_t* pos_to_row,
                     int32_t* row_to_pos, int32_t* bad_ids, void* xp, int xp_dtype, void* stream) {
  if (H <= 0 || H % 8 != 0) return MOE_ERR_SHAPE;
  if (H > 65536) return MOE_ERR_LIMIT;
  if (x_dtype == MOE_DT_BF16 && xp_dtype != MOE_DT_BF16) return MOE_ERR_DTYPE;
  constexpr int WAVES = 8;
  const auto go = [&](auto xt, auto ot, auto lt, auto ne) {
    using XT = decltype(xt);
    using OT = decltype(ot);
    using LT = decltype(lt);
    hipLaunchKernelGGL((place_rows_kernel<XT, OT, WAVES, LOGITS, decltype(ne)::value, LT>), dim3((unsigned)((T + WAVES - 1) / WAVES)),
                       dim3(WAVES * MOE_WAVE), 0, (hipStream_t)stream, (const XT*)x, nullptr, nullptr, (int)T, (int)E, (int)k, (int)H,
                       0, counts, offs, pos_to_row, row_to_pos, bad_ids, (OT*)xp, nullptr,
                       Selection<LT>{(const LT*)logits, bias, ids, gates});
    return moe_launch_status();
  };
  const auto of = [&](auto lt, auto ne) {
    if (x_dtype == MOE_DT_BF16) return go(uint16_t{}, uint16_t{}, lt, ne);
    return xp_dtype == MOE_DT_BF16 ? go(float{}, uint16_t{}, lt, ne) : go(float{}, float{}, lt, ne);
  };
  using Four = std::integral_constant<int, 4>;
  using Eight = std::integral_constant<int, 8>;
  if (logits_dtype == MOE_DT_BF16) return E == 4 ? of(uint16_t{}, Four{}) : of(uint16_t{}, Eight{});
  return E == 4 ? of(float{}, Four{}) : of(float{}, Eight{});
}
