// The router product and the selection in one launch: x [T,H] and the router weight [E,H] -> logits, expert ids, gates and the
// counts that the rows are placed by (place.hip).
//
// In launches of its own the product is a matrix product too small to fill the chip (4 to 20 us where x alone takes 1 to 4), then
// the logits go out and come back for the selection; and where the layer is narrow the library's call is half of the host's work.  Here a
// workgroup takes the 16 tokens that are counted together: their rows come in once, whole lines, into LDS (as bf16; where x is
// fp32 the rounded copy leaves from there for the later kernels), the waves multiply them with the experts' rows from L2 on the
// 16x16x32 matrix instruction, and select on the logits while those are still in LDS.
//
// What bounds it: one trip to memory for x, behind which the first router rows are on their way, E * H * 2 bytes of router rows a
// workgroup from L2, and the chain of the selection.
//
// A logit's sum is taken in the order in which the library's product takes it, so that logits, and with them the experts a
// token goes to, are the same bits whether the product is made here or by nn.Linear (a router with hooks, `router_linear`): for most sizes
// one chain of products along the contraction, for launches of few tiles four of them that take turns, a matrix instruction each, added up in
// the end.  router_chains() says which; sizes for which neither is known to hold stay with the library.
#include "common.h"
#include "internal.h"
#include "tile_ops.h"
#include "topk_core.h"

namespace {

constexpr int TOKENS = MOE_PLACE_CHUNK, BLOCK = 32;  // tokens of a workgroup, contraction of a matrix instruction
constexpr int MAX_E = 2 * MOE_WAVE, MAX_H = 2048;
static_assert(TOKENS == 16, "a matrix instruction's rows");

struct RouterArgs {
  const void *x, *wr;
  const float* bias;
  int T, H, E, k;
  uint16_t *xn, *wrb;  // bf16 copies of x and wr (NULL: not wanted)
  uint16_t* logits;
  int32_t* ids;
  float* gates;
  uint32_t* table;  // counts, a byte an expert and 16 tokens (NULL: not wanted)
};

__device__ __forceinline__ u32x4 bf16_bits(u32x4 v) { return v; }
__device__ __forceinline__ u32x4 bf16_bits(const Row8& r) {
  return u32x4{pack_bf16x2(r.v[0], r.v[1]), pack_bf16x2(r.v[2], r.v[3]), pack_bf16x2(r.v[4], r.v[5]), pack_bf16x2(r.v[6], r.v[7])};
}
template <typename T>
using Chunk = typename std::conditional<sizeof(T) == 2, u32x4, Row8>::type;  // eight elements as they lie in memory
template <typename T>
__device__ __forceinline__ Chunk<T> chunk_at(const T* p) {
  if constexpr (sizeof(T) == 2) return *reinterpret_cast<const u32x4*>(p);
  else return load8(p);
}

// Eight elements of the router's weight on their way, and in bf16.
template <typename T>
struct Bits {
  u32x4 v[sizeof(T) / 2];
  __device__ __forceinline__ u32x4 bf16() const {
    if constexpr (sizeof(T) == 2) {
      return v[0];
    } else {
      const f32x4 a = __builtin_bit_cast(f32x4, v[0]), b = __builtin_bit_cast(f32x4, v[1]);
      return u32x4{pack_bf16x2(a[0], a[1]), pack_bf16x2(a[2], a[3]), pack_bf16x2(b[0], b[1]), pack_bf16x2(b[2], b[3])};
    }
  }
};

constexpr int SLICE = 128;                   // of the contraction: a slice of the router's rows is in LDS at a time
constexpr int PER_ROW = SLICE / 8;           // pieces of eight elements of a slice's row

__host__ __device__ constexpr int row_stride(int H) { return (H + SLICE - 1) / SLICE * SLICE; }  // of x in LDS, in elements
// Where a row's piece lies: permuted inside its slice, so that a fragment's 16 rows lie in different banks, and so do two rows'
// pieces that are written together (rows padded by 16 bytes instead: both conflict, 1531 tokens of 64 experts, 2048 wide, 11.0 us, so 10.1).
__device__ __forceinline__ int placed(int row, int piece) { return (piece ^ (row & (PER_ROW - 1))) * 8; }
// Floats from one token's partial sums to the next.
__host__ __device__ constexpr int sum_stride(int E) { return (E + 15) / 16 * 16 + 4; }

// k rounds as moe_topk_softmax_wave makes them, for four tokens of up to 16 experts at once, 16 lanes each: lane l has the key of expert
// l % 16 of token l / 16.  The token's lane j < k gets slot j.
__device__ __forceinline__ void topk_softmax_rows(uint32_t key, int k, int lane, int& my_id, float& my_gate) {
#define MOE_ROW_ROR(v, n) (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(v), 0x120 + (n), 0xf, 0xf, false)
  const int l16 = lane & 15, row0 = lane & ~15;
  my_id = 0;
  float my_val = 0.f, vmax = 0.f;
  for (int j = 0; j < k; ++j) {
    uint32_t best = key, o;
    o = MOE_ROW_ROR(best, 8), best = o > best ? o : best;
    o = MOE_ROW_ROR(best, 4), best = o > best ? o : best;
    o = MOE_ROW_ROR(best, 2), best = o > best ? o : best;
    o = MOE_ROW_ROR(best, 1), best = o > best ? o : best;
    const uint32_t has = (uint32_t)(__ballot(key == best) >> row0) & 0xffffu;
    const int e = __builtin_ctz(has);  // (the first; every token's lanes have one)
    if (l16 == e) key = 0;
    const float val = moe_from_orderable(best);
    if (j == 0) vmax = val;
    if (l16 == j) my_id = e, my_val = val;
  }
  const float p = l16 < k ? expf(my_val - vmax) : 0.f;
  my_gate = p / moe_row_sum_f32(p);
#undef MOE_ROW_ROR
}

// Up to MAXE experts.  The waves are CHAINS by what is left of them; wave (c, g) multiplies blocks c, c + CHAINS, .. of the contraction
// for the groups of 16 experts g, g + GROUPS, ...
template <typename XT, typename WT, int CHAINS, int MAXE, int NT>
__global__ __launch_bounds__(NT) void router_select_kernel(const RouterArgs p) {
  constexpr int WAVES = NT / MOE_WAVE, GROUPS = WAVES / CHAINS, ROWS = TOKENS / WAVES;
  constexpr int GPW = (MAXE / 16 + GROUPS - 1) / GROUPS, VPL = (MAXE + MOE_WAVE - 1) / MOE_WAVE;
  constexpr int CH = MAXE * PER_ROW / NT;           // pieces of a slice to a thread
  constexpr int AHEAD = 32 / (CH * (int)sizeof(WT));  // slices on their way in registers
  static_assert(WAVES % CHAINS == 0 && TOKENS % WAVES == 0 && MAXE * PER_ROW % NT == 0 && AHEAD > 0, "waves");
  extern __shared__ __attribute__((aligned(16))) uint16_t rows[];  // x, then two slices of the router's rows
  __shared__ uint16_t own[TOKENS][MAXE];  // logits
  __shared__ uint32_t asked[MAXE];        // bit t: token t asks for the expert
  const int lane = lane_id(), wv = uniform((int)(threadIdx.x / MOE_WAVE)), c = wv % CHAINS, g = wv / CHAINS;
  const int l16 = lane & 15, q = lane >> 4;
  const int t0 = blockIdx.x * TOKENS, slices = (p.H + SLICE - 1) / SLICE, stride = row_stride(p.H), pieces = p.H / 8;
  const int groups = (p.E + 15) / 16;
  const XT* x = (const XT*)p.x;
  uint16_t* sw = rows + TOKENS * stride;
  const int slice_elems = groups * 16 * SLICE;

  // ---- x, a wave ROWS tokens; then the first slices of the router's rows
  Chunk<XT> in[ROWS][MAX_H / 8 / MOE_WAVE];
#pragma unroll
  for (int r = 0; r < ROWS; ++r) {
    const int t = t0 + wv * ROWS + r;
#pragma unroll
    for (int i = 0; i < MAX_H / 8 / MOE_WAVE; ++i) {
      const int at = i * MOE_WAVE + lane;
      if (at < pieces) in[r][i] = chunk_at(x + (size_t)(t < p.T ? t : p.T - 1) * p.H + at * 8);
    }
  }
  // (rows past the last expert's get an offset outside the window, which reads as zero there, as does what lies past the last row's end;
  // columns past the end of other rows are the next row's, and cleared on the way to LDS)
  const __amdgpu_buffer_rsrc_t wr_window = __builtin_amdgcn_make_buffer_rsrc((void*)p.wr, 0, p.E * p.H * (int)sizeof(WT), 0x00020000);
  int from[CH], put[CH];  // a thread's pieces: bytes from the slice's first column, elements of a slice in LDS
#pragma unroll
  for (int n = 0; n < CH; ++n) {
    const int i = n * NT + (int)threadIdx.x, e = i / PER_ROW, at = i % PER_ROW;
    from[n] = e < p.E ? (e * p.H + at * 8) * (int)sizeof(WT) : -(1 << 24);
    put[n] = e < groups * 16 ? e * SLICE + placed(e, at) : -1;
  }
  const int my_col = (int)threadIdx.x % PER_ROW * 8;  // (the same for all of them)
  Bits<WT> w[AHEAD][CH];
  const auto request = [&](int to, int slice) __attribute__((always_inline)) {
#pragma unroll
    for (int n = 0; n < CH; ++n)
#pragma unroll
      for (int h = 0; h < (int)(sizeof(Bits<WT>) / 16); ++h)
        w[to][n].v[h] = __builtin_amdgcn_raw_buffer_load_b128(wr_window, from[n] + slice * SLICE * (int)sizeof(WT) + h * 16, 0, 0);
  };
#pragma unroll
  for (int a = 0; a < AHEAD; ++a)
    if (a < slices) request(a, a);
  for (int i = threadIdx.x; i < MAXE; i += NT) asked[i] = 0;
#pragma unroll
  for (int r = 0; r < ROWS; ++r) {
    const int row = wv * ROWS + r, t = t0 + row;
#pragma unroll
    for (int i = 0; i < MAX_H / 8 / MOE_WAVE; ++i) {
      const int at = i * MOE_WAVE + lane;
      if (at * 8 < slices * SLICE) {
        u32x4 v = u32x4{0, 0, 0, 0};  // (zeros fill the last slice)
        if (at < pieces) {
          v = bf16_bits(in[r][i]);
          if (sizeof(XT) == 4 && p.xn && t < p.T) *reinterpret_cast<u32x4*>(p.xn + (size_t)t * p.H + at * 8) = v;
        }
        *reinterpret_cast<u32x4*>(rows + row * stride + placed(row, at)) = v;
      }
    }
  }

  // ---- the products: experts by tokens, lane l holds token l % 16, experts 4 * (l / 16) .. + 3 of a group.  One barrier a slice: a
  // wave writes the next one where all have done with the one before this.
  constexpr int MINE = SLICE / BLOCK / CHAINS;  // a wave's blocks of a slice
  static_assert(MINE * CHAINS * BLOCK == SLICE, "whole blocks");
  f32x4 acc[GPW];
  int read_at[MINE];  // a lane's place in a fragment, elements
#pragma unroll
  for (int b = 0; b < MINE; ++b) read_at[b] = placed(l16, (b * CHAINS + c) * 4 + q);
  const uint16_t *tokens_at = rows + l16 * stride, *experts_at = sw + (g * 16 + l16) * SLICE;
#pragma unroll
  for (int n = 0; n < GPW; ++n) acc[n] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int s0 = 0; s0 < slices; s0 += AHEAD) {
#pragma unroll
    for (int a = 0; a < AHEAD; ++a) {
      const int s = s0 + a;
      if (s < slices) {
        const int odd = (s & 1) * slice_elems;
        const bool past_end = s * SLICE + SLICE > p.H && s * SLICE + my_col >= p.H;
#pragma unroll
        for (int n = 0; n < CH; ++n) {
          u32x4 bits = w[a][n].bf16();
          if (past_end) bits = u32x4{0, 0, 0, 0};
          if (put[n] >= 0) *reinterpret_cast<u32x4*>(sw + odd + put[n]) = bits;
          if (sizeof(WT) == 4 && p.wrb && blockIdx.x == 0 && from[n] >= 0 && !past_end)
            *reinterpret_cast<u32x4*>(p.wrb + from[n] / 4 + s * SLICE) = bits;
        }
        if (s + AHEAD < slices) request(a, s + AHEAD);
        lds_barrier();
#pragma unroll
        for (int b = 0; b < MINE; ++b) {
          const bf16x8 tokens = *reinterpret_cast<const bf16x8*>(tokens_at + s * SLICE + read_at[b]);
#pragma unroll
          for (int n = 0; n < GPW; ++n)
            if (g + n * GROUPS < groups) {
              const bf16x8 experts = *reinterpret_cast<const bf16x8*>(experts_at + odd + n * GROUPS * 16 * SLICE + read_at[b]);
              acc[n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(experts, tokens, acc[n], 0, 0, 0);
            }
        }
      }
    }
  }
  const auto emit = [&](int token, int e, const f32x4& s) {  // (four experts)
    *reinterpret_cast<u32x2*>(&own[token][e]) = u32x2{pack_bf16x2(s[0], s[1]), pack_bf16x2(s[2], s[3])};
  };
  if constexpr (CHAINS == 1) {
#pragma unroll
    for (int n = 0; n < GPW; ++n)
      if (g + n * GROUPS < groups) emit(l16, (g + n * GROUPS) * 16 + q * 4, acc[n]);
  } else {
    float* sums = reinterpret_cast<float*>(rows);
    const int ss = sum_stride(p.E);
    __syncthreads();  // (the rows have been read)
#pragma unroll
    for (int n = 0; n < GPW; ++n)
      if (g + n * GROUPS < groups)
        *reinterpret_cast<f32x4*>(sums + (c * TOKENS + l16) * ss + (g + n * GROUPS) * 16 + q * 4) = acc[n];
    __syncthreads();
    for (int i = threadIdx.x; i < TOKENS * groups * 4; i += NT) {
      const int token = i & (TOKENS - 1), e = i / TOKENS * 4;
      f32x4 s = *reinterpret_cast<const f32x4*>(sums + token * ss + e);
#pragma unroll
      for (int n = 1; n < CHAINS; ++n) s += *reinterpret_cast<const f32x4*>(sums + (n * TOKENS + token) * ss + e);
      emit(token, e, s);
    }
  }
  __syncthreads();

  // ---- the selection, a wave ROWS tokens
  if constexpr (MAXE == 16) {
    static_assert(ROWS == 4, "16 lanes a token");
    const int token = wv * 4 + q, t = t0 + token;
    const uint16_t bits = own[token][l16];
    uint32_t key = 0;
    if (l16 < p.E) key = moe_orderable(bf16_to_f32(bits) + (p.bias ? p.bias[l16] : 0.f));
    int id;
    float gate;
    topk_softmax_rows(key, p.k, lane, id, gate);
    if (t < p.T) {
      if (l16 < p.E) p.logits[(size_t)t * p.E + l16] = bits;
      if (l16 < p.k) {
        p.ids[(size_t)t * p.k + l16] = id;
        p.gates[(size_t)t * p.k + l16] = gate;
        atomicOr(&asked[id], 1u << token);
      }
    }
  } else {
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
      const int token = wv * ROWS + r, t = t0 + token;
      if (t < p.T) {
#pragma unroll
        for (int i = 0; i < VPL; ++i)
          if (i * MOE_WAVE + lane < p.E) p.logits[(size_t)t * p.E + i * MOE_WAVE + lane] = own[token][i * MOE_WAVE + lane];
        uint32_t key[VPL];
        moe_topk_keys<VPL>(own[token], p.bias, p.E, lane, key);
        int id;
        float gate;
        moe_topk_softmax_wave<VPL>(key, p.k, lane, id, gate);
        if (lane < p.k) {
          p.ids[(size_t)t * p.k + lane] = id;
          p.gates[(size_t)t * p.k + lane] = gate;
          atomicOr(&asked[id], 1u << token);
        }
      }
    }
  }
  if (!p.table) return;
  __syncthreads();
  const int words = (p.E + 3) / 4;
  if ((int)threadIdx.x < words) {
    uint32_t n = 0;
#pragma unroll
    for (int b = 0; b < 4; ++b) n |= (uint32_t)__popc(asked[threadIdx.x * 4 + b]) << (8 * b);
    p.table[(size_t)blockIdx.x * words + threadIdx.x] = n;
  }
}

template <typename XT, typename WT, int CHAINS, int MAXE, int NT>
int launch(const RouterArgs& a, hipStream_t s) {
  const int sums = CHAINS > 1 ? CHAINS * TOKENS * sum_stride(MAXE) * 4 : 0;
  const auto bytes = [&](int H, int E) {
    const int n = (TOKENS * row_stride(H) + 2 * ((E + 15) / 16 * 16) * SLICE) * 2;
    return n > sums ? n : sums;
  };
  const auto kern = router_select_kernel<XT, WT, CHAINS, MAXE, NT>;
  static bool done[MOE_MAX_DEVICES];
  const int dev = moe_current_device();
  if (!done[dev]) {
    const hipError_t err = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, bytes(MAX_H, MAXE));
    if (err != hipSuccess) return (int)err;
    done[dev] = true;
  }
  hipLaunchKernelGGL(kern, dim3((unsigned)((a.T + TOKENS - 1) / TOKENS)), dim3(NT), bytes(a.H, a.E), s, a);
  return moe_launch_status();
}

// Chains that the library's product sums a logit in (0: not known): what the matrix library that PyTorch 2.10 for ROCm 7 calls does on 256 compute
// units, found by comparing results.  Sizes on both sides of every line here, and drawn ones, are compared to the bit in tests/test_gpu_router_select.py; another
// build of that library may sum in another order, and then a logit made here and nn.Linear's may differ in their last bit.  (Wider ones than MAX_H have more kinds
// of sums.)
int router_chains(int64_t T, int64_t H, int64_t E) {
  if (T <= 64 || H < 64 || H > MAX_H || H % 8 != 0 || E < 2 || E > MAX_E) return 0;
  if (E <= 16) {
    if (H >= 1024) return T <= 12288 ? 4 : 0;
    if (T <= 256) return 1;
    if (T <= 2048) return (E <= 12 && H >= 128) || H >= 320 ? 4 : 0;
    return T <= 3200 && H >= 512 ? 4 : 0;
  }
  if (E < 32 || T > 30000) return 0;
  if (H <= 1024) return 1;
  const int64_t groups = (E + 15) / 16, tiles = (T + 15) / 16 * groups;
  if (tiles == 511) return 0;  // (one short of two full rounds: not four chains)
  if (tiles <= 512) return 4;
  if (tiles > 1024) return 1;
  return groups % 2 ? 0 : E == 64 ? 4 : 1;
}

}  // namespace

// One launch where it is the faster one: 16 tokens a workgroup read all of the router's rows, which a compute unit takes 64 bytes a cycle
// of, so it is for few experts or for one workgroup to a compute unit.  Its time against that of the library's product and the
// selection's launch (fp32: and of the rounding's), us, on the GPU alone, x not in the caches: bf16, 2 of 8 experts, 1024 wide, 256 / 2048 / 8192 /
// 12288 tokens 5.0, 5.3, 7.5, 8.6 and 7.2, 7.4, 10.2, 12.1; 2048 wide, 8192 / 12288 tokens 11.3, 16.4 and 12.7, 15.4; 8 of 64, 1024 wide, 1024 / 4096 /
// 8192 tokens 8.2, 9.2, 17.5 and 10.2, 12.7, 14.5; 2048 wide, 1024 / 2048 / 4096 tokens 10.4, 11.6, 13.9 and 9.2, 12.8, 13.6; 8 of 128, 1024 wide, 256 /
// 2048 / 4096 tokens 9.9, 10.4, 11.7 and 9.5, 12.7, 13.8; 2048 wide, not taken, 2048 tokens 15.5 and 13.2; fp32, 8 of 128, 1024 wide, 4096 tokens
// 17.4 and 21.7.  Where the kernel is the longer one of the two by a microsecond the launch that goes is worth more: whole forward passes of the
// layer, 256 inside, bf16, without -> with it: 64 experts, 2048 wide, 1024 / 4096 tokens 87.6 -> 85.4, 183.5 -> 181.5; 128, 1024 wide, 256 / 4096 tokens
// 67.4 -> 65.6, 121.8 -> 118; 96, 1360 wide, 128 / 1024 / 4096 tokens 74.7 -> 75.4, 95.1 -> 94.2, 164.7 -> 156; of 70 sizes, 32 to 128 experts, none slower.  The host
// has 15 us less to do, which small steps take: training, 512 tokens, 2 of 8 experts, 256 <-> 128, 128 -> 104 us.
// Router rows in fp32 are twice the bytes a workgroup; with more than 64 experts and 1024 columns (two pieces a thread and slice, more than eight slices)
// that is the longer way while few tokens leave most compute units without a workgroup: with it -> without, 96, 1360 wide, forward, 70 / 512 / 1024 / 1531
// tokens 79.3 -> 75.0, 87.6 -> 83.0, 101.4 -> 97.9, 111.0 -> 111.0, training, 70 / 256 / 1024 227.9 -> 223.2, 236.5 -> 233.3, 315 -> 312; 80, 1536 wide, 70 / 1024
// 71.1 -> 67.0, 88.5 -> 83.3.  (Not so, or by no more than a GPU differs from the next: 64, 2048 wide, forward, 70 / 1024 tokens 69.5 -> 66 to 70, 93 -> 90 to 94,
// training, 70 / 512 213.5 -> 211.8, 256.1 -> 255.0; 128, 1024 wide, forward 66.6 -> 66 to 70, 78.6 -> 76 to 81, training 200 -> 202, 223 -> 230.)
bool moe_router_select_ok(int64_t T, int64_t H, int64_t E, int64_t k, int wr_dtype) {
  const bool long_rows = wr_dtype == MOE_DT_F32 && E > 64 && H > 1024 && T <= 1024;
  if (router_chains(T, H, E) == 0) return false;
  const bool pays = E <= 16 ? T <= (H <= 1024 ? 12288 : 8192) : T <= TOKENS * moe_compute_units() && E * H <= 128 * 1024 && !long_rows;
  return pays && k > 0 && k <= E && k <= MOE_MAX_TOPK;
}

int moe_router_select(const MoeRouter& r, int64_t T, int64_t H, int64_t E, int64_t k, int32_t* ids, float* gates, void* table,
                      hipStream_t s) {
  if (!moe_router_select_ok(T, H, E, k, r.wr_dtype)) return MOE_ERR_LIMIT;
  for (int d : {r.x_dtype, r.wr_dtype})
    if (d != MOE_DT_BF16 && d != MOE_DT_F32) return MOE_ERR_DTYPE;
  MOE_CHECK_PTR(r.x);
  MOE_CHECK_PTR(r.wr);
  MOE_CHECK_PTR(r.logits);
  if (!aligned16(r.xn) || !aligned16(r.wrb)) return MOE_ERR_ALIGN;
  if (!ids || !gates) return MOE_ERR_NULL;
  RouterArgs a{r.x, r.wr, r.bias, (int)T, (int)H, (int)E, (int)k, r.xn, r.wrb, r.logits, ids, gates, (uint32_t*)table};
  const int chains = router_chains(T, H, E);
  const auto of = [&](auto xt, auto wt) {
    using XT = decltype(xt);
    using WT = decltype(wt);
    if (E <= 16) return chains == 4 ? launch<XT, WT, 4, 16, 256>(a, s) : launch<XT, WT, 1, 16, 256>(a, s);
    if (chains == 4) return E <= 64 ? launch<XT, WT, 4, 64, 1024>(a, s) : launch<XT, WT, 4, 128, 1024>(a, s);
    return E <= 64 ? launch<XT, WT, 1, 64, 1024>(a, s) : launch<XT, WT, 1, 128, 1024>(a, s);
  };
  if (r.x_dtype == MOE_DT_BF16) return r.wr_dtype == MOE_DT_BF16 ? of(uint16_t{}, uint16_t{}) : of(uint16_t{}, float{});
  return r.wr_dtype == MOE_DT_BF16 ? of(float{}, uint16_t{}) : of(float{}, float{});
}
