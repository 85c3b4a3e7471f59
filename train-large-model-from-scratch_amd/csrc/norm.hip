// RMSNorm in front of the MoE layer, fused with the bf16 cast the layer needs anyway.
//
// The reference normalises in fp32 (its `LayerNorm`, model/modules/norm.py:14-19:
// x * rsqrt(mean(x^2) + eps), cast back to the input dtype, times the weight) and hands the
// fp32 result to the MoE module, where autocast rounds it to bf16 for every product
// (model/modules/mlp.py:100, :154-155).  Here one pass reads the residual stream once and
// writes the bf16 rows the router product and the dispatch kernel consume, plus one fp32
// reciprocal RMS per row for the backward pass.  The backward kernel sums the two gradient
// contributions of the normalised rows (expert path, router path), applies the RMSNorm
// Jacobian, adds the gradient of the residual branch and reduces the weight gradient in a
// fixed order (per-block partial sums over a fixed row assignment, then a column sum), so it
// is reproducible run to run.  Both kernels are HBM-bound: each row is read once and written
// once.
#include "common.h"
#include "internal.h"
#include "topk_core.h"
#include "row_sum.h"

namespace {

constexpr int NT = 256;
constexpr int NW = NT / MOE_WAVE;
constexpr int BWD_BLOCKS = 1024;  // upper bound on partial weight-gradient rows

__device__ __forceinline__ float block_sum(float v, float* red) {
#pragma unroll
  for (int o = MOE_WAVE / 2; o > 0; o >>= 1) v += __shfl_xor(v, o);
  __syncthreads();  // the previous use of `red` is over
  if (lane_id() == 0) red[threadIdx.x / MOE_WAVE] = v;
  __syncthreads();
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < NW; ++i) s += red[i];
  return s;
}

template <typename T>
struct is_bf16 {
  static constexpr bool value = std::is_same<T, uint16_t>::value;
};

// NV = 16-byte column groups per thread held in registers; H8 <= NT * NV.
template <typename XT, int NV>
__global__ __launch_bounds__(NT) void rmsnorm_fwd_kernel(const XT* __restrict__ x,
                                                        const float* __restrict__ w, float eps,
                                                        int T, int H8, uint16_t* __restrict__ xn,
                                                        float* __restrict__ rstd) {
  __shared__ float red[NW];
  const int H = H8 * 8;
  Row8 wv[NV];
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int c = threadIdx.x + i * NT;
    if (c < H8) wv[i] = load8(w + c * 8);
  }
  for (int t = blockIdx.x; t < T; t += gridDim.x) {
    Row8 xv[NV];
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int c = threadIdx.x + i * NT;
      if (c < H8) {
        xv[i] = load8(x + (size_t)t * H + c * 8);
#pragma unroll
        for (int j = 0; j < 8; ++j) ss += xv[i].v[j] * xv[i].v[j];
      }
    }
    ss = block_sum(ss, red);
    const float r = rsqrtf(ss / (float)H + eps);
    if (threadIdx.x == 0) rstd[t] = r;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int c = threadIdx.x + i * NT;
      if (c < H8) {
        Row8 o;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          float v = xv[i].v[j] * r;
          if (is_bf16<XT>::value) v = bf16_to_f32(f32_to_bf16(v));  // `.to(input_dtype)`, norm.py:19
          o.v[j] = wv[i].v[j] * v;
        }
        store8(xn + (size_t)t * H + c * 8, o);
      }
    }
  }
}

// The normalisation with the router behind it (model/gpt.py:32 into model/modules/mlp.py:100-103
// in one pass): a block normalises RB rows, keeps their bf16 form in LDS besides writing it out,
// multiplies them with the router weight on the matrix cores (v_mfma_f32_16x16x32_bf16: rows =
// tokens from LDS, columns = experts straight from L2, the contraction split in four and the
// partial products added through LDS), rounds the logits to bf16 (what the layer returns and
// selects on) and runs the wave-level top-k + softmax on them.  The normalised rows are not read
// again for the router, and the logits never leave the chip before selection.  Where place.hip takes the
// tokens, the block also leaves its experts' counts in that table, which takes three launches away from behind it.
constexpr int RB = 16;       // rows (tokens) per block
constexpr int RMAX_EB = 8;   // 16-expert column blocks: E <= 128
constexpr int ROUTER_WAVES = 16;
// Waves a SIMD that two blocks on a compute unit make (rows past 2048 wide leave LDS for one)
template <int NV, int WAVES>
constexpr int ROUTER_EU = (NV <= 4 ? 2 : 1) * WAVES / 4;

// What bounds it: all blocks of a launch of 8192 tokens are resident at once and go through load, product and selection
// together, each of them a chain of trips to memory or L2.  Sixteen waves, a row and a token's selection each, make the chains
// as short as they get; two such blocks fill a compute unit's wave slots (54 registers).  8192 rows of 2048 in fp32, 64 experts,
// 8 a token: 50.9 us with four waves of four rows, 39.9 here (100 MB: 19); with the launches up to the rows in expert
// order 123 -> 100.  A whole training pass of 24 drawn layers with it 1.00 to 1.10 times as fast where the GPU bounds it.
template <typename XT, int NV, int WAVES>
__global__ __launch_bounds__(WAVES* MOE_WAVE, (ROUTER_EU<NV, WAVES>)) void rmsnorm_router_fwd_kernel(
    const XT* __restrict__ x, const float* __restrict__ w, float eps, int T, int H8,
    const uint16_t* __restrict__ wr, int E, int k, uint16_t* __restrict__ xn, float* __restrict__ rstd,
    uint16_t* __restrict__ logits, int32_t* __restrict__ ids, float* __restrict__ gates, uint32_t* __restrict__ table) {
  static_assert(RB == MOE_PLACE_CHUNK && WAVES % NW == 0 && RB % WAVES == 0, "a block counts a chunk's tokens");
  extern __shared__ __attribute__((aligned(16))) uint16_t rows[];  // [RB][H + 8]; later fp32 partials
  __shared__ uint16_t lg16[RB * RMAX_EB * 16];
  __shared__ uint32_t asked[RMAX_EB * 16];  // bit t: token t of the block asks for the expert
  const int H = H8 * 8, LDT = H + 8;
  const int lane = lane_id(), wv = uniform((int)(threadIdx.x / MOE_WAVE));
  const int t0 = blockIdx.x * RB;
  if (threadIdx.x < RMAX_EB * 16) asked[threadIdx.x] = 0;
  // normalisation: a wave per row, all of a wave's rows requested before the first is reduced
  constexpr int OWN = RB / WAVES;
  Row8 xs[OWN][NV];
#pragma unroll
  for (int q = 0; q < OWN; ++q) {
    const int rr = wv + q * WAVES;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int c = lane + i * MOE_WAVE;
      if (t0 + rr < T && c < H8) xs[q][i] = load8(x + (size_t)(t0 + rr) * H + c * 8);
    }
  }
#pragma unroll
  for (int q = 0; q < OWN; ++q) {
    const int rr = wv + q * WAVES, t = t0 + rr;
    const Row8(&xv)[NV] = xs[q];
    if (t >= T) {  // wave-uniform: rows past the end are zero rows for the product
#pragma unroll
      for (int i = 0; i < NV; ++i) {
        const int c = lane + i * MOE_WAVE;
        if (c < H8) *reinterpret_cast<u32x4*>(rows + rr * LDT + c * 8) = u32x4{0, 0, 0, 0};
      }
      continue;
    }
    // (four partial sums, as the block of rmsnorm_fwd_kernel forms them: the same bits)
    float sum = 0.f;
#pragma unroll
    for (int g = 0; g < NW && g < NV; ++g) {
      float ss = 0.f;
#pragma unroll
      for (int i = g; i < NV; i += NW) {
        if (lane + i * MOE_WAVE < H8) {
#pragma unroll
          for (int j = 0; j < 8; ++j) ss += xv[i].v[j] * xv[i].v[j];
        }
      }
      sum += moe_wave_sum_f32(ss);
    }
    const float r = rsqrtf(sum / (float)H + eps);
    if (lane == 0) rstd[t] = r;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int c = lane + i * MOE_WAVE;
      if (c < H8) {
        const Row8 wn = load8(w + c * 8);
        Row8 o;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          float v = xv[i].v[j] * r;
          if (is_bf16<XT>::value) v = bf16_to_f32(f32_to_bf16(v));  // `.to(input_dtype)`, norm.py:19
          o.v[j] = wn.v[j] * v;
        }
        store8(xn + (size_t)t * H + c * 8, o);
        store8(rows + rr * LDT + c * 8, o);
      }
    }
  }
  __syncthreads();
  // logits[m][e] = sum_h rows[m][h] * wr[e][h]: lane l holds A row l % 16 (token) and B row
  // l % 16 of the column block (expert), 8 consecutive h at (l / 16) * 8 of the 32-wide k-step.
  // Wave wv has every NW-th k-step from wv % NW on, and of the column blocks every GROUPS-th from wv / NW on: the sums do not depend on
  // the number of waves.
  constexpr int GROUPS = WAVES / NW, MINE = RMAX_EB / GROUPS;
  const int EB = E / 16, kg = wv % NW, cg = wv / NW;
  f32x4 acc[MINE];
#pragma unroll
  for (int nb = 0; nb < MINE; ++nb) acc[nb] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int l16 = lane & 15, lq = lane >> 4;
  // (the router's rows come from L2: so many k-steps' are requested while as many before are multiplied)
  const auto product = [&](auto eb_c) {
    constexpr int EBT = decltype(eb_c)::value;  // column blocks, rounded up: the surplus repeats the last
    constexpr int AHEAD = EBT <= 2 ? 4 / EBT : 1;
    bf16x8 b[2][AHEAD][EBT];
    const int n = (H / 32 - kg + NW - 1) / NW;  // this wave's k-steps
    const auto request = [&](int s, bf16x8(&to)[AHEAD][EBT]) {
#pragma unroll
      for (int d = 0; d < AHEAD; ++d) {
        if (s + d >= n) break;
        const int ks = kg + (s + d) * NW;
#pragma unroll
        for (int nb = 0; nb < EBT; ++nb) {
          const int c = cg + nb * GROUPS < EB ? cg + nb * GROUPS : EB - 1;
          to[d][nb] = *reinterpret_cast<const bf16x8*>(wr + (size_t)(c * 16 + l16) * H + ks * 32 + lq * 8);
        }
      }
    };
    const auto multiply = [&](int s, const bf16x8(&from)[AHEAD][EBT]) {
#pragma unroll
      for (int d = 0; d < AHEAD; ++d) {
        if (s + d >= n) break;
        const bf16x8 a = *reinterpret_cast<const bf16x8*>(rows + l16 * LDT + (kg + (s + d) * NW) * 32 + lq * 8);
#pragma unroll
        for (int nb = 0; nb < EBT; ++nb) acc[nb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, from[d][nb], acc[nb], 0, 0, 0);
      }
    };
    request(0, b[0]);
    for (int s = 0; s < n; s += 2 * AHEAD) {
      request(s + AHEAD, b[1]);
      multiply(s, b[0]);
      request(s + 2 * AHEAD, b[0]);
      multiply(s + AHEAD, b[1]);
    }
  };
  if (cg < EB) {
    const int mine = (EB - cg + GROUPS - 1) / GROUPS;
    if (mine <= 1) product(std::integral_constant<int, 1>{});
    else if (MINE <= 2 || mine <= 2) product(std::integral_constant<int, 2>{});
    else product(std::integral_constant<int, MINE>{});
  }
  __syncthreads();  // every wave is done with the rows: their memory takes the partial products
  float* part = reinterpret_cast<float*>(rows);  // [NW][RB][E]
  // accumulator layout: lane l holds column l % 16 (expert) of rows 4 * (l / 16) .. + 3 (tokens)
#pragma unroll
  for (int nb = 0; nb < MINE; ++nb) {
    const int c = cg + nb * GROUPS;
    if (c < EB) {
#pragma unroll
      for (int i = 0; i < 4; ++i) part[(kg * RB + lq * 4 + i) * E + c * 16 + l16] = acc[nb][i];
    }
  }
  __syncthreads();
  for (int idx = threadIdx.x; idx < RB * E; idx += WAVES * MOE_WAVE) {
    float v = 0.f;
#pragma unroll
    for (int q = 0; q < NW; ++q) v += part[q * RB * E + idx];  // fixed order: reproducible
    const uint16_t b = f32_to_bf16(v);
    lg16[idx] = b;
    const int m = idx / E;
    if (t0 + m < T) logits[(size_t)(t0 + m) * E + (idx - m * E)] = b;
  }
  __syncthreads();
  // selection: one wave per token
#pragma unroll
  for (int q = 0; q < OWN; ++q) {
    const int m = wv + q * WAVES, t = t0 + m;
    if (t >= T) break;
    uint32_t key[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int e = i * MOE_WAVE + lane;
      key[i] = e < E ? moe_orderable(bf16_to_f32(lg16[m * E + e])) : 0;
    }
    int my_id;
    float my_gate;
    if (E <= MOE_WAVE) {
      uint32_t one[1] = {key[0]};
      moe_topk_softmax_wave<1>(one, k, lane, my_id, my_gate);
    } else {
      moe_topk_softmax_wave<2>(key, k, lane, my_id, my_gate);
    }
    if (lane < k) {
      ids[(size_t)t * k + lane] = my_id;
      gates[(size_t)t * k + lane] = my_gate;
      if (table) atomicOr(&asked[my_id], 1u << m);
    }
  }
  if (!table) return;
  __syncthreads();
  const int words = (E + 3) / 4;  // (a row of place.hip's table)
  if (threadIdx.x < words) {
    uint32_t c = 0;
#pragma unroll
    for (int b = 0; b < 4; ++b) c |= (uint32_t)__popc(asked[threadIdx.x * 4 + b]) << (8 * b);
    table[(size_t)blockIdx.x * words + threadIdx.x] = c;
  }
}

// dx[t] = dres[t] + rstd * (w*g - xhat * mean(w*g*xhat)),  g = d1[t] + d2[t],  xhat = x*rstd;
// part[block] = sum over the block's rows of g*xhat.
template <typename XT, typename DT, int NV>
__global__ __launch_bounds__(NT) void rmsnorm_bwd_kernel(
    const XT* __restrict__ x, const float* __restrict__ w, const float* __restrict__ rstd,
    const DT* __restrict__ d1, const uint16_t* __restrict__ d2, const XT* __restrict__ dres, int T,
    int H8, XT* __restrict__ dx, float* __restrict__ part) {
  __shared__ float red[NW];
  const int H = H8 * 8;
  Row8 wv[NV], dwv[NV];
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int c = threadIdx.x + i * NT;
    if (c < H8) wv[i] = load8(w + c * 8);
#pragma unroll
    for (int j = 0; j < 8; ++j) dwv[i].v[j] = 0.f;
  }
  for (int t = blockIdx.x; t < T; t += gridDim.x) {
    const float r = rstd[t];
    Row8 xh[NV], gw[NV];
    float dot = 0.f;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int c = threadIdx.x + i * NT;
      if (c < H8) {
        const size_t at = (size_t)t * H + c * 8;
        xh[i] = load8(x + at);
        Row8 g = load8(d1 + at);
        if (d2) {
          const Row8 g2 = load8(d2 + at);
#pragma unroll
          for (int j = 0; j < 8; ++j) g.v[j] += g2.v[j];
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          xh[i].v[j] *= r;
          dwv[i].v[j] += g.v[j] * xh[i].v[j];
          gw[i].v[j] = g.v[j] * wv[i].v[j];
          dot += gw[i].v[j] * xh[i].v[j];
        }
      }
    }
    dot = block_sum(dot, red);
    const float m = dot / (float)H;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int c = threadIdx.x + i * NT;
      if (c < H8) {
        const size_t at = (size_t)t * H + c * 8;
        Row8 o;
#pragma unroll
        for (int j = 0; j < 8; ++j) o.v[j] = r * (gw[i].v[j] - xh[i].v[j] * m);
        if (dres) {
          const Row8 a = load8(dres + at);
#pragma unroll
          for (int j = 0; j < 8; ++j) o.v[j] += a.v[j];
        }
        store8(dx + at, o);
      }
    }
  }
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int c = threadIdx.x + i * NT;
    if (c < H8) store8(part + (size_t)blockIdx.x * H + c * 8, dwv[i]);
  }
}

// rmsnorm_bwd_kernel with d1 = what moe_permute_bwd_router makes of the rows of dxp, in x's type, in the arithmetic of both.
// Two passes write d1 and read it, a launch apart.  Whole steps, fp32 x, us, two passes -> this, the same bits: 8192 tokens, 8 of 64 experts, 2048
// wide, 2877 -> 2855; 2 of 16 639 -> 611; 12000, 1 of 8, 1024 wide, 288 -> 273; 3000, 8 of 24, 4096 wide, 893 -> 852; 700, 4 of 48, 1400 wide, 355 ->
// 354; 64, 2 of 16, 1024 wide, 165 -> 159.  A block a token, as the norm's mean has it (the rows by themselves have a wave a token): narrow
// rows leave its waves without columns, which is less than the launch only while tokens are few: 832 wide, 9312 tokens 446 -> 438 without; below 4096 tokens
// steps that the host bounds gain 2 % (384 wide, 2563 tokens 174 -> 169; 704 wide, 2188 212 -> 208.5), others are within 1 % (576 wide, 3929 tokens 511 -> 516; 448
// wide, 2837 196 -> 195).  From 1024 columns on none of 25 drawn sizes is slower by more than 0.6 %, 1.013 in the mean.
template <typename XT, int NV>
__global__ __launch_bounds__(NT, NV == 1 ? 4 : 2) void rmsnorm_bwd_rows_kernel(
    const XT* __restrict__ x, const float* __restrict__ w, const float* __restrict__ rstd, const uint16_t* __restrict__ dxp,
    const int32_t* __restrict__ row_to_pos, const RouterGrad rg, const XT* __restrict__ dres, int T, int H8, int k,
    XT* __restrict__ dx, float* __restrict__ part) {
  __shared__ float red[NW];
  const int H = H8 * 8;
  const bool first_wave = uniform((int)(threadIdx.x / MOE_WAVE)) == 0;
  Row8 wv[NV], dwv[NV];
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int c = threadIdx.x + i * NT;
    if (c < H8) wv[i] = load8(w + c * 8);
#pragma unroll
    for (int j = 0; j < 8; ++j) dwv[i].v[j] = 0.f;
  }
  for (int t = blockIdx.x; t < T; t += gridDim.x) {
    const float r = rstd[t];
    int id;
    const float dsel = router_dsel<uint16_t>(rg, row_to_pos, T, k, t, first_wave, id);
    Row8 xh[NV], gw[NV];
    float dot = 0.f;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int c = threadIdx.x + i * NT;
      if (c < H8) {
        xh[i] = load8(x + (size_t)t * H + c * 8);
        Row8 g, d2;
        sum_rows<true, false>(dxp, nullptr, row_to_pos, rg, id, dsel, t * k, k, H, c * 8, g, d2);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          g.v[j] += bf16_to_f32(f32_to_bf16(d2.v[j]));
          if (sizeof(XT) == 2) g.v[j] = bf16_to_f32(f32_to_bf16(g.v[j]));
          xh[i].v[j] *= r;
          dwv[i].v[j] += g.v[j] * xh[i].v[j];
          gw[i].v[j] = g.v[j] * wv[i].v[j];
          dot += gw[i].v[j] * xh[i].v[j];
        }
      }
    }
    dot = block_sum(dot, red);
    const float m = dot / (float)H;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int c = threadIdx.x + i * NT;
      if (c < H8) {
        const size_t at = (size_t)t * H + c * 8;
        Row8 o;
#pragma unroll
        for (int j = 0; j < 8; ++j) o.v[j] = r * (gw[i].v[j] - xh[i].v[j] * m);
        if (dres) {
          const Row8 a = load8(dres + at);
#pragma unroll
          for (int j = 0; j < 8; ++j) o.v[j] += a.v[j];
        }
        store8(dx + at, o);
      }
    }
  }
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int c = threadIdx.x + i * NT;
    if (c < H8) store8(part + (size_t)blockIdx.x * H + c * 8, dwv[i]);
  }
}

// dw[c] = sum_b part[b][c], b ascending within each of CG row groups, groups combined in ascending order:
// one fixed order whatever the launch.  A block owns 64 columns, a wave a group of rows: the launch has
// few blocks (32 at H = 2048), so what bounds it is the length of a wave's chain of loads; with 16 groups
// and eight loads in flight it takes 6 us where 4 groups with one took 64 (1024 partial rows of 2048).
constexpr int CG = 16;
__global__ __launch_bounds__(CG* MOE_WAVE) void colsum_kernel(const float* __restrict__ part, int nb, int H,
                                                             float* __restrict__ dw) {
  __shared__ float red[CG][MOE_WAVE];
  const int c = blockIdx.x * MOE_WAVE + lane_id(), g = threadIdx.x / MOE_WAVE;
  const int per = (nb + CG - 1) / CG;
  const int lo = g * per, hi = lo + per < nb ? lo + per : nb;
  float s = 0.f;
  if (c < H) {
    int b = lo;
    for (; b + 8 <= hi; b += 8) {
      float v[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) v[i] = part[(size_t)(b + i) * H + c];
#pragma unroll
      for (int i = 0; i < 8; ++i) s += v[i];
    }
    for (; b < hi; ++b) s += part[(size_t)b * H + c];
  }
  red[g][lane_id()] = s;
  __syncthreads();
  if (g == 0 && c < H) {
    float tot = 0.f;
#pragma unroll
    for (int i = 0; i < CG; ++i) tot += red[i][lane_id()];
    dw[c] = tot;
  }
}

inline int bwd_blocks(int64_t T) { return (int)(T < BWD_BLOCKS ? (T < 1 ? 1 : T) : BWD_BLOCKS); }

inline int pick_nv(int64_t H) {
  const int64_t need = (H / 8 + NT - 1) / NT;
  return need <= 1 ? 1 : need <= 2 ? 2 : need <= 4 ? 4 : 0;  // H <= 8192
}

template <typename XT>
int launch_fwd(const void* x, const float* w, float eps, int64_t T, int64_t H, uint16_t* xn,
               float* rstd, hipStream_t s) {
  const dim3 grid((unsigned)(T < 256 * 16 ? T : 256 * 16)), block(NT);
#define MOE_NORM_FWD(NV)                                                                          \
  hipLaunchKernelGGL((rmsnorm_fwd_kernel<XT, NV>), grid, block, 0, s, (const XT*)x, w, eps, (int)T, \
                     (int)(H / 8), xn, rstd)
  switch (pick_nv(H)) {
    case 1: MOE_NORM_FWD(1); break;
    case 2: MOE_NORM_FWD(2); break;
    case 4: MOE_NORM_FWD(4); break;
    default: return MOE_ERR_LIMIT;
  }
#undef MOE_NORM_FWD
  return moe_launch_status();
}

template <typename XT, typename DT>
int launch_bwd(const void* x, const float* w, const float* rstd, const void* d1, const uint16_t* d2,
               const void* dres, int64_t T, int64_t H, void* dx, float* part, hipStream_t s) {
  const dim3 grid((unsigned)bwd_blocks(T)), block(NT);
#define MOE_NORM_BWD(NV)                                                                       \
  hipLaunchKernelGGL((rmsnorm_bwd_kernel<XT, DT, NV>), grid, block, 0, s, (const XT*)x, w, rstd, \
                     (const DT*)d1, d2, (const XT*)dres, (int)T, (int)(H / 8), (XT*)dx, part)
  switch (pick_nv(H)) {
    case 1: MOE_NORM_BWD(1); break;
    case 2: MOE_NORM_BWD(2); break;
    case 4: MOE_NORM_BWD(4); break;
    default: return MOE_ERR_LIMIT;
  }
#undef MOE_NORM_BWD
  return moe_launch_status();
}

int check_norm(int64_t T, int64_t H) {
  if (T < 0 || H <= 0 || (H % 8) != 0) return MOE_ERR_SHAPE;
  if (T > (int64_t)1 << 30 || pick_nv(H) == 0) return MOE_ERR_LIMIT;
  return 0;
}

}  // namespace

extern "C" int moe_rmsnorm_fwd(const void* x, int x_dtype, const float* weight, float eps, int64_t T,
                               int64_t H, uint16_t* xn, float* rstd, void* stream) {
  if (int rc = check_norm(T, H)) return rc;
  if (T == 0) return 0;
  MOE_CHECK_PTR(x);
  MOE_CHECK_PTR(weight);
  MOE_CHECK_PTR(xn);
  if (!rstd) return MOE_ERR_NULL;
  hipStream_t s = (hipStream_t)stream;
  if (x_dtype == MOE_DT_BF16) return launch_fwd<uint16_t>(x, weight, eps, T, H, xn, rstd, s);
  if (x_dtype == MOE_DT_F32) return launch_fwd<float>(x, weight, eps, T, H, xn, rstd, s);
  return MOE_ERR_DTYPE;
}

extern "C" int moe_rmsnorm_router_supported(int64_t H, int64_t E, int64_t k) {
  return (H > 0 && E > 0 && k > 0 && (H % 32) == 0 && H <= 4096 && (E % 16) == 0 && E <= 16 * RMAX_EB && k <= E &&
          k <= MOE_MAX_TOPK)
             ? 1 : 0;
}

int moe_rmsnorm_router_count(const void* x, int x_dtype, const float* weight, float eps, const uint16_t* router_weight,
                             int64_t T, int64_t H, int64_t E, int64_t k, uint16_t* xn, float* rstd, uint16_t* logits,
                             int32_t* ids, float* gates, void* table, void* stream) {
  if (int rc = check_norm(T, H)) return rc;
  if (E <= 0 || k <= 0 || k > E) return MOE_ERR_SHAPE;
  if (!moe_rmsnorm_router_supported(H, E, k)) return MOE_ERR_LIMIT;
  if (T == 0) return 0;
  MOE_CHECK_PTR(x);
  MOE_CHECK_PTR(weight);
  MOE_CHECK_PTR(router_weight);
  MOE_CHECK_PTR(xn);
  if (!rstd || !logits || !ids || !gates) return MOE_ERR_NULL;
  hipStream_t s = (hipStream_t)stream;
  const dim3 grid((unsigned)((T + RB - 1) / RB)), block(ROUTER_WAVES * MOE_WAVE);
  const size_t lds = (size_t)RB * (H + 8) * 2 > (size_t)NW * RB * E * 4 ? (size_t)RB * (H + 8) * 2 : (size_t)NW * RB * E * 4;
  constexpr int MAX_ROUTER_LDS = RB * (4096 + 8) * 2 > NW * RB * 16 * RMAX_EB * 4 ? RB * (4096 + 8) * 2 : NW * RB * 16 * RMAX_EB * 4;
  if (lds > (size_t)MAX_ROUTER_LDS) return MOE_ERR_LIMIT;
#define MOE_NORM_ROUTER(XT, NV)                                                                          \
  do {                                                                                                   \
    auto kern = rmsnorm_router_fwd_kernel<XT, NV, ROUTER_WAVES>;                                                     \
    static bool attr_done[MOE_MAX_DEVICES]; /* per GPU and instantiation: set once, to the largest */    \
    const int dev = moe_current_device();   /* footprint any supported shape asks for              */    \
    if (!attr_done[dev]) {                                                                               \
      hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize,  \
                                         MAX_ROUTER_LDS);                                                \
      if (e != hipSuccess) return (int)e;                                                                \
      attr_done[dev] = true;                                                                             \
    }                                                                                                    \
    hipLaunchKernelGGL(kern, grid, block, lds, s, (const XT*)x, weight, eps, (int)T, (int)(H / 8),       \
                       router_weight, (int)E, (int)k, xn, rstd, logits, ids, gates, (uint32_t*)table);   \
  } while (0)
  const int64_t groups = (H / 8 + MOE_WAVE - 1) / MOE_WAVE;  // 16-byte column groups per lane (H <= 4096: at most 8)
  if (x_dtype == MOE_DT_BF16) {
    if (groups <= 2) MOE_NORM_ROUTER(uint16_t, 2);
    else if (groups <= 4) MOE_NORM_ROUTER(uint16_t, 4);
    else MOE_NORM_ROUTER(uint16_t, 8);
  } else if (x_dtype == MOE_DT_F32) {
    if (groups <= 2) MOE_NORM_ROUTER(float, 2);
    else if (groups <= 4) MOE_NORM_ROUTER(float, 4);
    else MOE_NORM_ROUTER(float, 8);
  } else {
    return MOE_ERR_DTYPE;
  }
#undef MOE_NORM_ROUTER
  return moe_launch_status();
}

extern "C" int moe_rmsnorm_router_fwd(const void* x, int x_dtype, const float* weight, float eps,
                                      const uint16_t* router_weight, int64_t T, int64_t H, int64_t E,
                                      int64_t k, uint16_t* xn, float* rstd, uint16_t* logits,
                                      int32_t* ids, float* gates, void* stream) {
  return moe_rmsnorm_router_count(x, x_dtype, weight, eps, router_weight, T, H, E, k, xn, rstd, logits, ids, gates, nullptr,
                                  stream);
}

extern "C" int64_t moe_rmsnorm_bwd_workspace_bytes(int64_t T, int64_t H) {
  if (T < 0 || H <= 0) return 0;
  return (int64_t)bwd_blocks(T) * H * (int64_t)sizeof(float);
}

extern "C" int moe_rmsnorm_bwd(const void* x, int x_dtype, const float* weight, const float* rstd,
                               const void* d1, int d1_dtype, const uint16_t* d2, const void* dres,
                               int64_t T, int64_t H, void* dx, float* dweight, void* workspace,
                               int64_t workspace_bytes, void* stream) {
  if (int rc = check_norm(T, H)) return rc;
  MOE_CHECK_PTR(dweight);
  hipStream_t s = (hipStream_t)stream;
  if (T == 0) {  // no rows: the weight gradient is zero
    hipLaunchKernelGGL(colsum_kernel, dim3((unsigned)((H + MOE_WAVE - 1) / MOE_WAVE)), dim3(CG * MOE_WAVE), 0, s,
                       (const float*)dweight, 0, (int)H, dweight);
    return moe_launch_status();
  }
  MOE_CHECK_PTR(x);
  MOE_CHECK_PTR(weight);
  MOE_CHECK_PTR(d1);
  MOE_CHECK_PTR(dx);
  MOE_CHECK_PTR(workspace);
  if (!rstd) return MOE_ERR_NULL;
  if (d2 && !aligned16(d2)) return MOE_ERR_ALIGN;
  if (dres && !aligned16(dres)) return MOE_ERR_ALIGN;
  if (workspace_bytes < moe_rmsnorm_bwd_workspace_bytes(T, H)) return MOE_ERR_WORKSPACE;
  float* part = (float*)workspace;
  int rc;
  if (x_dtype == MOE_DT_BF16 && d1_dtype == MOE_DT_BF16)
    rc = launch_bwd<uint16_t, uint16_t>(x, weight, rstd, d1, d2, dres, T, H, dx, part, s);
  else if (x_dtype == MOE_DT_BF16 && d1_dtype == MOE_DT_F32)
    rc = launch_bwd<uint16_t, float>(x, weight, rstd, d1, d2, dres, T, H, dx, part, s);
  else if (x_dtype == MOE_DT_F32 && d1_dtype == MOE_DT_BF16)
    rc = launch_bwd<float, uint16_t>(x, weight, rstd, d1, d2, dres, T, H, dx, part, s);
  else if (x_dtype == MOE_DT_F32 && d1_dtype == MOE_DT_F32)
    rc = launch_bwd<float, float>(x, weight, rstd, d1, d2, dres, T, H, dx, part, s);
  else
    return MOE_ERR_DTYPE;
  if (rc) return rc;
  hipLaunchKernelGGL(colsum_kernel, dim3((unsigned)((H + MOE_WAVE - 1) / MOE_WAVE)), dim3(CG * MOE_WAVE), 0, s,
                     (const float*)part, bwd_blocks(T), (int)H, dweight);
  return moe_launch_status();
}

bool moe_norm_rows_ok(int64_t T, int64_t H) {
  return T > 0 && T <= (int64_t)1 << 30 && H % 8 == 0 && pick_nv(H) != 0 && (H >= 1024 || T <= 4096);
}

int moe_rmsnorm_bwd_rows(const MoeNormBackward& n, const uint16_t* dxp, const int32_t* row_to_pos, const float* part, int64_t P,
                         const float* gates, const int32_t* ids, const uint16_t* wr, int64_t T, int64_t H, int64_t k, int64_t ld,
                         uint16_t* dlogits, void* dx, hipStream_t s) {
  if (int rc = check_norm(T, H)) return rc;
  if (T == 0) return MOE_ERR_SHAPE;
  for (const void* q : {n.x, (const void*)n.weight, (const void*)n.dweight, (const void*)n.workspace, (const void*)dxp, (const void*)wr,
                        (const void*)dx})
    MOE_CHECK_PTR(q);
  if (!n.rstd || !part || !gates || !ids || !dlogits || !row_to_pos) return MOE_ERR_NULL;
  if (!aligned16(n.dres)) return MOE_ERR_ALIGN;
  if (n.workspace_bytes < moe_rmsnorm_bwd_workspace_bytes(T, H)) return MOE_ERR_WORKSPACE;
  const RouterGrad rg{part, (int)P, gates, ids, wr, dlogits, (int)ld};
  const auto go = [&](auto xt, auto nv) {
    using XT = decltype(xt);
    hipLaunchKernelGGL((rmsnorm_bwd_rows_kernel<XT, decltype(nv)::value>), dim3((unsigned)bwd_blocks(T)), dim3(NT), 0, s,
                       (const XT*)n.x, n.weight, n.rstd, dxp, row_to_pos, rg, (const XT*)n.dres, (int)T, (int)(H / 8), (int)k, (XT*)dx,
                       (float*)n.workspace);
    return moe_launch_status();
  };
  const auto of = [&](auto xt) {
    const int nv = pick_nv(H);
    return nv == 1 ? go(xt, std::integral_constant<int, 1>{}) : nv == 2 ? go(xt, std::integral_constant<int, 2>{})
                                                                       : go(xt, std::integral_constant<int, 4>{});
  };
  if (n.x_dtype != MOE_DT_BF16 && n.x_dtype != MOE_DT_F32) return MOE_ERR_DTYPE;
  if (const int rc = n.x_dtype == MOE_DT_BF16 ? of(uint16_t{}) : of(float{})) return rc;
  hipLaunchKernelGGL(colsum_kernel, dim3((unsigned)((H + MOE_WAVE - 1) / MOE_WAVE)), dim3(CG * MOE_WAVE), 0, s, (const float*)n.workspace,
                     bwd_blocks(T), (int)H, n.dweight);
  return moe_launch_status();
}
