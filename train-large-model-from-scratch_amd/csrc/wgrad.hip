// Weight gradients of small launches: all three stacks and the router in one kernel.
//
// The tiled kernel of gemm.hip makes one workgroup per 256 x 256 tile of one stack and walks an
// expert's rows; with few experts or small matrices that fills a part of the chip, three launches in a
// row, and under skewed routing the largest expert's tiles set the time.  It used to be cut into row
// segments stack by stack: eight launches, and two thirds of the work went through fp32 partial sums (8192
// tokens, 8 experts, Zipf: 107 us of products and 34 us of sums).  Here a job is a 128 x 128 tile of any
// of the results over at most L rows of an expert, in one launch: there are jobs enough for the chip at three
// times the segment length, and only experts of more than L rows are cut at all (the others are written
// straight to their result).  One more launch adds up what was cut.
#include "tile_ops.h"

#include "internal.h"

namespace {

constexpr int WBM = 128, WBN = 128;  // tile
constexpr int WK = 64;               // rows per step
constexpr int WNT = 256;             // threads: 2 x 2 waves
constexpr int WFM = WBM / 64, WFN = WBN / 64;  // 32 x 32 blocks per wave
using WOpA = OpOuter<WBM, WK, WNT>;
using WOpB = OpOuter<WBN, WK, WNT>;

struct Stack {
  const uint16_t *a, *b;  // [R, M] and [R, N] with row strides lda, ldb
  void* out;              // [E, M, N]
  float* part;            // partial sums [slot][M][N]
  int lda, ldb, M, N, n_tiles, tiles, out_f32, accumulate;
};
struct MultiArgs {
  Stack s[3];
  Stack router;           // one "expert" of T rows, cut into r_slices slices of r_rows
  const int32_t* offs;
  int E, L, n_stacks, tiles;   // tiles: of all stacks together
  int T, r_rows, r_slices;
};

// Segment `seg` of the experts' rows: experts of more than L / 2 rows come first (so that the short jobs fill
// the end), each cut into ceil(n / L) equal parts, an empty one still being a part.
struct Segment {
  int e, row0, row_end, parts, slot;  // slot: of its partial sums, where the expert has several parts
};
__device__ __forceinline__ int expert_rows(const int32_t* offs, int e, int E) {
  const int n = e < E ? offs[e + 1] - offs[e] : 0;
  return n > 0 ? n : 0;
}
__device__ __forceinline__ int parts_of(int n, int L) { return n > L ? (n + L - 1) / L : 1; }

// Number of partial-sum slots of the experts before e.
__device__ __forceinline__ int slots_before(const int32_t* offs, int E, int L, int e) {
  const int lane = lane_id();
  int slots = 0;
  for (int b = 0; b < e; b += MOE_WAVE) {
    const int p = b + lane < e ? parts_of(expert_rows(offs, b + lane, E), L) : 1;
    slots += uniform(__shfl(wave_inclusive(p > 1 ? p : 0), MOE_WAVE - 1, MOE_WAVE));
  }
  return slots;
}
__device__ __forceinline__ bool find_segment(const int32_t* offs, int E, int L, int seg, Segment& s) {
  const int lane = lane_id();
  int carry = 0;
  for (int pass = 0; pass < 2; ++pass)
    for (int b = 0; b < E; b += MOE_WAVE) {
      const int n = expert_rows(offs, b + lane, E);
      const bool mine = b + lane < E && (2 * n > L) == (pass == 0);
      const int p = mine ? parts_of(n, L) : 0;
      const int incl = wave_inclusive(p);
      const int total = uniform(__shfl(incl, MOE_WAVE - 1, MOE_WAVE));
      if (seg < carry + total) {
        const int f = __builtin_ctzll(__ballot(carry + incl > seg));
        // (read into scalar registers: everything derived from these is then known to be the same in every
        // lane, which the buffer resources of the operands need)
        s.e = uniform(b + f);
        s.parts = uniform(__shfl(p, f, MOE_WAVE));
        const int j = seg - (carry + uniform(__shfl(incl, f, MOE_WAVE)) - s.parts);
        const int lo = uniform(offs[s.e]), rows = uniform(__shfl(n, f, MOE_WAVE));
        s.row0 = lo + uniform((int)((long long)rows * j / s.parts));
        s.row_end = lo + uniform((int)((long long)rows * (j + 1) / s.parts));
        s.slot = s.parts > 1 ? slots_before(offs, E, L, s.e) + j : 0;
        return true;
      }
      carry += total;
    }
  return false;
}

// One job per workgroup; three workgroups share a compute unit (41 KB of LDS, four waves of 64 x 64) and hide
// each other's barriers, loads and epilogues, so the loop is the plain one: the step's lines go from registers to
// LDS, the next step's are requested, the products run.  Lines keep their memory order in LDS and are read
// through the transposing read.
__global__ __launch_bounds__(WNT, 3) void wgrad_multi_kernel(const MultiArgs p) {
  __shared__ __attribute__((aligned(16))) uint16_t sm[WOpA::LDS_ELEMS + WOpB::LDS_ELEMS];
  const int lane = lane_id(), wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / MOE_WAVE));
  const int wm = wv >> 1, wn = wv & 1;
  // workgroup b runs on XCD b % 8: of 512 consecutive jobs each XCD takes 64 consecutive ones, which
  // share an expert's rows
  const int nb = gridDim.x, b = blockIdx.x;
  int job = b;
  if ((b | 511) < nb) job = (b & ~511) + (b & 7) * 64 + ((b & 511) >> 3);
  Stack st;
  Segment sg;
  int tile;
  const int r_jobs = p.r_slices * p.router.tiles;
  if (job < r_jobs) {
    st = p.router;
    const int sl = job / st.tiles;
    tile = job - sl * st.tiles;
    sg.e = 0;
    sg.row0 = sl * p.r_rows;
    sg.row_end = sg.row0 + p.r_rows < p.T ? sg.row0 + p.r_rows : p.T;
    sg.parts = 2;  // (its sums always go through the second kernel, which may have fewer rows to write)
    sg.slot = sl;
  } else {
    job -= r_jobs;
    const int seg = job / p.tiles;
    tile = job - seg * p.tiles;
    if (!find_segment(p.offs, p.E, p.L, seg, sg)) return;
    int k = 0;
    while (k + 1 < p.n_stacks && tile >= p.s[k].tiles) tile -= p.s[k++].tiles;
    st = p.s[k];
  }
  const int m0 = tile / st.n_tiles * WBM, n0 = tile % st.n_tiles * WBN;
  const int rows = uniform(sg.row_end - sg.row0);
  WOpA opA;
  WOpB opB;
  opA.init(st.lda);
  opB.init(st.ldb);
  const View vA = make_view(st.a + (long long)sg.row0 * st.lda + m0, (long long)rows * st.lda - m0);
  const View vB = make_view(st.b + (long long)sg.row0 * st.ldb + n0, (long long)rows * st.ldb - n0);
  uint16_t *sA = sm, *sB = sm + WOpA::LDS_ELEMS;
  u32x4 stage[WOpA::CH + WOpB::CH];
  const auto request = [&](int k0) {
    const __amdgpu_buffer_rsrc_t ra = view_rsrc(vA, WOpA::k_bytes(k0, st.lda)), rb = view_rsrc(vB, WOpB::k_bytes(k0, st.ldb));
#pragma unroll
    for (int c = 0; c < WOpA::CH; ++c) stage[c] = opA.load_one(c, ra);
#pragma unroll
    for (int c = 0; c < WOpB::CH; ++c) stage[WOpA::CH + c] = opB.load_one(c, rb);
  };
  f32x16 acc[WFM][WFN];
#pragma unroll
  for (int i = 0; i < WFM; ++i)
#pragma unroll
    for (int j = 0; j < WFN; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;
  const int offA = WOpA::lane_off(lane), offB = WOpB::lane_off(lane);
  if (rows > 0) request(0);
  for (int k0 = 0; k0 < rows; k0 += WK) {
    lds_barrier();  // the step before is read
#pragma unroll
    for (int c = 0; c < WOpA::CH; ++c) opA.store_one(c, sA, stage[c]);
#pragma unroll
    for (int c = 0; c < WOpB::CH; ++c) opB.store_one(c, sB, stage[WOpA::CH + c]);
    lds_barrier();
    if (k0 + WK < rows) request(k0 + WK);
    // (a step's fragments are read in the shadow of the products of the step before: the fences keep the
    // compiler from clumping the reads in front of their use)
    bf16x8 fa[2][WFM], fb[2][WFN];
    const auto read_one = [&](int u, int ks) {  // in the order the products need them
      if (u == 0) fa[ks & 1][0] = WOpA::frag(sA, offA, wm * (WBM / 2), ks);
      else if (u <= WFN) fb[ks & 1][u - 1] = WOpB::frag(sB, offB, wn * (WBN / 2) + (u - 1) * 32, ks);
      else fa[ks & 1][u - WFN] = WOpA::frag(sA, offA, wm * (WBM / 2) + (u - WFN) * 32, ks);
    };
#pragma unroll
    for (int u = 0; u < WFM + WFN; ++u) read_one(u, 0);
#pragma unroll
    for (int ks = 0; ks < WK / 16; ++ks)
#pragma unroll
      for (int n = 0; n < WFM * WFN; ++n) {
        const int i = n / WFN, j = (i & 1) ? WFN - 1 - n % WFN : n % WFN;  // neighbours share an operand
        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fb[ks & 1][j], fa[ks & 1][i], acc[i][j], 0, 0, 0);
        if (ks + 1 < WK / 16 && n < WFM + WFN) read_one(n, ks + 1);
        __builtin_amdgcn_sched_barrier(0);
      }
  }
  lds_barrier();
  // results leave through LDS in strips of 32 rows x 64 columns, fp32: a wave's accumulators hold row l % 32 and
  // columns 8 q + 4 (l / 32) .. + 3 of each block
  constexpr int SS = 64 + 4;  // words per strip row
  float* strip = reinterpret_cast<float*>(sm) + wv * 32 * SS;
  static_assert(WBN == 128 && 4 * 32 * SS * 4 <= (WOpA::LDS_ELEMS + WOpB::LDS_ELEMS) * 2, "strips fit in the stage");
  const bool partial = sg.parts > 1;
  const bool wide = partial || st.out_f32;
  const long long MN = (long long)st.M * st.N;
  char* out = partial ? (char*)(st.part + sg.slot * MN) : (char*)st.out + sg.e * MN * (wide ? 4 : 2);
  const bool add = !partial && st.accumulate;
#pragma unroll
  for (int i = 0; i < WFM; ++i) {
#pragma unroll
    for (int j = 0; j < WFN; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        *reinterpret_cast<f32x4*>(strip + (lane & 31) * SS + j * 32 + 8 * q + 4 * (lane >> 5)) =
            f32x4{acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]};
    // (a wave's strip is its own: its LDS accesses are in order)
#pragma unroll
    for (int it = 0; it < 4; ++it) {  // 8 lanes a row, 8 columns a lane
      const int r = it * 8 + (lane >> 3), c = (lane & 7) * 8;
      const int m = m0 + wm * (WBM / 2) + i * 32 + r, n = n0 + wn * (WBN / 2) + c;
      const f32x4 lo = *reinterpret_cast<const f32x4*>(strip + r * SS + c);
      const f32x4 hi = *reinterpret_cast<const f32x4*>(strip + r * SS + c + 4);
      if (m < st.M && n < st.N) {
        Row8 v;
#pragma unroll
        for (int x = 0; x < 4; ++x) v.v[x] = lo[x], v.v[4 + x] = hi[x];
        const long long at = (long long)m * st.N + n;
        if (wide) {
          float* dst = reinterpret_cast<float*>(out) + at;
          if (add) {
            const Row8 o = load8(dst);
#pragma unroll
            for (int x = 0; x < 8; ++x) v.v[x] += o.v[x];
          }
          store8(dst, v);
        } else {
          uint16_t* dst = reinterpret_cast<uint16_t*>(out) + at;
          if (add) {  // (the product rounded first, as the tiled kernel adds it)
            const Row8 o = load8(dst);
#pragma unroll
            for (int x = 0; x < 8; ++x) v.v[x] = bf16_to_f32(f32_to_bf16(v.v[x])) + o.v[x];
          }
          store8(dst, v);
        }
      }
    }
  }
}

// dw[e] (+)= the sums of e's parts, ascending, for the experts that were cut (blockIdx.y: which of them; the last:
// the router).  8 elements a thread, the stacks' elements one after the other.
__global__ __launch_bounds__(256) void wgrad_multi_sum_kernel(const MultiArgs p) {
  const int lane = lane_id();
  int e = 0, parts = p.r_slices, slot = 0;
  const bool router = p.r_slices > 0 && blockIdx.y == gridDim.y - 1;
  if (!router) {
    int carry = 0, slots = 0;
    bool found = false;
    for (int b = 0; b < p.E && !found; b += MOE_WAVE) {
      const int n = expert_rows(p.offs, b + lane, p.E);
      const int c = b + lane < p.E && n > p.L ? parts_of(n, p.L) : 0;
      const unsigned long long m = __ballot(c > 0);
      const int incl = wave_inclusive(c);
      const int want = (int)blockIdx.y - carry;
      if (want < __popcll(m)) {
        const bool me = c > 0 && __popcll(m & ((1ull << lane) - 1)) == want;
        const int f = __builtin_ctzll(__ballot(me));
        e = b + f;
        parts = __shfl(c, f, MOE_WAVE);
        slot = slots + __shfl(incl, f, MOE_WAVE) - parts;
        found = true;
      }
      carry += __popcll(m);
      slots += __shfl(incl, MOE_WAVE - 1, MOE_WAVE);
    }
    if (!found) return;
  }
  const int first = router ? 3 : 0, last = router ? 4 : p.n_stacks;
  long long i = blockIdx.x * 256ll + threadIdx.x;
  for (int k = first; k < last; ++k) {
    const Stack& st = router ? p.router : p.s[k];
    const long long n8 = (long long)st.M * st.N / 8;
    // (the router's padded rows are not part of its result)
    const long long o8 = router ? (long long)p.E * st.N / 8 : n8;
    for (; i < n8; i += (long long)gridDim.x * 256) {
      if (i >= o8) continue;
      Row8 acc;
#pragma unroll
      for (int v = 0; v < 8; ++v) acc.v[v] = 0.f;
#pragma unroll 4
      for (int s = 0; s < parts; ++s) {
        const Row8 r = load8(st.part + ((slot + s) * n8 + i) * 8);
#pragma unroll
        for (int v = 0; v < 8; ++v) acc.v[v] += r.v[v];
      }
      const long long at = (e * o8 + i) * 8;
      if (st.out_f32) {
        float* dst = (float*)st.out + at;
        if (st.accumulate) {
          const Row8 o = load8(dst);
#pragma unroll
          for (int v = 0; v < 8; ++v) acc.v[v] += o.v[v];
        }
        store8(dst, acc);
      } else {
        uint16_t* dst = (uint16_t*)st.out + at;
        if (st.accumulate) {
          const Row8 o = load8(dst);
#pragma unroll
          for (int v = 0; v < 8; ++v) acc.v[v] += o.v[v];
        }
        store8(dst, acc);
      }
    }
    i -= n8;
  }
}

int tiles_m(int64_t m) { return (int)((m + WBM - 1) / WBM); }
int tiles_n(int64_t n) { return (int)((n + WBN - 1) / WBN); }

// Longest segment: the rows that would fall to one of two workgroups on every compute unit, were all rows one
// expert's; at least 512.  (8192 tokens, 8 experts, Zipf: 3072; products and sums together 80 us, at 2048 92, at 1024
// 103: what shorter segments balance better, their partial sums cost again.)
int64_t segment_rows(int64_t R, int64_t H, int64_t I) {
  const int64_t tiles = (int64_t)tiles_m(H) * tiles_n(I) + 2 * (int64_t)tiles_m(I) * tiles_n(H);
  int64_t L = R * tiles / (2 * (int64_t)moe_compute_units());
  L = (L + WK - 1) / WK * WK;
  return L < 512 ? 512 : (L > (1 << 30) ? 1 << 30 : L);
}

}  // namespace

int64_t moe_wgrad_multi_part_bytes(int64_t R, int64_t H, int64_t I) {
  return 2 * (R / segment_rows(R, H, I)) * H * I * 4;  // an expert of n > L rows has at most 2 n / L parts
}

int moe_wgrad_multi(const MoeWgradStack (&stacks)[3], int n_stacks, const MoeWgradStack* router, const int32_t* offs,
                    int64_t E, int64_t R, int64_t H, int64_t I, int64_t T, int64_t router_slices,
                    int64_t router_rows, hipStream_t s) {
  MultiArgs a{};
  const auto fill = [](Stack& d, const MoeWgradStack& m) {
    d.a = m.a, d.b = m.b, d.out = m.out, d.part = m.part;
    d.lda = (int)m.lda, d.ldb = (int)m.ldb, d.M = (int)m.M, d.N = (int)m.N;
    d.n_tiles = tiles_n(m.N), d.tiles = tiles_m(m.M) * d.n_tiles;
    d.out_f32 = m.dtype == MOE_DT_F32, d.accumulate = m.accumulate;
  };
  for (int i = 0; i < n_stacks; ++i) {
    fill(a.s[i], stacks[i]);
    a.tiles += a.s[i].tiles;
  }
  a.n_stacks = n_stacks;
  a.offs = offs;
  a.E = (int)E;
  // (from the shapes alone, whichever stacks are wanted: the room for the partial sums was made for it)
  a.L = n_stacks ? (int)segment_rows(R, H, I) : 1;
  a.T = (int)T;
  if (router) {
    fill(a.router, *router);
    a.r_rows = (int)router_rows;
    a.r_slices = (int)router_slices;
  }
  const long long segs = n_stacks ? R / a.L + E : 0;
  const long long jobs = segs * a.tiles + (long long)a.r_slices * a.router.tiles;
  if (jobs <= 0) return 0;
  if (jobs > 0x7fffffffll) return MOE_ERR_LIMIT;
  hipLaunchKernelGGL(wgrad_multi_kernel, dim3((unsigned)jobs), dim3(WNT), 0, s, a);
  const long long cut = n_stacks ? R / a.L : 0;  // experts of more than L rows, at most
  const long long ys = (cut < E ? cut : E) + (router ? 1 : 0);
  if (ys > 0) {
    long long n8 = 0;
    for (int i = 0; i < n_stacks; ++i) n8 += (long long)a.s[i].M * a.s[i].N / 8;
    const long long nr = router ? (long long)a.router.M * a.router.N / 8 : 0;
    if (nr > n8) n8 = nr;
    long long bx = (n8 + 255) / 256;
    if (bx > 2048) bx = 2048;
    hipLaunchKernelGGL(wgrad_multi_sum_kernel, dim3((unsigned)bx, (unsigned)ys), dim3(256), 0, s, a);
  }
  return moe_launch_status();
}
