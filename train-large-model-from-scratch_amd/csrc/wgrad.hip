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
#include "internal.h"
#include "ring.h"

#include <type_traits>

namespace {

constexpr int WBM = 128, WBN = 128;            // tile
constexpr int WK = 32, WSTAGES = 3;            // rows per step, stages of the ring
constexpr int WNT = 256;                       // threads: 2 x 2 waves
constexpr int WFM = WBM / 64, WFN = WBN / 64;  // 32 x 32 blocks per wave
using WOpA = RingOuter<WBM, WK>;
using WOpB = RingOuter<WBN, WK>;
constexpr int WSTAGE = WOpA::BYTES + WOpB::BYTES;

struct Stack {
  const uint16_t *a, *b;  // [R, M] and [R, N] with row strides lda, ldb
  void* out;              // [E, M, N]
  float* part;            // partial sums [slot][M][N]
  int lda, ldb, M, N, n_tiles, tiles, out_f32, accumulate;
  int from;               // row r of b is where row_at[r] says
  float per_n;            // 1 / n_tiles
};
struct MultiArgs {
  Stack s[3];
  Stack router;           // one "expert" of T rows, cut into r_slices slices of r_rows
  const int32_t* offs;
  int E, L, n_stacks, tiles;   // tiles: of all stacks together
  int many;                    // experts of more rows than this come first
  int T, r_rows, r_slices;
  int each, e_each, r_each;  // tiles of a segment to an XCD, its jobs of all segments, its router jobs
  int r_first;               // the router's jobs come first, or last
  int streaming;             // results that replace what is there leave with streaming stores, where rows allow it
  float per_each, r_per_tiles;
  const uint32_t* row_at;    // bytes from b's beginning
  long long from_bytes;      // of a `from` stack's b, less than 2^31
};
// n / d of a wave-uniform n, 1 / d given (exact: n is far below 2^23)
__device__ __forceinline__ int quotient(int n, int d, float per_d) {
  int q = uniform((int)((float)n * per_d));
  q -= q * d > n;
  return q + ((q + 1) * d <= n);
}

// A segment of the experts' rows: experts of many rows (more than L / 2) come first (so that the short jobs fill
// the end), each cut into ceil(n / L) parts, an empty one still being a part.
struct Segment {
  int e, row0, row_end, parts, slot;  // slot: of its partial sums, where the expert has several parts
};
__device__ __forceinline__ int expert_rows(const int32_t* offs, int e, int E) {
  const int n = e < E ? offs[e + 1] - offs[e] : 0;
  return n > 0 ? n : 0;
}
__device__ __forceinline__ int parts_of(int n, int L) {
  if (n <= L) return 1;
  const int q = (int)((float)n * __builtin_amdgcn_rcpf((float)L));  // within one of n / L
  return q + (q * L < n) + ((q + 1) * L < n);
}

// Number of partial-sum slots of the experts before e.
__device__ __forceinline__ int slots_before(const int32_t* offs, int E, int L, int e) {
  const int lane = lane_id();
  int slots = 0;
  for (int b = 0; b < e; b += MOE_WAVE) {
    const int p = b + lane < e ? parts_of(expert_rows(offs, b + lane, E), L) : 1;
    slots += read_lane(wave_inclusive(p > 1 ? p : 0), MOE_WAVE - 1);
  }
  return slots;
}
// Part j of an expert's rows: equal multiples of 64, the last one what is left (maybe nothing).
__device__ __forceinline__ void part_rows(int lo, int rows, int j, Segment& s) {
  const int size = ((int)uniform((int)((float)rows * __builtin_amdgcn_rcpf((float)s.parts))) + 1 + 63) & ~63;
  const int from = j * size < rows ? j * size : rows;
  s.row0 = lo + from;
  s.row_end = lo + (j + 1 < s.parts && from + size < rows ? from + size : rows);
}
// Segment `seg`; first and n: the first row and the number of rows of expert `lane`.
__device__ __forceinline__ bool find_segment(const int32_t* offs, int E, int L, int many, int seg, int first, int n, Segment& s) {
  const int lane = lane_id();
  int carry = 0;
  if (E <= MOE_WAVE) {
    const int p = lane < E ? parts_of(n, L) : 0;
    const bool big = n > many;
    const int ib = wave_inclusive(big ? p : 0);
    const int nbig = read_lane(ib, 63);
    const int is = nbig + wave_inclusive(big ? 0 : p);
    const int sl = wave_inclusive(p > 1 ? p : 0);
    if (seg >= read_lane(is, 63)) return false;
    const int f = __builtin_ctzll(__ballot(lane < E && big == (seg < nbig) && (big ? ib : is) > seg));
    s.e = f;
    s.parts = read_lane(p, f);
    const int j = seg - (read_lane(seg < nbig ? ib : is, f) - s.parts);
    const int lo = read_lane(first, f), rows = read_lane(n, f);
    part_rows(lo, rows, j, s);
    s.slot = s.parts > 1 ? read_lane(sl, f) - s.parts + j : 0;
    return true;
  }
  for (int pass = 0; pass < 2; ++pass)
    for (int b = 0; b < E; b += MOE_WAVE) {
      const int n = expert_rows(offs, b + lane, E);
      const bool mine = b + lane < E && (n > many) == (pass == 0);
      const int p = mine ? parts_of(n, L) : 0;
      const int incl = wave_inclusive(p);
      const int total = read_lane(incl, MOE_WAVE - 1);
      if (seg < carry + total) {
        const int f = __builtin_ctzll(__ballot(carry + incl > seg));
        // (read into scalar registers: everything derived from these is then known to be the same in every
        // lane, which the buffer resources of the operands need)
        s.e = uniform(b + f);
        s.parts = read_lane(p, f);
        const int j = seg - (carry + read_lane(incl, f) - s.parts);
        const int lo = uniform(offs[s.e]), rows = read_lane(n, f);
        part_rows(lo, rows, j, s);
        s.slot = s.parts > 1 ? slots_before(offs, E, L, s.e) + j : 0;
        return true;
      }
      carry += total;
    }
  return false;
}

// One job per workgroup; three workgroups share a compute unit (48 KB of LDS each, four waves of 64 x 64) and hide each
// other's barriers, set-up and epilogues.  Lines come straight into a ring of three 32-row stages, two steps on
// their way.  What bounds it: LDS (a step's fragments and lines take 1.5 times as long there as its products do), then
// the jobs' ends (2.0 to 2.5 of 3 workgroups are there on average) and starts (some 6000 cycles until the first lines are
// asked for, of 28000 and more in the loop).  8192 tokens of 8 experts, 1024 <-> 512, Zipf, and 3333 tokens of 12
// experts, 1416 <-> 568: through staging registers, 41 KB of LDS, the tiles of a segment dealt to one XCD 99 and
// 95 us; this one 79 and 81, and with 16 slices of the router's tokens, at the end of the list, instead of 32 at its start
// 72 and 82.  Two workgroups with two stages of 64 rows or four of 32: 84 and 92, 80 and 93; two with 256 x 128 tiles
// and three stages: 99 and 103; four with two stages of 32 rows 77 and 85 where this one takes 72 and 82.
// FROM: some stack's rows are where row_at says; each kind of stack has a loop of its own.  (With the question asked in one loop, launches that have none
// such pay for it too; asked -> not asked, us: 16936 rows of 128, 320 <-> 512, 61 -> 57 to 65 -> 60; 10065, 1 of 12, 536 <-> 504, 36.8 -> 35.2; 2317, 2 of 8,
// 2304 <-> 832, 84 -> 79; whole steps 226.6 -> 221.5, 174.3 -> 172.7, 301.6 -> 298.9.)
template <bool FROM>
__global__ __launch_bounds__(WNT, 3) void wgrad_multi_kernel(const MultiArgs p) {
  constexpr int KS = WK / 16;
  constexpr int PLACES = MOE_WAVE * 4;  // bytes a wave and stage
  __shared__ __attribute__((aligned(1024))) char sm[WSTAGES * (WSTAGE + (FROM ? 4 * PLACES : 0))];
  const int lane = lane_id(), wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / MOE_WAVE));
  const int wm = wv >> 1, wn = wv & 1;
  // Workgroup b runs on XCD b % 8.  Every XCD takes an eighth of each segment's tiles (neighbours, which share operands
  // in its L2), so that all of them have the same list of segments, long ones first.  (64 consecutive tiles to an
  // XCD, Zipf: 1.30 workgroups a compute unit on average where it is 1.55 now, with two resident.)
  const int b = blockIdx.x, x = b & 7;
  int job = (b >> 3) - (p.r_first ? p.r_each : 0);  // (the experts' from 0)
  Stack st;
  Segment sg;
  int tile;
  // (asked for first: on the way while the job's numbers are worked out)
  const bool of_router = job < 0 || job >= p.e_each, experts = !of_router && lane < p.E;
  const int first = experts ? p.offs[lane] : 0, count = experts ? max(p.offs[lane + 1] - first, 0) : 0;
  if (of_router) {
    job += x * p.r_each + (p.r_first ? p.r_each : -p.e_each);
    if (job >= p.r_slices * p.router.tiles) return;
    st = p.router;
    const int sl = quotient(job, st.tiles, p.r_per_tiles);
    tile = job - sl * st.tiles;
    sg.e = 0;
    sg.row0 = sl * p.r_rows;
    sg.row_end = sg.row0 + p.r_rows < p.T ? sg.row0 + p.r_rows : p.T;
    sg.parts = p.r_slices;
    sg.slot = sl;
  } else {
    const int seg = quotient(job, p.each, p.per_each);
    tile = x * p.each + job - seg * p.each;
    if (tile >= p.tiles || !find_segment(p.offs, p.E, p.L, p.many, seg, first, count, sg)) return;
    const int t0 = p.s[0].tiles, t1 = t0 + p.s[1].tiles;
    st = tile < t0 ? p.s[0] : (tile < t1 ? p.s[1] : p.s[2]);
    tile -= tile < t0 ? 0 : (tile < t1 ? t0 : t1);
  }
  const int tm = quotient(tile, st.n_tiles, st.per_n);
  const int m0 = tm * WBM, n0 = (tile - tm * st.n_tiles) * WBN;
  const int rows = uniform(sg.row_end - sg.row0);
  const View vA = make_view(st.a + (long long)sg.row0 * st.lda + m0, (long long)rows * st.lda - m0);
  const int steps = (rows + WK - 1) / WK;
  const uint32_t stages = lds_address(sm);
  f32x16 acc[WFM][WFN];
#pragma unroll
  for (int i = 0; i < WFM; ++i)
#pragma unroll
    for (int j = 0; j < WFN; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;
  const auto products = [&](auto lines_c) __attribute__((always_inline)) {
    constexpr bool LINES = decltype(lines_c)::value;  // b's lines are where row_at says
    constexpr int LOADS = WOpA::PER_WAVE + WOpB::PER_WAVE + (LINES ? 1 : 0);
    const View vB = LINES ? View{st.b + n0, p.from_bytes - n0 * 2}
                          : make_view(st.b + (long long)sg.row0 * st.ldb + n0, (long long)rows * st.ldb - n0);
    WOpA opA;
    WOpB opB;
    opA.init(st.lda, wv);
    if constexpr (!LINES) opB.init(st.ldb, wv);
    long long askA = 0, askB = 0;
    uint32_t ask_at = 0;
    // (LINES: where a step's lines are comes through LDS, with the stage two steps before; a wave has its own eight.  As vector loads they would have
    // to be waited for with the ring's behind them.  Through the scalar cache, whose loads come in any order and are counted with the LDS reads, a step
    // stood behind them before its first product: 10342 tokens, 2 of 4 experts, 832 <-> 704, 131 us, so and from copies 106.)
    static_assert(WOpB::PER_WAVE == 2 && WOpB::LPP == 4, "a wave's lines");
    const int q = lane / WOpB::CPL;
    const uint32_t piece = ((lane % WOpB::CPL) ^ WOpB::swizzle(q)) * 16;
    const uint32_t places = stages + WSTAGES * WSTAGE + wv * PLACES;  // of step 0; a step's 4 * PLACES further
    uint32_t places_from = lane < 8 ? (((lane >> 2) * 4 + wv) * 4 + (lane & 3) + (WSTAGES - 1) * WK) * 4 : NO_ROW;
    const u32x4 list = ring_rsrc(View{(const uint16_t*)(p.row_at + sg.row0), (long long)rows * 4}, 0, true);
    uint32_t line[2];
    int ask_row = q + wv * 4;
    const auto ask = [&](bool live) {  // (past the last step: empty loads, which the counting of loads relies on)
      opA.load(stages + ask_at, wv, ring_rsrc(vA, askA, live));
      if constexpr (LINES) {
        const u32x4 window = ring_rsrc(vB, 0, live);
#pragma unroll
        for (int i = 0; i < 2; ++i)
          ring_load(stages + ask_at + WOpA::BYTES + (i * 4 + wv) * 1024, window, ask_row + i * 16 < rows ? line[i] + piece : NO_ROW);
        const uint32_t slot = ask_at == 0 ? WSTAGES - 1 : ask_at == WSTAGE ? 0 : 1;  // of two steps on
        ring_load_word(places + slot * (4 * PLACES), list, places_from);
        places_from += WK * 4;
        ask_row += WK;
      } else {
        opB.load(stages + ask_at + WOpA::BYTES, wv, ring_rsrc(vB, askB, live));
        askB += (long long)st.ldb * (WK * 2);
      }
      askA += (long long)st.lda * (WK * 2);
      ask_at = ask_at == (WSTAGES - 1) * WSTAGE ? 0 : ask_at + WSTAGE;
    };
    if constexpr (LINES) {
      const __amdgpu_buffer_rsrc_t first_lines = __builtin_amdgcn_make_buffer_rsrc((void*)(p.row_at + sg.row0), 0, rows * 4, 0x00020000);
      uint32_t at[WSTAGES - 1][2];
#pragma unroll
      for (int i = 0; i < (WSTAGES - 1) * 2; ++i)
        at[i / 2][i & 1] = __builtin_amdgcn_raw_buffer_load_b32(first_lines, (ask_row + i * 16) * 4, 0, 0);
      asm volatile("" : "+v"(at[0][0]), "+v"(at[0][1]), "+v"(at[1][0]), "+v"(at[1][1]));  // (waited for here, not behind the ring's first loads)
#pragma unroll
      for (int i = 0; i < WSTAGES - 1; ++i) {
        line[0] = at[i][0], line[1] = at[i][1];
        ask(i < steps);
      }
    } else {
#pragma unroll
      for (int i = 0; i < WSTAGES - 1; ++i) ask(i < steps);
    }
    const WOpA::Place inA = WOpA::place(wm * (WBM / 2));
    const WOpB::Place inB = WOpB::place(wn * (WBN / 2));
    uint32_t at = 0;
    for (int s = 0; s < steps; ++s) {
      ring_wait<(WSTAGES - 2) * LOADS>();
      const char *sA = sm + at, *sB = sA + WOpA::BYTES;
      bf16x8 fa[2][WFM], fb[2][WFN];
      const auto read_one = [&](int u, int ks) {  // in the order the products need them
        if (u == 0) fa[ks & 1][0] = WOpA::frag(sA, inA, 0, ks);
        else if (u <= WFN) fb[ks & 1][u - 1] = WOpB::frag(sB, inB, (u - 1) * 32, ks);
        else fa[ks & 1][u - WFN] = WOpA::frag(sA, inA, (u - WFN) * 32, ks);
      };
      if constexpr (LINES) {
        const uint32_t slot = ask_at == 0 ? 0 : ask_at == WSTAGE ? 1 : WSTAGES - 1;  // of the step asked for
        const char* here = sm + WSTAGES * WSTAGE + slot * (4 * PLACES) + wv * PLACES + q * 4;
#pragma unroll
        for (int i = 0; i < 2; ++i) line[i] = *reinterpret_cast<const uint32_t*>(here + i * 16);
      }
#pragma unroll
      for (int u = 0; u < WFM + WFN; ++u) read_one(u, 0);
      // (the stage of the step before is free; the requests go out while the first fragments are on their way, and the
      // fences keep the compiler from clumping the other reads in front of their use)
      __builtin_amdgcn_sched_barrier(0);
      ask(s + WSTAGES - 1 < steps);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
#pragma unroll
        for (int n = 0; n < WFM * WFN; ++n) {
          const int i = n / WFN, j = (i & 1) ? WFN - 1 - n % WFN : n % WFN;  // neighbours share an operand
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fb[ks & 1][j], fa[ks & 1][i], acc[i][j], 0, 0, 0);
          if (ks + 1 < KS && n < WFM + WFN) read_one(n, ks + 1);
          __builtin_amdgcn_sched_barrier(0);
        }
      at = at == (WSTAGES - 1) * WSTAGE ? 0 : at + WSTAGE;
    }
  };
  if (FROM && st.from) products(std::true_type{});
  else products(std::false_type{});
  ring_wait<0>();
  // results leave through LDS in strips of 32 rows x 64 columns, fp32: a wave's accumulators hold row l % 32 and
  // columns 8 q + 4 (l / 32) .. + 3 of each block
  constexpr int SS = 64 + 4;  // words per strip row
  float* strip = reinterpret_cast<float*>(sm) + wv * 32 * SS;
  static_assert(WBN == 128 && 4 * 32 * SS * 4 <= WSTAGES * WSTAGE, "strips fit in the stages");
  const bool partial = sg.parts > 1;
  const bool wide = partial || st.out_f32;
  const long long MN = (long long)st.M * st.N;
  char* out = partial ? (char*)(st.part + sg.slot * MN) : (char*)st.out + sg.e * MN * (wide ? 4 : 2);
  const bool add = !partial && st.accumulate;
  // (large results: streaming stores of whole pieces of 64 bytes, a row's in one instruction: the operands' lines stay in L2.  Ordinary ones ->
  // these, whole steps, us: 75 tokens, 3 of 96 experts, 384 <-> 1152, 234 -> 193; 2753 tokens, 24 experts, 1520 <-> 576, fp32, 276 -> 218; of
  // 100 drawn steps of one or two rounds of jobs none is slower.  With ends inside such a piece, which memory then reads
  // first, some are: 958 rows of 64, 3128 <-> 1064, 756 -> 1028 in the tiled kernel)
  const bool stream = p.streaming && !partial && !st.accumulate && st.N * (wide ? 4 : 2) % 64 == 0;
#pragma unroll
  for (int i = 0; i < WFM; ++i) {
#pragma unroll
    for (int j = 0; j < WFN; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        *reinterpret_cast<f32x4*>(strip + (lane & 31) * SS + j * 32 + 8 * q + 4 * (lane >> 5)) =
            f32x4{acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]};
    // (a wave's strip is its own: its LDS accesses are in order)
    if (wide) {  // 16 lanes a row, 4 columns a lane
#pragma unroll
      for (int it = 0; it < 8; ++it) {
        const int r = it * 4 + (lane >> 4), c = (lane & 15) * 4;
        const int m = m0 + wm * (WBM / 2) + i * 32 + r, n = n0 + wn * (WBN / 2) + c;
        f32x4 v = *reinterpret_cast<const f32x4*>(strip + r * SS + c);
        if (m < st.M && n < st.N) {
          f32x4* dst = reinterpret_cast<f32x4*>(reinterpret_cast<float*>(out) + (long long)m * st.N + n);
          if (stream) {
            asm volatile("" ::: "memory");
            __builtin_nontemporal_store(v, dst);
            asm volatile("" ::: "memory");
          } else {
            if (add) v += *dst;
            *dst = v;
          }
        }
      }
    } else {
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
          uint16_t* dst = reinterpret_cast<uint16_t*>(out) + (long long)m * st.N + n;
          if (stream) {
            asm volatile("" ::: "memory");
            store8_nt(dst, v);
            asm volatile("" ::: "memory");
          } else {
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
}

// dw[e] (+)= the sums of e's parts, ascending, for the experts that were cut (blockIdx.y: which of them; the last:
// the router).  8 elements a thread, the stacks' elements one after the other.
__global__ __launch_bounds__(256) void wgrad_multi_sum_kernel(const MultiArgs p) {
  const int lane = lane_id();
  int e = 0, parts = p.r_slices, slot = 0;
  const bool router = p.r_slices > 1 && blockIdx.y == gridDim.y - 1;
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
  L = (L + 63) / 64 * 64;
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
    d.n_tiles = tiles_n(m.N), d.tiles = tiles_m(m.M) * d.n_tiles, d.per_n = 1.f / d.n_tiles;
    d.out_f32 = m.dtype == MOE_DT_F32, d.accumulate = m.accumulate;
  };
  for (int i = 0; i < n_stacks; ++i) {
    fill(a.s[i], stacks[i]);
    a.tiles += a.s[i].tiles;
    if (const MoeWgradStack& m = stacks[i]; m.row_at) {  // (the same of all that have one)
      if (!moe_rows_from_ok(m.from_rows, m.N)) return MOE_ERR_LIMIT;
      a.s[i].from = 1;
      a.row_at = m.row_at, a.from_bytes = m.from_rows * m.N * 2;
    }
  }
  int64_t bytes = 0;
  for (int i = 0; i < n_stacks; ++i) bytes += E * stacks[i].M * stacks[i].N * (a.s[i].out_f32 ? 4 : 2);
  a.streaming = bytes >= MOE_STREAMED_RESULTS;
  a.n_stacks = n_stacks;
  a.offs = offs;
  a.E = (int)E;
  // (from the shapes alone, whichever stacks are wanted: the room for the partial sums was made for it)
  a.L = n_stacks ? (int)segment_rows(R, H, I) : 1;
  a.many = a.L / 2;
  if (T <= a.L) a.L = (int)(R > 1 ? R : 1);  // (no expert has more rows than there are tokens: nothing to cut)
  a.T = (int)T;
  if (router) {
    fill(a.router, *router);
    a.r_rows = (int)router_rows;
    a.r_slices = (int)router_slices;
    // (one slice is written straight to its result, which may have fewer rows than the padded product, and is as long as
    // any expert's jobs)
    a.r_first = router_slices == 1;
    if (router_slices == 1) a.router.M = (int)E;
  }
  a.each = a.tiles > 0 ? (a.tiles + 7) / 8 : 1, a.per_each = 1.f / a.each;
  a.r_each = (a.r_slices * a.router.tiles + 7) / 8, a.r_per_tiles = a.router.tiles ? 1.f / a.router.tiles : 0.f;
  const long long segs = n_stacks ? (R > a.L ? R / a.L : 0) + E : 0;
  const long long e_each = n_stacks ? segs * a.each : 0, jobs = 8 * (e_each + (long long)a.r_each);
  if (jobs <= 0) return 0;
  if (jobs > 0x7fffffffll) return MOE_ERR_LIMIT;
  a.e_each = (int)e_each;
  if (a.row_at) hipLaunchKernelGGL(wgrad_multi_kernel<true>, dim3((unsigned)jobs), dim3(WNT), 0, s, a);
  else hipLaunchKernelGGL(wgrad_multi_kernel<false>, dim3((unsigned)jobs), dim3(WNT), 0, s, a);
  const long long cut = n_stacks && R > a.L ? R / a.L : 0;  // experts of more than L rows, at most
  const bool sliced = router && router_slices > 1;
  const long long ys = (cut < E ? cut : E) + (sliced ? 1 : 0);
  if (ys > 0) {
    long long n8 = 0;
    for (int i = 0; i < n_stacks; ++i) n8 += (long long)a.s[i].M * a.s[i].N / 8;
    const long long nr = sliced ? (long long)a.router.M * a.router.N / 8 : 0;
    if (nr > n8) n8 = nr;
    long long bx = (n8 + 255) / 256;
    if (bx > 2048) bx = 2048;
    hipLaunchKernelGGL(wgrad_multi_sum_kernel, dim3((unsigned)bx, (unsigned)ys), dim3(256), 0, s, a);
  }
  return moe_launch_status();
}
