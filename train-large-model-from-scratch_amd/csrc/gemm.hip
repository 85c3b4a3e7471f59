// Grouped (per-expert, ragged) bf16 GEMMs on the gfx950 matrix cores.
//
// One kernel template covers the five products of the expert FFN and its backward.  All of
// them are   C[rows, cols] = sum_k A[rows, k] * B[cols, k]   computed per expert with
// v_mfma_f32_32x32x16_bf16 (fp32 accumulation); they differ in which dimension is ragged,
// in how the operands lie in memory, and in the epilogue:
//
//   GATEUP        rows = expert's tokens, k = H.  A = xp [R,H]; B = W1 and W3 [E,I,H] (two
//                 accumulator sets share every A fragment); epilogue act = silu(g)*u.
//   DOWN          rows = tokens, k = I.  A = act [R,I]; B = W2 [E,H,I].
//   DGRAD_DOWN    rows = tokens, k = H.  A = dy [R,H]; B = W2 [E,H,I] read as [k][col];
//                 epilogue dg = dact*u*silu'(g), du = dact*silu(g).
//   DGRAD_GATEUP  rows = tokens, k runs over two segments of I.  A = dg | du [R,I];
//                 B = W1 | W3 [E,I,H] read as [k][col].
//   WGRAD         k = expert's tokens (ragged).  A = a [R,M] and B = b [R,N], both read as
//                 [k][row]; C = dw[e] [M,N].
//
// Memory plan.  A workgroup owns one BM x BN output tile.  A and B tiles of depth BK travel
// HBM -> registers (buffer loads whose hardware bounds check returns zero past the end of
// the expert's rows, so ragged tails cost no instructions) -> LDS (two stages) -> MFMA
// operand fragments.  The loop is software-pipelined: while the MFMAs of k-step s run, the
// fragments of step s+1 are read from LDS, the tile for iteration t+1 is written to the
// other LDS stage and the tile for iteration t+2 is requested from HBM.  There is one
// workgroup barrier per iteration, placed before the last k-step so that the first
// fragment reads of the next stage hide behind that step's MFMAs.
// Operands that are k-contiguous in memory are kept k-contiguous in LDS (16-byte fragment
// reads, rows padded by 16 bytes against bank conflicts); operands that are not are kept
// as they lie in memory and read through the transposing LDS read of gfx950.
// Workgroups are numbered so that each XCD (own L2) works on a contiguous range of tiles,
// i.e. on its own experts' weights.
#include "row_ring.h"
#include "tile_ops.h"

namespace {

template <int BM_, int BN_, int BK_, int WM_, int WN_>
struct TileCfg {
  static constexpr int BM = BM_, BN = BN_, BK = BK_, WM = WM_, WN = WN_;
  static constexpr int NT = WM * WN * MOE_WAVE;
  static constexpr int WTM = BM / WM, WTN = BN / WN;
  static constexpr int FM = WTM / 32, FN = WTN / 32;
  static constexpr int KS = BK / 16;
  // workgroups meant to share a CU (their LDS footprints must fit together in 160 KB)
  static constexpr int WGS_PER_CU = (NT >= 512) ? 1 : 2;
  static constexpr int WAVES_PER_SIMD = NT / 256 * WGS_PER_CU;
  static_assert(WTM % 32 == 0 && WTN % 32 == 0 && BK % 32 == 0, "tile shape");
};

template <int MODE, typename Cfg>
constexpr int lds_bytes() {
  constexpr bool a_outer = (MODE == WGRAD);
  constexpr bool b_outer = (MODE == DGRAD_DOWN || MODE == DGRAD_GATEUP || MODE == WGRAD);
  constexpr int a = a_outer ? OpOuter<Cfg::BM, Cfg::BK, Cfg::NT>::LDS_ELEMS : OpInner<Cfg::BM, Cfg::BK, Cfg::NT>::LDS_ELEMS;
  constexpr int b = b_outer ? OpOuter<Cfg::BN, Cfg::BK, Cfg::NT>::LDS_ELEMS : OpInner<Cfg::BN, Cfg::BK, Cfg::NT>::LDS_ELEMS;
  return 2 * (a + b) * 2;
}

constexpr int GEMM_MAX_E = 1024;  // per-expert tile prefix lives in LDS
constexpr int ROW_TILE = 256;     // rows of a tile of the row-ragged modes
constexpr int FROM_A = 1, FROM_B = 2;

// The expert of a row-tile slot, the last e with tile_start[e] <= slot (which skips those without rows), by a whole wave for a slot
// that its lanes share: a count over the lanes and one trip to LDS for 128 experts, where a search takes seven, one after the
// other.  (tile_start as number_tiles leaves it.  With number_tiles' single trip and the divisions by multiplication, us: a training pass of
// 4096 tokens, 8 of 128 experts, 1024 <-> 256, 419.1 -> 412.0; 8192, 2 of 8, 1024 <-> 512, 303.4 -> 300.1; a prefill of 1531, 8 of 64, 238.7 -> 237.2.)
__device__ __forceinline__ int expert_of(const int* tile_start, int slot, int E) {
  const int lane = lane_id();
  int n = 0;
  for (int b = 0; b < E; b += 2 * MOE_WAVE) {
    const int first = tile_start[b + lane], second = tile_start[b + MOE_WAVE + lane];
    n += __popcll(__ballot(first <= slot)) + __popcll(__ballot(second <= slot));
  }
  return n - 1;
}

// BLK (GATEUP and DGRAD_DOWN only): g and u, which nothing but the SwiGLU backward reads, are kept
// in a layout private to the library instead of as [R, I] rows: one 4 KB record per 32 x 32 block
// of a row tile, holding the block exactly as the matrix cores leave it in a wave's accumulators
// (see gu_block below).  The forward kernel then stores them straight from its registers and the
// backward kernel loads them straight into the layout it computes in: neither passes them
// through LDS.
//
// The kernel's tile walk: the tiles at positions t_next, t_next + t_step, .. below t_hi of the launch's tile
// list, or of `list` where one is given.  The rows of a row-ragged launch are numbered in tiles of UNIT rows; where
// the configuration's are half as high, a list entry is 2 * tile + half.  (tile_start and, there, offs: in LDS.)
// TO (DOWN and DGRAD_GATEUP only): the rows leave to where p.row_map says.  FROM (GATEUP and DGRAD_DOWN:
// A's rows; WGRAD: A's lines, FROM_A, or B's, FROM_B): they come from where p.row_from says.
template <int MODE, typename Cfg, typename OutT, bool BLK, int UNIT = ROW_TILE, bool TO = false, int FROM = 0>
__device__ __forceinline__ void walk_tiles(const GemmArgs& p, uint16_t* smem, const int* tile_start, const int* offs,
                                           const uint32_t* list, int t_next, const int t_hi, const int t_step) {
  static_assert(!BLK || MODE == GATEUP || MODE == DGRAD_DOWN, "only g and u have the blocked layout");
  static_assert(!FROM || MODE == GATEUP || MODE == DGRAD_DOWN || MODE == WGRAD, "only x and dy are read where the caller has them");
  constexpr bool ROWS_FROM = FROM && MODE != WGRAD, LINES_FROM = FROM && MODE == WGRAD, A_LINES = LINES_FROM && FROM == FROM_A;
  static_assert(!TO || MODE == DOWN || MODE == DGRAD_GATEUP, "only y and dxp are rows that somebody else has a place for");
  constexpr int BM = Cfg::BM, BN = Cfg::BN, BK = Cfg::BK, NT = Cfg::NT, KS = Cfg::KS;
  constexpr int FM = Cfg::FM, FN = Cfg::FN, WTM = Cfg::WTM, WTN = Cfg::WTN;
  constexpr bool DUAL = (MODE == GATEUP);
  constexpr int BNC = DUAL ? BN / 2 : BN;  // output columns covered by the tile
  constexpr bool A_OUTER = (MODE == WGRAD);
  constexpr bool B_OUTER = (MODE == DGRAD_DOWN || MODE == DGRAD_GATEUP || MODE == WGRAD);
  constexpr int NSEG = (MODE == DGRAD_GATEUP) ? 2 : 1;
  static_assert(!DUAL || (FN % 2 == 0), "dual mode needs an even number of column fragments");
  static_assert(KS % 2 == 0, "fragment double buffering assumes an even number of k-steps");

  using StA = typename std::conditional<A_OUTER, OpOuter<BM, BK, NT>, OpInner<BM, BK, NT>>::type;
  using StB = typename std::conditional<B_OUTER, OpOuter<BN, BK, NT>, OpInner<BN, BK, NT>>::type;
  using StBh = OpInner<BN / 2, BK, NT>;  // dual mode: the W1 half and the W3 half of the B tile
  static_assert(!DUAL || !B_OUTER, "dual mode stages k-contiguous weights");

  uint16_t* sA = smem;                       // [2][StA::LDS_ELEMS]
  uint16_t* sB = smem + 2 * StA::LDS_ELEMS;  // [2][StB::LDS_ELEMS]

  // (the wave's index is the same in all of its lanes: read it once so that everything derived
  // from it lives in scalar registers)
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int wm = wv / Cfg::WN, wn = wv % Cfg::WN;

  auto tile_at = [&](int pos) { return list ? (uint32_t)__builtin_amdgcn_readfirstlane((int)list[pos]) : (uint32_t)pos; };

  struct Tile {
    int e, row0, row_end, n0, m0;
    int block0;  // first of its 32-row blocks in the blocked g/u layout
    int Kseg, kt_per_seg, nkt;
    int kt0;  // k-tile it starts with (it goes round)
    bool need_mask;
    View vA0, vA1, vB0, vB1;
  };
  int lda, ldb;
  if constexpr (MODE == GATEUP || MODE == DOWN) lda = ldb = p.K;
  else if constexpr (MODE == WGRAD) { lda = p.M; ldb = p.N; }
  else { lda = p.ld_a ? p.ld_a : p.K; ldb = p.N; }

  // Fills `t` for tile slot `logical`; false when the slot lies past the last real tile.
  // Every lane computes the same thing from the same LDS words / scalar loads.
  auto locate = [&](uint32_t entry, Tile& t) -> bool {
    constexpr bool HALF = MODE != WGRAD && BM < UNIT;
    const int logical = (int)(HALF ? entry >> 1 : entry);
    const int slot = p.by_n_tiles(logical), n_tile = logical - slot * p.n_tiles;
    t.m0 = 0;
    if constexpr (MODE == WGRAD) {
      t.e = p.by_m_slots(slot);
      t.m0 = (slot - t.e * p.m_slots) * BM;
      t.row0 = offs[t.e];
      t.row_end = offs[t.e + 1];
    } else {
      if (slot >= tile_start[p.E]) return false;
      t.e = expert_of(tile_start, slot, p.E);
      const int off = __builtin_amdgcn_readfirstlane(offs[t.e]);
      int in_expert = (slot - __builtin_amdgcn_readfirstlane(tile_start[t.e])) * UNIT;
      if (HALF) in_expert += (int)(entry & 1) * BM;
      t.row0 = off + in_expert;
      t.row_end = __builtin_amdgcn_readfirstlane(offs[t.e + 1]);
      // (off / 32 + e grows from one expert to the next by at least the expert's blocks, whatever the tile height)
      t.block0 = off / 32 + t.e + in_expert / 32;
    }
    t.n0 = n_tile * BNC;
    t.Kseg = (MODE == WGRAD) ? (t.row_end - t.row0) : p.K;
    t.kt_per_seg = (t.Kseg + BK - 1) / BK;
    t.nkt = t.kt_per_seg * NSEG;
    // k-contiguous operands whose contraction length is not a multiple of BK need their
    // last k-tile cleared by hand (outside the static schedule)
    t.need_mask = ((t.Kseg % BK) != 0) && (!A_OUTER || !B_OUTER);
    const long long rows = t.row_end - t.row0;
    // With few rows an expert is bound by its weights, each line of which is read once.  Where their rows are a
    // multiple of 4 KB long, experts that sweep k side by side ask for the same lines of every page, which lie on few
    // of the memory channels; started at different k-tiles they do not (all tiles of an expert at the same one, so
    // that they go on sharing the operands in L2).  Gate/up of 64 experts, 2048 <-> 1024, again and again on the same
    // rows, rows per expert and us: 16, 128 -> 94; 64, 130 -> 100; 128, 138 -> 118; 191, 149 -> 141; 256, 186 -> 185.
    // The whole forward: 100 / 257 / 1000 / 1531 / 2600 tokens (12 to 325 rows an expert) 198 -> 185, 213 -> 188, 237 ->
    // 218, 269 -> 264, 389 -> 388; above that within 0.6 % either way.  16 experts, 4096 <-> 1536: 64 rows 168 -> 158, 175
    // rows 196 -> 195.  With rows of 2 KB there is nothing to gain.
    t.kt0 = 0;
    if constexpr (MODE == GATEUP || MODE == DOWN) {
      if (p.K % 2048 == 0) t.kt0 = (t.e * 13) & 31;  // (32 k-tiles to 4 KB)
    }
    if constexpr (MODE == GATEUP) {
      t.vA0 = ROWS_FROM ? View{p.A0, p.from_bytes} : make_view(p.A0 + (long long)t.row0 * lda, rows * lda);
      const long long wofs = ((long long)t.e * p.N + t.n0) * p.K;
      const long long wvalid = (long long)(p.N - t.n0) * p.K;
      t.vB0 = make_view(p.B0 + wofs, wvalid);
      t.vB1 = make_view(p.B1 + wofs, wvalid);
    } else if constexpr (MODE == DOWN) {
      t.vA0 = make_view(p.A0 + (long long)t.row0 * lda, rows * lda);
      t.vB0 = make_view(p.B0 + ((long long)t.e * p.N + t.n0) * p.K, (long long)(p.N - t.n0) * p.K);
    } else if constexpr (MODE == DGRAD_DOWN || MODE == DGRAD_GATEUP) {
      // A = dy [R,K] (or dg|du [R,K]); B = W[e] as [K][N]
      t.vA0 = ROWS_FROM ? View{p.A0, p.from_bytes} : make_view(p.A0 + (long long)t.row0 * lda, rows * lda);
      t.vB0 = make_view(p.B0 + (long long)t.e * p.K * p.N + t.n0, (long long)p.K * p.N - t.n0);
      if constexpr (MODE == DGRAD_GATEUP) {
        t.vA1 = make_view(p.A1 + (long long)t.row0 * lda, rows * lda);
        t.vB1 = make_view(p.B1 + (long long)t.e * p.K * p.N + t.n0, (long long)p.K * p.N - t.n0);
      }
    } else {  // WGRAD: A = a [R,M] as [k][m]; B = b [R,N] as [k][n]; k = rows of expert e
      t.vA0 = A_LINES ? View{p.A0 + t.m0, p.from_bytes - t.m0 * 2} : make_view(p.A0 + (long long)t.row0 * lda + t.m0, rows * lda - t.m0);
      t.vB0 = LINES_FROM && !A_LINES ? View{p.B0 + t.n0, p.from_bytes - t.n0 * 2}
                         : make_view(p.B0 + (long long)t.row0 * ldb + t.n0, rows * ldb - t.n0);
    }
    return true;
  };

  // ---- loader addressing (the same for every tile) and staging registers
  StA opA;
  StB opB;
  StBh opB0, opB1;
  opA.init(lda);
  if constexpr (DUAL) {
    opB0.init(ldb);
    opB1.init(ldb);
  } else {
    opB.init(ldb);
  }
  // (FROM) A lane has the place of one of the rows that its wave requests: asked for a tile ahead, worked out and dealt to the lanes
  // that request the row where the first k-tile of its tile is asked for.
  int row_from = 0;
  auto ask_rows = [&](const Tile& t) {
    if constexpr (ROWS_FROM) {
      const int r = t.row0 + StA::own_row(wv, lane);
      row_from = r < t.row_end ? p.row_from[r] : -1;
    }
  };
  auto set_rows = [&]() {
    if constexpr (ROWS_FROM) opA.set_rows(row_from < 0 ? NO_ROW : (uint32_t)p.by_k(row_from) * (uint32_t)(lda * 2));
  };
  // (WGRAD: the lines of a k-tile, asked for while the k-tile before is requested.  `lines_left`: how many of them the expert has.)
  int lines_left = 0;
  const auto own_line = [&]() {
    if constexpr (A_LINES) return StA::own_line(wv, lane);
    else if constexpr (LINES_FROM) return StB::own_line(wv, lane);
    else return 0;
  };
  auto ask_lines = [&](int first, int end) {
    if constexpr (LINES_FROM) {
      lines_left = end - first;
      const __amdgpu_buffer_rsrc_t rs =
          __builtin_amdgcn_make_buffer_rsrc((void*)(p.row_from + first), 0, lines_left > 0 ? lines_left * 4 : 0, 0x00020000);
      row_from = __builtin_amdgcn_raw_buffer_load_b32(rs, own_line() * 4, 0, 0);
    }
  };
  auto set_lines = [&]() {
    if constexpr (LINES_FROM) {
      const uint32_t at = own_line() < lines_left ? (uint32_t)p.by_k(row_from) * (uint32_t)((A_LINES ? lda : ldb) * 2) : NO_ROW;
      if constexpr (A_LINES) opA.set_lines(at);
      else opB.set_lines(at);
    }
  };
  // One set of registers carries a k-tile from HBM to LDS: it is requested one iteration
  // before it is written to LDS, which is what hides the latency of a load that misses L2.
  constexpr int CHA = StA::CH, CHB = DUAL ? StBh::CH : StB::CH;
  constexpr int NCH = CHA + (DUAL ? 2 : 1) * CHB;  // 16-byte chunks per thread per k-tile
  struct Stage {
    u32x4 v[NCH];
  };
  Stage stg;
  // Where a k-tile lies: the windows of the operands from it on (DUAL: three of them).
  constexpr int NOP = DUAL ? 3 : 2;
  struct TileSrc {
    Window w[NOP];
    int k_left;
  };
  auto k_of = [&](const Tile& t, int kt) {  // (of its segment)
    if constexpr (MODE == GATEUP || MODE == DOWN) {
      const int at = kt + t.kt0;
      return (at >= t.nkt ? at - t.nkt : at) * BK;
    } else {
      return (NSEG == 2 && kt >= t.kt_per_seg ? kt - t.kt_per_seg : kt) * BK;
    }
  };
  auto operand_src = [&](const Tile& t, int kt, int op) {
    const int k0 = k_of(t, kt);
    const bool second = NSEG == 2 && kt >= t.kt_per_seg;
    if (op == 0) return window(second ? t.vA1 : t.vA0, A_LINES ? 0 : StA::k_bytes(k0, lda));
    if constexpr (DUAL) return window(op == 1 ? t.vB0 : t.vB1, StBh::k_bytes(k0, ldb));
    else return window(second ? t.vB1 : t.vB0, LINES_FROM && !A_LINES ? 0 : StB::k_bytes(k0, ldb));
  };
  auto tile_src = [&](const Tile& t, int kt) {
    TileSrc ts;
#pragma unroll
    for (int op = 0; op < NOP; ++op) ts.w[op] = operand_src(t, kt, op);
    ts.k_left = t.Kseg - k_of(t, kt);
    return ts;
  };
  constexpr auto operand_of = [](int c) { return c < CHA ? 0 : DUAL && c >= CHA + CHB ? 2 : 1; };  // a chunk's
  auto load_chunk = [&](int c, Stage& st, const TileSrc& ts) {
    const __amdgpu_buffer_rsrc_t rs = ts.w[operand_of(c)].rsrc();
    if (c < CHA) st.v[c] = opA.load_one(c, rs);
    else if constexpr (DUAL) {
      if (c < CHA + CHB) st.v[c] = opB0.load_one(c - CHA, rs);
      else st.v[c] = opB1.load_one(c - CHA - CHB, rs);
    } else {
      st.v[c] = opB.load_one(c - CHA, rs);
    }
  };
  auto clear_past_k = [&](int c, Stage& st, int k_left) {
    bool past;
    if (c < CHA) past = opA.past_k(k_left);
    else if constexpr (DUAL) past = opB0.past_k(k_left);
    else past = opB.past_k(k_left);
    if (past) st.v[c] = u32x4{0, 0, 0, 0};
  };
  auto store_chunk = [&](int c, const Stage& st, int buf) {
    if (c < CHA) opA.store_one(c, sA + buf * StA::LDS_ELEMS, st.v[c]);
    else if constexpr (DUAL) {
      if (c < CHA + CHB) opB0.store_one(c - CHA, sB + buf * StB::LDS_ELEMS, st.v[c]);
      else opB1.store_one(c - CHA - CHB, sB + buf * StB::LDS_ELEMS + StBh::LDS_ELEMS, st.v[c]);
    } else {
      opB.store_one(c - CHA, sB + buf * StB::LDS_ELEMS, st.v[c]);
    }
  };
  auto load_tile = [&](const Tile& t, int kt, Stage& st) {
    const TileSrc ts = tile_src(t, kt);
    set_lines();
#pragma unroll
    for (int c = 0; c < NCH; ++c) load_chunk(c, st, ts);
    if (t.need_mask && ts.k_left < BK) {
#pragma unroll
      for (int c = 0; c < NCH; ++c) clear_past_k(c, st, ts.k_left);
    }
  };
  auto store_tile = [&](const Stage& st, int buf) {
#pragma unroll
    for (int c = 0; c < NCH; ++c) store_chunk(c, st, buf);
  };
  using std::integral_constant;
  const int a_off = StA::lane_off(lane), b_off = StB::lane_off(lane);
  // LDS row of column-fragment jn for this wave
  auto bfrag_row = [&](int jn) {
    if constexpr (DUAL)
      return (jn < FN / 2) ? wn * (WTN / 2) + jn * 32 : BN / 2 + wn * (WTN / 2) + (jn - FN / 2) * 32;
    else
      return wn * WTN + jn * 32;
  };

  struct Frags {
    bf16x8 a[FM];
    bf16x8 b[FN];
  };
  f32x16 acc[FM][FN];
  Frags fr[2];
  constexpr int NMMA = FM * FN;  // MFMAs per k-step
  constexpr int NFR = FM + FN;   // fragment reads per k-step
  // u-th fragment read of a k-step: a0, b0 .. b(FN-1), a1 .. a(FM-1) -- the order in which
  // the MFMAs (row-major over the fragment grid) first need them
  auto f_read_one = [&](int u, int buf, int ks, Frags& f) {
    const uint16_t* a_lds = sA + buf * StA::LDS_ELEMS;
    const uint16_t* b_lds = sB + buf * StB::LDS_ELEMS;
    if (u == 0) f.a[0] = StA::frag(a_lds, a_off, wm * WTM, ks);
    else if (u <= FN) f.b[u - 1] = StB::frag(b_lds, b_off, bfrag_row(u - 1), ks);
    else f.a[u - FN] = StA::frag(a_lds, a_off, wm * WTM + (u - FN) * 32, ks);
  };
  auto mma_one = [&](int n, const Frags& f) {
    // boustrophedon over the fragment grid: consecutive MFMAs share one operand register (about
    // half a percent on every mode, measured); operands swapped: acc holds the transposed block
    const int i = n / FN, j = (i & 1) ? FN - 1 - n % FN : n % FN;
    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f.b[j], f.a[i], acc[i][j], 0, 0, 0);
  };
  auto f_read_all = [&](int buf, int ks, Frags& f) {
#pragma unroll
    for (int u = 0; u < NFR; ++u) f_read_one(u, buf, ks, f);
  };
  auto mma_all = [&](const Frags& f) {
#pragma unroll
    for (int n = 0; n < NMMA; ++n) mma_one(n, f);
  };

  // ---- one steady-state iteration, written out instruction by instruction: each MFMA is
  // followed by at most one chunk hand-over (registers -> LDS, then the same registers are
  // re-requested from HBM for the tile after next) and one fragment read, and a scheduling
  // fence after each slot keeps the compiler from clumping them, so a wave issues its
  // memory traffic in the shadow of its own MFMAs.
  //   phases 0..KS-2  MFMAs of k-step s | chunks of tile kt+1 -> other LDS stage, chunks of
  //                   tile kt+2 requested | fragments of step s+1 read
  //   last phase      barrier (stage kt fully read, stage kt+1 fully written) | MFMAs of the
  //                   last step | first fragment reads of stage kt+1 hide behind them
  // Where tile kt+3 lies is worked out behind the last request for an operand of kt+2, between two products: in front
  // of the first one the forty scalar instructions, with six 64-bit comparisons in the vector unit among them, held up both waves of a
  // SIMD, which come from the same barrier.  Whole passes, us, in turn on one GPU: 1531 tokens, 8 of 64 experts, forward, 265.4 -> 262.6; 8192, 2 of
  // 8, 1024 <-> 512, 317.7 -> 313.7; smaller ones 1.00 to 1.02; 16384 tokens of 64, where power is the bound, equal.
  auto body = [&](auto par_c, const Tile& t, int kt, TileSrc& ts, auto&& lines_behind) {
    constexpr int buf = decltype(par_c)::value;  // LDS stage of k-tile kt == parity of kt
    Stage& st = stg;                             // holds k-tile kt+1, refilled with kt+2, which lies at `ts`
    constexpr int NSLOT = (KS - 1) * NMMA;  // MFMA slots before the barrier
#pragma unroll
    for (int ks = 0; ks < KS - 1; ++ks) {
#pragma unroll
      for (int n = 0; n < NMMA; ++n) {
        mma_one(n, fr[ks & 1]);
        const int slot = ks * NMMA + n;
#pragma unroll
        for (int c = 0; c < NCH; ++c) {
          if (c * NSLOT / NCH == slot) {
            store_chunk(c, st, buf ^ 1);
            if (LINES_FROM && c == 0) {
              set_lines();
              lines_behind(kt + 2);
            }
            load_chunk(c, st, ts);
            if (c + 1 == NCH || operand_of(c + 1) != operand_of(c)) {
              Window& w = ts.w[operand_of(c)];
              int ahead = kt + 3;
              asm volatile("" : "+s"(ahead));  // (else most of it moves up in front of the first product all the same)
              w = operand_src(t, ahead, operand_of(c));
              w.stay_here();
            }
          }
        }
        if (n < NFR) f_read_one(n, buf, ks + 1, fr[(ks + 1) & 1]);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    lds_barrier();
#pragma unroll
    for (int n = 0; n < NMMA; ++n) {
      mma_one(n, fr[(KS - 1) & 1]);
      if (n < NFR) f_read_one(n, buf ^ 1, 0, fr[0]);
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  // ---- epilogue pieces.  The MFMAs were issued with the operands swapped (B fragment
  // first), so acc[i][j] holds the transposed 32x32 block: lane l owns output row (l % 32)
  // and, for q = 0..3, the four consecutive columns 8*q + 4*(l/32) .. +3 in
  // acc[i][j][4*q .. 4*q+3].  Results leave through LDS: each wave owns a strip of 32 rows
  // x its output columns, writes its accumulators there four columns at a time and reads
  // the strip back row-wise, so that global memory sees 16-byte stores that cover whole
  // 128-byte lines.  The strips live in the (then idle) operand stages, one region per
  // wave, so only wave-local ordering is needed between the two barriers that fence the
  // epilogue off from the main loops before and after it.
  constexpr int WTNC = DUAL ? WTN / 2 : WTN;  // output columns per wave
  constexpr int FNC = DUAL ? FN / 2 : FN;
  constexpr int OSZ = (MODE == WGRAD) ? (int)sizeof(OutT) : 2;
  constexpr int SSTRIDE = WTNC * OSZ + 16;  // bytes per strip row (16 bytes of padding)
  constexpr int SBYTES = 32 * SSTRIDE;
  constexpr int NSTRIP = (MODE == GATEUP) ? (BLK ? 1 : 3) : (MODE == DGRAD_DOWN ? 2 : 1);
  constexpr int CPRO = WTNC * OSZ / 16;  // 16-byte chunks per strip row
  constexpr int RPI = 64 / CPRO;         // rows covered by one wave-wide 16-byte access
  static_assert(64 % CPRO == 0 && 32 % RPI == 0, "strip shape");
  // Where they fit, the strips take one LDS stage only (half of the waves in its A part, half in its B part): the
  // one that the tile's last k-tile was read from.  The k-tiles of the next tile then follow this one's without a
  // break: its first is asked for in the last but one iteration and moves to the other stage in the last one, which
  // asks for its second.  A unit answers its loads and stores in order: loads sent between the stores of the strips
  // wait behind them, and the stores behind the loads' trip to memory (65536 rows of 64 experts, 2048 <-> 1024, with the next
  // tile's loads in the epilogue and without: an epilogue takes half as long, half of that comes back as a slower start of the next
  // loop, and power takes its share: gate/up 528 -> 518 us, down 282 -> 272, weight gradients 786 -> 777, in fp32 925 -> 893; 32768
  // rows of 128, 1024 <-> 256: down 36.4 -> 35.1, dgrad-gate/up 53.4 -> 51.9).
  // (the SwiGLU-backward epilogue needs the staging registers' room for its g/u rows: the next tile's first k-tile
  // moves to LDS all the same, and its second is asked for during the last strip, when that room is free.  With the first
  // strip's g and u on their way behind the last products, dgrad-down of 131072 rows of 64 experts, 2048 <-> 1024, 610 -> 596 us;
  // 65536 rows 333 -> 326; 32768 of 128, 1024 <-> 256, 44.7 -> 43.1; 30000 of 64, 512 <-> 1024, 71.4 -> 68.2)
  constexpr bool EARLY_REQUEST = (MODE != DGRAD_DOWN);
  constexpr int HALF_WAVES = Cfg::WM * Cfg::WN / 2;
  constexpr bool STREAM = NSTRIP * SBYTES * HALF_WAVES <= StA::LDS_ELEMS * 2 &&
                          NSTRIP * SBYTES * HALF_WAVES <= StB::LDS_ELEMS * 2;
  static_assert(NSTRIP * SBYTES * Cfg::WM * Cfg::WN <= lds_bytes<MODE, Cfg>(), "strips fit in the stages");
  const auto strip_in = [&](int stage) {
    return STREAM ? reinterpret_cast<char*>(wv < HALF_WAVES ? sA + stage * StA::LDS_ELEMS : sB + stage * StB::LDS_ELEMS) +
                        (wv % HALF_WAVES) * (NSTRIP * SBYTES)
                  : reinterpret_cast<char*>(smem) + wv * (NSTRIP * SBYTES);
  };
  char* strip = strip_in(0);
  const int ldc = p.ld_c ? p.ld_c : p.N;  // outputs
  const int ldx = p.N;                    // epilogue inputs (g, u)
  // The accumulators of a strip are cleared for the next tile as soon as they are in LDS: the
  // moves fill the waits of the strip's LDS and global traffic instead of a slot before the
  // next main loop.
  auto zero_row = [&](int i) {
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;
  };
  // Blocked g/u (BLK): record of the 32 x 32 block (row block rb of the tile, column
  // block cb = column / 32), GU_BLOCK_BYTES each: [g: q0q1 of lanes 0..63 | g: q2q3 | u: q0q1 |
  // u: q2q3], 16 bytes per lane and part, where lane l of the wave that owns the block holds row
  // l % 32 and columns 8*q + 4*(l/32) .. +3 of it for q = 0..3 (the accumulator layout above).
  // A wave-wide 16-byte access to one part covers 1 KB of consecutive addresses.  Row blocks are
  // numbered expert by expert from the offsets alone (Tile::block0), so that the forward and the backward
  // kernel agree on them whatever tiles either of them takes.
  constexpr int GU_BLOCK_BYTES = 4096;
  const int n_cb = (p.N + 31) / 32;
  auto gu_block = [&](const void* base, const Tile& t, int rb, int cb, int ln) {
    return (char*)base + (((long long)t.block0 + rb) * n_cb + cb) * GU_BLOCK_BYTES + ln * 16;
  };
  // (BLK) the two 16-byte parts of g and of u for each of the strip's column blocks
  struct BlkRegs {
    u32x4 g[FNC][2], u[FNC][2];
  };
  auto request_block = [&](const Tile& t, int i, int j, BlkRegs& b, int ln) {
    const int cb = (t.n0 + wn * WTNC + j * 32) / 32;
    const u32x4 zero = u32x4{0, 0, 0, 0};
    b.g[j][0] = b.g[j][1] = b.u[j][0] = b.u[j][1] = zero;
    if (t.row0 + wm * WTM + i * 32 < t.row_end && cb < n_cb) {
      const u32x4* rec = reinterpret_cast<const u32x4*>(gu_block(p.X0, t, wm * FM + i, cb, ln));
      // (read exactly once: streamed past the L2 lines the operand panels live in)
      b.g[j][0] = __builtin_nontemporal_load(rec + 0);
      b.g[j][1] = __builtin_nontemporal_load(rec + 64);
      b.u[j][0] = __builtin_nontemporal_load(rec + 128);
      b.u[j][1] = __builtin_nontemporal_load(rec + 192);
    }
  };
  BlkRegs blk_in;
  // (TO) where the wave's rows go, a lane a row: asked for at the top of the tile, there when its contraction is done
  int row_to[TO ? (WTM + MOE_WAVE - 1) / MOE_WAVE : 1];
  // `last_rows_in` runs once the SwiGLU-backward epilogue has taken the last g/u rows out of their registers
  auto epilogue = [&](const Tile& t, auto&& last_rows_in) {
    // Every per-lane address of the epilogue is derived from this copy of the lane index, which
    // the empty asm makes opaque: the compiler then recomputes them here, a handful of integer
    // operations per tile, instead of hoisting them out of the tile loop and holding a dozen
    // registers through the main loop for them.
    int lane_e = lane;
    asm volatile("" : "+v"(lane_e));
    const int l32 = lane_e & 31, lh = lane_e >> 5;
    const int row_in_pass = lane_e / CPRO, chunk_in_row = lane_e % CPRO;
    auto acc_ptr = [&](int plane, int j, int q) {  // 4 consecutive columns in accumulator layout
      return strip + plane * SBYTES + l32 * SSTRIDE + (j * 32 + 8 * q + 4 * lh) * OSZ;
    };
    auto put4 = [&](int plane, int j, int q, float a, float b, float c, float d) {
      if constexpr (OSZ == 4) *reinterpret_cast<f32x4*>(acc_ptr(plane, j, q)) = f32x4{a, b, c, d};
      else *reinterpret_cast<u32x2*>(acc_ptr(plane, j, q)) = u32x2{pack_bf16x2(a, b), pack_bf16x2(c, d)};
    };
    const int col_w0 = t.n0 + wn * WTNC;  // first output column of the wave
    char* C0 = (char*)p.C0;
    int m_shift = 0;  // WGRAD with two results: the rows of the second one start at m_split
    int m_lim = p.M;
    if constexpr (MODE == WGRAD) {
      if (p.m_split > 0) {
        if (t.m0 >= p.m_split) {
          C0 = (char*)p.C1 + (long long)t.e * (p.M - p.m_split) * p.N * OSZ;
          m_shift = p.m_split;
        } else {
          C0 += (long long)t.e * p.m_split * p.N * OSZ;
          m_lim = p.m_split;
        }
      } else {
        C0 += (long long)t.e * p.M * p.N * OSZ;
      }
    }
    const int row_lim = (MODE == WGRAD) ? m_lim : t.row_end;
    // row-wise pass over a strip: lane handles chunk (lane % CPRO) of row it*RPI + lane/CPRO
    auto store_rows = [&](int plane, int i, char* gbase /* element (0,0) of the output */) {
      const int rbase = (MODE == WGRAD ? t.m0 : t.row0) + wm * WTM + i * 32;
#pragma unroll
      for (int it = 0; it < 32 / RPI; ++it) {
        const int rr = it * RPI + row_in_pass, ch = chunk_in_row;
        const u32x4 v = *reinterpret_cast<const u32x4*>(strip + plane * SBYTES + rr * SSTRIDE + ch * 16);
        const int r = rbase + rr, c = col_w0 + ch * (16 / OSZ);
        int to = r - m_shift;
        if constexpr (TO) to = __shfl(row_to[i / 2], (i & 1) * 32 + rr, MOE_WAVE);
        if (r < row_lim && c < p.N) {
          u32x4* dst = reinterpret_cast<u32x4*>(gbase + ((long long)to * ldc + c) * OSZ);
          if (MODE == WGRAD && p.accumulate) {
            const u32x4 o = *dst;
            if constexpr (OSZ == 4) {
              const f32x4 sum = __builtin_bit_cast(f32x4, v) + __builtin_bit_cast(f32x4, o);
              *dst = __builtin_bit_cast(u32x4, sum);
            } else {
              *dst = u32x4{pack_bf16x2(bf16lo(v[0]) + bf16lo(o[0]), bf16hi(v[0]) + bf16hi(o[0])),
                           pack_bf16x2(bf16lo(v[1]) + bf16lo(o[1]), bf16hi(v[1]) + bf16hi(o[1])),
                           pack_bf16x2(bf16lo(v[2]) + bf16lo(o[2]), bf16hi(v[2]) + bf16hi(o[2])),
                           pack_bf16x2(bf16lo(v[3]) + bf16lo(o[3]), bf16hi(v[3]) + bf16hi(o[3]))};
            }
          } else if (MODE == WGRAD && p.streaming) {
            asm volatile("" ::: "memory");  // (without the two fences this store and the next become one, an ordinary one)
            __builtin_nontemporal_store(v, dst);
            asm volatile("" ::: "memory");
          } else {
            *dst = v;
          }
        }
      }
    };
    // DGRAD_DOWN reads g and u in the accumulator layout too: their rows come in as whole
    // 128-byte lines into registers (requested one strip ahead), pass through the strip and
    // are overwritten in place by dg and du.
    struct RowRegs {
      u32x4 g[32 / RPI], u[32 / RPI];
    };
    auto request_rows = [&](int i, RowRegs& rr_) {
      const int rbase = t.row0 + wm * WTM + i * 32;
#pragma unroll
      for (int it = 0; it < 32 / RPI; ++it) {
        const int rr = it * RPI + row_in_pass, ch = chunk_in_row;
        const int r = rbase + rr, c = col_w0 + ch * (16 / OSZ);
        rr_.g[it] = u32x4{0, 0, 0, 0};
        rr_.u[it] = u32x4{0, 0, 0, 0};
        if (r < row_lim && c < p.N) {
          rr_.g[it] = *reinterpret_cast<const u32x4*>((const char*)p.X0 + ((long long)r * ldx + c) * OSZ);
          rr_.u[it] = *reinterpret_cast<const u32x4*>((const char*)p.X1 + ((long long)r * ldx + c) * OSZ);
        }
      }
    };
    auto rows_to_strip = [&](const RowRegs& rr_) {
#pragma unroll
      for (int it = 0; it < 32 / RPI; ++it) {
        const int rr = it * RPI + row_in_pass, ch = chunk_in_row;
        *reinterpret_cast<u32x4*>(strip + 0 * SBYTES + rr * SSTRIDE + ch * 16) = rr_.g[it];
        *reinterpret_cast<u32x4*>(strip + 1 * SBYTES + rr * SSTRIDE + ch * 16) = rr_.u[it];
      }
    };
    RowRegs rows_in;
    if constexpr (MODE == DGRAD_DOWN && !BLK) request_rows(0, rows_in);
#pragma unroll
    for (int i = 0; i < FM; ++i) {
      if constexpr (MODE == GATEUP) {
        // (BLK) blocks of a strip that starts past the end of the expert's rows are never read
        const bool strip_live = t.row0 + wm * WTM + i * 32 < t.row_end;
#pragma unroll
        for (int j = 0; j < FNC; ++j) {
          u32x2 gq[2], uq[2];
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            float g[4], u[4], a[4];
#pragma unroll
            for (int x = 0; x < 4; ++x) {
              g[x] = acc[i][j][4 * q + x];
              u[x] = acc[i][j + FNC][4 * q + x];
              a[x] = swiglu(g[x], u[x]);
            }
            put4(0, j, q, a[0], a[1], a[2], a[3]);
            if constexpr (BLK) {
              gq[q & 1] = u32x2{pack_bf16x2(g[0], g[1]), pack_bf16x2(g[2], g[3])};
              uq[q & 1] = u32x2{pack_bf16x2(u[0], u[1]), pack_bf16x2(u[2], u[3])};
              if (q & 1) {  // a 16-byte part of the record is complete: it leaves at once
                const int cb = (col_w0 + j * 32) / 32;
                if (p.C0 && strip_live && cb < n_cb) {
                  u32x4* rec = reinterpret_cast<u32x4*>(gu_block(p.C0, t, wm * FM + i, cb, lane_e));
                  // (written once, read by the backward pass much later: streaming stores)
                  __builtin_nontemporal_store(u32x4{gq[0][0], gq[0][1], gq[1][0], gq[1][1]}, rec + 64 * (q >> 1));
                  __builtin_nontemporal_store(u32x4{uq[0][0], uq[0][1], uq[1][0], uq[1][1]},
                                              rec + 128 + 64 * (q >> 1));
                }
              }
            } else if (p.C0) {
              put4(1, j, q, g[0], g[1], g[2], g[3]);
              put4(2, j, q, u[0], u[1], u[2], u[3]);
            }
          }
        }
        zero_row(i);
        store_rows(0, i, (char*)p.C2);
        if constexpr (!BLK) {
          if (p.C0) {
            store_rows(1, i, (char*)p.C0);
            store_rows(2, i, (char*)p.C1);
          }
        }
      } else if constexpr (MODE == DGRAD_DOWN && BLK) {
        // g and u arrive in the accumulator layout: nothing to rearrange.  The registers of column
        // block j are asked for the next strip's block as soon as this strip's block is computed.
        float rowdot = 0.f;
#pragma unroll
        for (int j = 0; j < FNC; ++j) {
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const u32x4 gv = blk_in.g[j][q >> 1], uv = blk_in.u[j][q >> 1];
            const uint32_t g01 = gv[2 * (q & 1)], g23 = gv[2 * (q & 1) + 1];
            const uint32_t u01 = uv[2 * (q & 1)], u23 = uv[2 * (q & 1) + 1];
            const float g[4] = {bf16lo(g01), bf16hi(g01), bf16lo(g23), bf16hi(g23)};
            const float u[4] = {bf16lo(u01), bf16hi(u01), bf16lo(u23), bf16hi(u23)};
            float dg[4], du[4];
#pragma unroll
            for (int x = 0; x < 4; ++x) swiglu_bwd(acc[i][j][4 * q + x], g[x], u[x], dg[x], du[x], rowdot);
            put4(0, j, q, dg[0], dg[1], dg[2], dg[3]);
            put4(1, j, q, du[0], du[1], du[2], du[3]);
            // (the running sum is wanted here, not at the end of the strip: left alone the compiler
            // may defer its chain of additions and keep every du and u alive for it)
            asm volatile("" : "+v"(rowdot));
          }
          __builtin_amdgcn_sched_barrier(0);  // (the loads must not move up: their registers are in use)
          if (i + 1 < FM) request_block(t, i + 1, j, blk_in, lane_e);
          __builtin_amdgcn_sched_barrier(0);
        }
        if (i + 1 == FM) last_rows_in();
        {
          rowdot += __shfl_xor(rowdot, 32, MOE_WAVE);
          const int r = t.row0 + wm * WTM + i * 32 + l32;
          if (lh == 0 && r < row_lim && p.C2)
            reinterpret_cast<float*>(p.C2)[(long long)((t.n0 / BNC) * Cfg::WN + wn) * p.R + r] = rowdot;
        }
        zero_row(i);
        store_rows(0, i, (char*)p.C0);
        store_rows(1, i, (char*)p.C1);
      } else if constexpr (MODE == DGRAD_DOWN) {
        rows_to_strip(rows_in);
        if (i + 1 < FM) request_rows(i + 1, rows_in);
        else last_rows_in();
        float rowdot = 0.f;  // this lane's share of <dact[row,:], act[row,:]>
#pragma unroll
        for (int j = 0; j < FNC; ++j)
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const u32x2 gw = *reinterpret_cast<const u32x2*>(acc_ptr(0, j, q));
            const u32x2 uw = *reinterpret_cast<const u32x2*>(acc_ptr(1, j, q));
            const float g[4] = {bf16lo(gw[0]), bf16hi(gw[0]), bf16lo(gw[1]), bf16hi(gw[1])};
            const float u[4] = {bf16lo(uw[0]), bf16hi(uw[0]), bf16lo(uw[1]), bf16hi(uw[1])};
            float dg[4], du[4];
#pragma unroll
            for (int x = 0; x < 4; ++x) swiglu_bwd(acc[i][j][4 * q + x], g[x], u[x], dg[x], du[x], rowdot);
            put4(0, j, q, dg[0], dg[1], dg[2], dg[3]);
            put4(1, j, q, du[0], du[1], du[2], du[3]);
            asm volatile("" : "+v"(rowdot));  // (summed here: see the blocked variant above)
          }
        {
          // One partial per 64-column block and row (block-major, so that a wave writes 32
          // consecutive floats): the row's sum over all blocks is
          // gate * <dy[token], y[row]>, i.e. what the gate's gradient needs, so that nobody
          // has to read y again.  Written, not accumulated: the caller adds the blocks up in
          // a fixed order.
          rowdot += __shfl_xor(rowdot, 32, MOE_WAVE);
          const int r = t.row0 + wm * WTM + i * 32 + l32;
          if (lh == 0 && r < row_lim && p.C2)
            reinterpret_cast<float*>(p.C2)[(long long)((t.n0 / BNC) * Cfg::WN + wn) * p.R + r] = rowdot;
        }
        zero_row(i);
        store_rows(0, i, (char*)p.C0);
        store_rows(1, i, (char*)p.C1);
      } else {
#pragma unroll
        for (int j = 0; j < FNC; ++j)
#pragma unroll
          for (int q = 0; q < 4; ++q)
            put4(0, j, q, acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]);
        zero_row(i);
        store_rows(0, i, C0);
      }
    }
  };

  // ---- the tile loop
  // At the top of the loop the first k-tile of `cur` has been asked for: with `staged` it sits in LDS stage s0 and the second
  // is on its way into the staging registers, else the first is.
  auto request_k = [&](const Tile& t, int kt) {
    if (kt < t.nkt) {
      load_tile(t, kt, stg);
    } else {
      // (nothing will be read from the staging registers: say so, or they stay alive through the
      // epilogue on account of this path)
#pragma unroll
      for (int c = 0; c < NCH; ++c) asm volatile("" : "=v"(stg.v[c]));
    }
  };
  auto request_first = [&](const Tile& t) {
    ask_lines(t.row0, t.row_end);
    request_k(t, 0);
    ask_lines(t.row0 + BK, t.row_end);
  };
  Tile cur;
  if (t_next >= t_hi || !locate(tile_at(t_next), cur)) return;
  ask_rows(cur);
  set_rows();
  request_first(cur);
  bool staged = false;
  int s0 = 0;           // the LDS stage of the tile's first k-tile; they alternate from there
#pragma unroll
  for (int i = 0; i < FM; ++i) zero_row(i);  // later tiles find them cleared by the epilogue
  for (;;) {
    // The last row tile of an expert is mostly short.  A wave whose rows all lie past its end
    // multiplies nothing: it only keeps moving operand chunks and meets the barriers (the
    // same ones in the same order as the waves that work), so that such a tile costs the
    // matrix pipe half of a full one.
    // The fragment registers carry nothing from one tile to the next.  The compiler cannot see that
    // (their first reads sit behind conditions it does not correlate with the loops that use them)
    // and would keep all of them alive through the epilogue; an empty asm that "writes" them ends
    // their live ranges here at no cost.
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
      for (int i = 0; i < FM; ++i) asm volatile("" : "=v"(fr[h].a[i]));
#pragma unroll
      for (int j = 0; j < FN; ++j) asm volatile("" : "=v"(fr[h].b[j]));
    }
    const bool idle =
        (MODE != WGRAD) && __builtin_amdgcn_readfirstlane((int)(wm * WTM >= cur.row_end - cur.row0)) != 0;
    // where the next tile lies is worked out now (a count over the lanes, a trip to LDS and some address
    // arithmetic), in the shadow of this tile's first MFMAs, not between the tiles
    Tile nxt;
    t_next += t_step;
    const bool more = t_next < t_hi && locate(tile_at(t_next), nxt);
    if (more) ask_rows(nxt);
    if constexpr (TO) {
#pragma unroll
      for (int h = 0; h < (WTM + MOE_WAVE - 1) / MOE_WAVE; ++h) {
        const int r = cur.row0 + wm * WTM + h * MOE_WAVE + lane;
        row_to[h] = r < cur.row_end ? p.row_map[r] : 0;
      }
    }
    const int nkt = cur.nkt;
    // the k-tiles of the next tile follow this one's.  (Lines from anywhere: unless this tile would request all of them, and the lines of
    // a tile behind it would have to be asked for, which is not known yet; the registers for asking at one place more are not there.)
    const bool stream = STREAM && more && nkt > 1 && nxt.nkt > (LINES_FROM ? 2 : 0);
    // the lines of the k-tile behind kt
    auto lines_behind = [&](int kt) {
      if constexpr (LINES_FROM) {
        const int next = kt + 1;
        const bool here = next < nkt;
        ask_lines(here ? cur.row0 + next * BK : stream ? nxt.row0 + (next - nkt) * BK : 0, here ? cur.row_end : stream ? nxt.row_end : 0);
      }
    };
    // the k-tile two behind kt
    auto request_ahead = [&](int kt) {
      if (kt + 2 < nkt) {
        load_tile(cur, kt + 2, stg);
        lines_behind(kt + 2);
      }
      else if (stream && kt + 2 - nkt < (EARLY_REQUEST ? nxt.nkt : 1)) {
        if (kt + 2 == nkt) set_rows();
        load_tile(nxt, kt + 2 - nkt, stg);
        lines_behind(kt + 2);
      }
    };
    if (nkt > 0) {
      if (!staged) {
        s0 = 0;
        store_tile(stg, 0);
        if (1 < nkt) {
          load_tile(cur, 1, stg);
          lines_behind(1);
        }
        lds_barrier();
      }
      if (!idle) f_read_all(s0, 0, fr[0]);
    }
    int kt = 0;
    if (idle) {
      for (; kt < nkt; ++kt) {
        if (kt + 1 < nkt || stream) {
          store_tile(stg, ((kt + s0) & 1) ^ 1);
          request_ahead(kt);
          lds_barrier();
        }
      }
    }
    // Steady iterations (two at a time: the stage index is a compile-time constant) request k-tile
    // kt+2 as it lies in memory.  The last k-tiles, and the iterations that request a k-tile with
    // columns past the end of a segment (to be cleared), take the loop around them: the same order of
    // events, conditions evaluated, no static schedule.  (Segments of 1416 and 568, 9999 rows of 12 experts, when any
    // tail sent every iteration there: gate/up 54.9 us, now 46.1; dgrad-gate/up 71.5, now 62.5.)
    auto request_blocks = [&]() {
      int ln = lane;
      asm volatile("" : "+v"(ln));
#pragma unroll
      for (int j = 0; j < FNC; ++j) request_block(cur, 0, j, blk_in, ln);
    };
    auto one = [&](int kt) {
      const int buf = (kt + s0) & 1;
      const bool has1 = kt + 1 < nkt;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        if (ks + 1 < KS) f_read_all(buf, ks + 1, fr[(ks + 1) & 1]);
        if (ks == 0 && (has1 || stream)) {
          store_tile(stg, buf ^ 1);
          request_ahead(kt);
        }
        if (ks == KS - 1 && (has1 || stream)) {
          lds_barrier();
          if (has1) f_read_all(buf ^ 1, 0, fr[0]);
        }
        mma_all(fr[ks & 1]);
      }
    };
    // The tile's last k-tile, behind whose products the first g and u are on their way, in the registers of the staging and
    // of the second set of fragments.
    auto last = [&](int kt) {
      const int buf = (kt + s0) & 1;
      if (stream) store_tile(stg, buf ^ 1);
      __builtin_amdgcn_sched_barrier(0);
      request_blocks();
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        if (ks > 0) f_read_all(buf, ks, fr[0]);
        if (ks == KS - 1 && stream) lds_barrier();
        mma_all(fr[0]);
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    constexpr bool PEEL = MODE == DGRAD_DOWN && BLK;
    const int looped = PEEL ? nkt - 1 : nkt;
    while (kt < looped) {
      int steady_end = nkt - 2;
      if (cur.need_mask) steady_end = (NSEG == 2 && kt + 2 < cur.kt_per_seg ? cur.kt_per_seg : nkt) - 3;
      if (!((kt + s0) & 1)) {
        TileSrc ts = tile_src(cur, kt + 2);
        for (; kt + 1 < steady_end; kt += 2) {
          body(integral_constant<int, 0>{}, cur, kt, ts, lines_behind);
          body(integral_constant<int, 1>{}, cur, kt + 1, ts, lines_behind);
        }
      }
      one(kt);
      ++kt;
    }
    if constexpr (PEEL) {
      if (kt < nkt) {
        last(kt);
      } else {  // (a wave without rows: it will not read them, or they stay alive on its account)
#pragma unroll
        for (int j = 0; j < FNC; ++j)
#pragma unroll
          for (int h = 0; h < 2; ++h) asm volatile("" : "=v"(blk_in.g[j][h]), "=v"(blk_in.u[j][h]));
      }
    }
    if (!stream) {
      if (EARLY_REQUEST && more) {
        set_rows();
        request_first(nxt);
      }
      lds_barrier();  // every wave is done reading the operand stages
    }
    if (STREAM && nkt > 0) strip = strip_in((s0 + nkt - 1) & 1);
    s0 = (s0 + nkt) & 1;
    staged = stream;
    // Where the epilogue needs the staging registers' room for most of its length, the request
    // goes out as soon as that room is free: during the last of its strips.
    bool requested = EARLY_REQUEST;
    auto request_next = [&]() {
      if (!stream) {
        set_rows();
        request_first(nxt);
      } else {
        request_k(nxt, 1);
      }
    };
    auto late_request = [&]() {
      if constexpr (!EARLY_REQUEST) {
        if (more) request_next();
        requested = true;
      }
    };
    if (!idle) epilogue(cur, late_request);
    if (!more) break;
    if (!requested) request_next();
    lds_barrier();  // every wave is done with its strip, and stage s0 is complete if staged
    cur = nxt;
  }
}

using CfgMain = TileCfg<ROW_TILE, 256, 64, 2, 4>;
// Row tiles of half the height (the eight waves 64 x 64 each), at 0.65 to 0.7 of a tile's cost.
using CfgHalf = TileCfg<ROW_TILE / 2, 256, 64, 2, 4>;

// tile_start[e] = number of tiles of UNIT rows of the experts before e (and of all from E up to the next multiple of 128 on), offs =
// p.offs, both in LDS (wave 0 scans, two experts a lane: past 64 of them one trip to memory instead of two, 2.2 -> 1.3 us
// from the kernel's start).
template <int UNIT>
__device__ __forceinline__ void number_tiles(const GemmArgs& p, int* tile_start, int* offs) {
  const int lane = threadIdx.x & 63;
  if (threadIdx.x < MOE_WAVE) {
    int carry = 0;
    for (int b = 0; b < p.E; b += 2 * MOE_WAVE) {
      int first[2], end[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int e = b + h * MOE_WAVE + lane;
        first[h] = e < p.E ? p.offs[e] : 0, end[h] = e < p.E ? p.offs[e + 1] : 0;
      }
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int e = b + h * MOE_WAVE + lane;
        const int nt = (end[h] - first[h] + UNIT - 1) / UNIT, incl = wave_inclusive(nt);
        if (e < GEMM_MAX_E) tile_start[e] = carry + incl - nt;
        if (e < p.E) {
          offs[e] = first[h];
          if (e == p.E - 1) offs[p.E] = end[h];
        }
        carry += read_lane(incl, MOE_WAVE - 1);
      }
    }
    if (lane == 0) tile_start[p.E] = carry;
  }
  __syncthreads();
}

// Every tile of a row-ragged launch costs about the same.  Of the XCDs that have workgroups (all 8 unless the
// grid is tiny) XCD x takes the x-th contiguous eighth of the n positions of the list and its workgroups
// sweep it side by side: at any time they share a few experts' weights and row blocks in L2.
struct Sweep {
  int first, end, step;
};
__device__ __forceinline__ Sweep sweep_of(int n) {
  const int nb = gridDim.x, x = blockIdx.x & 7, j = blockIdx.x >> 3;
  const int nx = nb < 8 ? nb : 8;
  const int q = n / nx, r = n % nx;
  const int lo = x * q + (x < r ? x : r);
  return {lo + j, lo + q + (x < r ? 1 : 0), (nb >> 3) + (x < (nb & 7) ? 1 : 0)};
}

// The last round is mostly partial.  What is left after the whole rounds is done in half tiles where that is at most
// one to every workgroup, and the round before with it where that is at most two (at 0.65 of a tile two are less
// than a whole one and a half one).  Which halves have rows follows from the offsets; every workgroup works it
// out for itself, a tile a thread.  Whole tiles -> this, gate/up, down, dgrad-down and dgrad-gate/up in us:
//   16384 rows of 8 experts, 1024 <-> 512    54 -> 48, 32 -> 29, 40 (0.53 rounds, 264 halves), 53 -> 48
//   9999 rows of 12 experts, 1416 <-> 568    40 (0.9), 36 -> 29, 49 -> 36 (0.53 rounds, 252 halves), 61 -> 47
// From some ten rounds on it makes no difference.
// Except in dgrad-down, what is left is done in quarters of 64 x 256 instead where that is at most one with rows to every
// workgroup (a quarter of a round, or a round of tiles with up to 64 rows), through the ring of direct loads
// (csrc/row_ring.h): a short round waits for memory k-tile by k-tile, and the ring has two of them on their way.  Halves ->
// quarters, gate/up, down and dgrad-gate/up: 16384 rows of 8 experts as above 55, 32, 52 -> 52, 30, 48 us; 4321 rows of 24, 2880
// <-> 1440, 123, 81, 130 -> 113, 74, 120; over 8 layers, 4 to 64 experts and 12 to 1500 rows an expert 1.05, 1.04, 1.07 times as
// fast, 0.94 to 1.25.  (The same quarters with the staging registers of the other tiles: two thirds of that.)  Dgrad-down is
// 0.79 times as fast in quarters where they are all there is, and 0.94 after whole rounds (577 rows of 24 experts, 4096 <->
// 1536, 60 -> 96 us; 8641 rows of 48 193 -> 225), never more than 1.05.
template <int MODE, typename OutT, bool BLK, bool TO, bool FROM>
__global__ __launch_bounds__(CfgMain::NT, CfgMain::WAVES_PER_SIMD) void rows_gemm_kernel(const GemmArgs p) {
  static_assert(CfgHalf::NT == CfgMain::NT, "one workgroup runs both");
  constexpr int WAVES = CfgMain::NT / MOE_WAVE;
  constexpr int MAX_LISTED = CfgMain::NT;
  extern __shared__ __attribute__((aligned(16))) uint16_t smem[];
  __shared__ int tile_start[GEMM_MAX_E + 1], offs[GEMM_MAX_E + 1];
  __shared__ uint32_t half_list[MAX_LISTED];
  __shared__ int wave_halves[3][WAVES];
  number_tiles<ROW_TILE>(p, tile_start, offs);
  const int nb = gridDim.x;
  const int total = __builtin_amdgcn_readfirstlane(tile_start[p.E]) * p.n_tiles;
  int whole = total;  // tiles 0 .. whole are done whole
  int halves = 0;     // halves with rows of the others, or quarters
  bool quarters = false;
  const int left = total % nb;
  const bool can_quarter = MODE == DOWN || MODE == DGRAD_GATEUP || (MODE == GATEUP && (BLK || !p.C0));  // (g and u in rows: not)
  if (!p.whole_only && left > 0 && nb <= MAX_LISTED) {
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int round = total > nb && 2 * nb <= MAX_LISTED ? nb : 0;  // (of whole tiles that may be halved too)
    const int tile = total - left - round + (int)threadIdx.x;
    const bool last = tile >= total - left;
    int n = 0, n4 = 0;  // this tile's halves and quarters with rows
    if (tile < total) {
      const int slot = p.by_n_tiles(tile);
      int e = 0, hi = p.E;
      while (hi - e > 1) {
        const int mid = (e + hi) >> 1;
        if (tile_start[mid] <= slot) e = mid;
        else hi = mid;
      }
      const int rows = offs[e + 1] - offs[e] - (slot - tile_start[e]) * ROW_TILE;
      n = rows > CfgHalf::BM ? 2 : 1;
      n4 = last && can_quarter ? ((rows < ROW_TILE ? rows : ROW_TILE) + 63) / 64 : 0;
    }
    const unsigned long long some = __ballot(n > 0), both = __ballot(n > 1), in_last = __ballot(last);
    const unsigned long long below = (1ull << lane) - 1;
    int at4 = 0, all4 = 0;
#pragma unroll
    for (int h = 0; h < 4; ++h) {
      const unsigned long long b = __ballot(n4 > h);
      at4 += __popcll(b & below), all4 += __popcll(b);
    }
    if (lane == 0) {
      wave_halves[0][wv] = __popcll(some) + __popcll(both);
      wave_halves[1][wv] = __popcll(some & in_last) + __popcll(both & in_last);
      wave_halves[2][wv] = all4;
    }
    __syncthreads();
    int at = __popcll(some & below) + __popcll(both & below), all = 0, in_left = 0;
    all4 = 0;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) {
      const int c = __builtin_amdgcn_readfirstlane(wave_halves[0][w]);
      at += w < wv ? c : 0;
      all += c;
      in_left += __builtin_amdgcn_readfirstlane(wave_halves[1][w]);
      const int c4 = __builtin_amdgcn_readfirstlane(wave_halves[2][w]);
      at4 += w < wv ? c4 : 0;
      all4 += c4;
    }
    int skip = 0;  // halves of the round before, when that stays whole
    if (round > 0 && all <= 2 * nb) {
      halves = all;
      whole = total - left - round;
    } else if (can_quarter && all4 <= nb) {
      halves = all4;
      whole = total - left;
      quarters = true;
      for (int h = 0; h < n4; ++h) half_list[at4 + h] = 4u * (uint32_t)tile + h;
    } else if (in_left <= nb) {
      halves = in_left;
      whole = total - left;
      skip = all - in_left;
    }
    if (tile >= whole && !quarters)
      for (int h = 0; h < n; ++h) half_list[at + h - skip] = 2u * (uint32_t)tile + h;
  }
  const Sweep s = sweep_of(whole);
  walk_tiles<MODE, CfgMain, OutT, BLK, ROW_TILE, TO, FROM>(p, smem, tile_start, offs, nullptr, s.first, s.end, s.step);
  if (halves == 0) return;
  __syncthreads();  // (the operand stages are free, the list is complete)
  const Sweep h = sweep_of(halves);
  if constexpr (MODE != DGRAD_DOWN) {
    if (quarters) {
      using Quarter = RingTile<MODE, 1, CfgMain::NT / MOE_WAVE>;
      static_assert(Quarter::LDS <= lds_bytes<MODE, CfgMain>() && Quarter::BM * 4 == ROW_TILE, "fits");
      for (int at = h.first; at < h.end; at += h.step) {
        const int entry = __builtin_amdgcn_readfirstlane((int)half_list[at]), tile = entry >> 2, slot = p.by_n_tiles(tile);
        const int e = expert_of(tile_start, slot, p.E);
        const int first = __builtin_amdgcn_readfirstlane(offs[e]), end = __builtin_amdgcn_readfirstlane(offs[e + 1]);
        const int row = (slot - __builtin_amdgcn_readfirstlane(tile_start[e])) * ROW_TILE + (entry & 3) * Quarter::BM;
        ring_tile<MODE, BLK, 1, WAVES, TO, FROM>(p, (char*)smem, e, first, end, row, (tile - slot * p.n_tiles) * Quarter::BNC);
        __syncthreads();
      }
      return;
    }
  }
  walk_tiles<MODE, CfgHalf, OutT, BLK, ROW_TILE, TO, FROM>(p, smem, tile_start, offs, half_list, h.first, h.end, h.step);
}

// All in half tiles: launches of so few tiles that there is nothing to decide and that csrc/row_ring.hip does not take (4096 rows
// of 8 experts, 1024 <-> 512, gate/up 19.5 us; in ring tiles of 64 rows, a few more than fit at once, 23.3).
template <int MODE, typename OutT, bool BLK, bool TO, bool FROM>
__global__ __launch_bounds__(CfgHalf::NT, CfgHalf::WAVES_PER_SIMD) void small_rows_gemm_kernel(const GemmArgs p) {
  extern __shared__ __attribute__((aligned(16))) uint16_t smem[];
  __shared__ int tile_start[GEMM_MAX_E + 1], offs[GEMM_MAX_E + 1];
  number_tiles<CfgHalf::BM>(p, tile_start, offs);
  const Sweep s = sweep_of(__builtin_amdgcn_readfirstlane(tile_start[p.E]) * p.n_tiles);
  walk_tiles<MODE, CfgHalf, OutT, BLK, CfgHalf::BM, TO, FROM>(p, smem, tile_start, offs, nullptr, s.first, s.end, s.step);
}

// Weight gradients: of up to three problems that share their experts' rows, one's tiles behind the other's without a launch
// between them.  (What a launch's end, in which workgroups wait for the last ones, and the next one's start cost.  Whole steps, us,
// a launch a problem and one: 9000 rows of 64 experts, 1024 <-> 1024, by Dirichlet's shares 443 -> 428; 4096 tokens, 8 of 128, 1024 <->
// 256 459 -> 452; 450, 3 of 96, 3584 <-> 296 (three problems) 628 -> 616; 1558, 8 of 64 by Zipf's shares, 1792 <-> 1152 1014 -> 959; steps of a
// few ms 1.00 to 1.02; of 24 layers one is slower by more than the noise, 160 tokens, 1 of 12, 3952 <-> 1936, 579 -> 581.)
constexpr int WGRAD_PROBLEMS = 3;
struct WgradArgs {
  GemmArgs p[WGRAD_PROBLEMS];
  int n;
};
// ---- which tiles a workgroup computes
// The kernel is persistent: the grid has one workgroup per compute unit and each walks a
// list of tiles.  Hardware hands workgroup b to XCD b % 8 (each XCD has its own L2).
// With more tiles than workgroups: a tile of expert e contracts over that expert's rows,
// so under skewed routing tiles differ in cost by orders of magnitude and a contiguous range is
// all heavy or all light.  The (expert-major) list is dealt in groups of as many consecutive
// tiles as an XCD has workgroups, group g to XCD g % 8, one tile to each of its workgroups: the
// workgroups of an XCD stay on one expert (or two) and walk its rows together, and every XCD
// sees every part of the list.  With at most 64 experts, whole groups per expert and skewed
// routing (the largest expert above 1.25 times the mean) the groups are not dealt round-robin
// but longest first: experts in descending order of their rows, each group to the XCD with the
// least work so far; every workgroup works that out for itself from the offsets, the same way,
// and keeps its own tiles' numbers in LDS.  (A generated power-law skew over 16 experts: 10-12 %
// faster dealt in groups than with contiguous ranges of equal work, another 9-10 % longest
// first; near-uniform routing: the same in all three.)  A tile of an expert costs the same in every problem: the next one's
// groups are dealt on from where the last one's left the XCDs.
template <typename OutT, int FROM>
__global__ __launch_bounds__(CfgMain::NT, CfgMain::WAVES_PER_SIMD) void wgrad_gemm_kernel(const WgradArgs a) {
  extern __shared__ __attribute__((aligned(16))) uint16_t smem[];
  const int lane = threadIdx.x & 63;
  constexpr int MAX_GROUPS = 512;
  __shared__ uint32_t glist[MAX_GROUPS];   // this XCD's groups, problem by problem
  __shared__ int gcount[WGRAD_PROBLEMS];   // up to the end of each; -1: dealt round-robin
  const int nb = gridDim.x, x = blockIdx.x & 7, j = blockIdx.x >> 3, wgs = nb >> 3;
  const int E = a.p[0].E;
  const auto tiles_of = [&](int w) { return a.p[w].m_slots * a.p[w].n_tiles; };  // of an expert
  bool dealt = (nb & 7) == 0, ranked = E <= MOE_WAVE;
  int groups = 0;
  for (int w = 0; w < a.n; ++w) {
    const int n = tiles_of(w);
    dealt = dealt && E * n > nb;
    ranked = ranked && dealt && n % wgs == 0;
    if (ranked) groups += E * (n / wgs);
  }
  ranked = ranked && groups <= MAX_GROUPS;
  if (ranked) {
    if (threadIdx.x < MOE_WAVE) {
      constexpr long long FIXED = 4 * CfgMain::BK;  // fill, tile switch and epilogue, in rows' worth
      int rows = 0;
      if (lane < E) {
        rows = a.p[0].offs[lane + 1] - a.p[0].offs[lane];
        rows = rows < 0 ? 0 : rows;
      }
      const long long cost = rows + FIXED;
      // (only worth it when the routing is skewed: with near-equal experts the plain dealing is
      // as balanced and keeps neighbouring experts on neighbouring XCDs)
      int mx = rows, sum = rows;
#pragma unroll
      for (int off = MOE_WAVE / 2; off > 0; off >>= 1) {
        const int om = __shfl_xor(mx, off, MOE_WAVE);
        mx = om > mx ? om : mx;
        sum += __shfl_xor(sum, off, MOE_WAVE);
      }
      const bool skewed = 4ll * mx * E > 5ll * sum;
      int rank = 0;  // position of expert `lane` in descending order of cost (ties: lower index first)
      for (int o = 0; o < E; ++o) {
        const long long co = __shfl(cost, o, MOE_WAVE);
        rank += (co > cost || (co == cost && o < lane)) ? 1 : 0;
      }
      if (lane >= E) rank = -1;
      // lanes 0..7 carry the XCDs' loads, packed with the XCD index for the arg-min
      long long load = 0;
      int cnt = 0;
      for (int w = 0; skewed && w < a.n; ++w) {
        const int gpe = tiles_of(w) / wgs;  // groups per expert
        for (int s_ = 0; s_ < E; ++s_) {
          const int e = __builtin_ctzll(__ballot(rank == s_));
          const long long ce = __shfl(cost, e, MOE_WAVE);
          for (int gi = 0; gi < gpe; ++gi) {
            long long key = lane < 8 ? ((load << 3) | lane) : 0x7fffffffffffffffll;
#pragma unroll
            for (int off = 1; off < 8; off <<= 1) {
              const long long other = __shfl_xor(key, off, MOE_WAVE);
              key = other < key ? other : key;
            }
            const int xmin = (int)(__shfl(key, 0, MOE_WAVE) & 7);
            if (lane == xmin) load += ce;
            if (xmin == x) {
              if (lane == 0) glist[cnt] = (e * gpe + gi) * wgs + j;
              ++cnt;
            }
          }
        }
        if (lane == 0) gcount[w] = cnt;
      }
      if (lane == 0 && !skewed) gcount[0] = -1;
    }
    __syncthreads();
    ranked = gcount[0] >= 0;
  }
  int done = 0;  // tiles of the problems before
#pragma unroll 1
  for (int w = 0; w < a.n; ++w) {
    const GemmArgs p = a.p[w];  // (in registers: read where it is used, a tile of one k-tile is 1 % longer)
    const int total = E * tiles_of(w);
    int first, end, step;
    if (ranked) {
      first = w ? gcount[w - 1] : 0, end = gcount[w], step = 1;
    } else if (dealt) {
      // (a problem begins with the workgroups, in whole XCDs, that have one tile less of those before)
      const int skip = done % nb / wgs * wgs, at = x * wgs + j;
      first = at >= skip ? at - skip : at - skip + nb, end = total, step = nb;
    } else {
      const int nx = nb < 8 ? nb : 8, q = total / nx, r = total % nx, lo = x * q + (x < r ? x : r);
      first = lo + j, end = lo + q + (x < r ? 1 : 0), step = (nb >> 3) + (x < (nb & 7) ? 1 : 0);
    }
    if (w) __syncthreads();  // (the operand stages are free)
    if (FROM && p.row_from)
      walk_tiles<WGRAD, CfgMain, OutT, false, ROW_TILE, false, FROM>(p, smem, nullptr, p.offs, ranked ? glist : nullptr, first, end, step);
    else walk_tiles<WGRAD, CfgMain, OutT, false>(p, smem, nullptr, p.offs, ranked ? glist : nullptr, first, end, step);
    done += total;
  }
}

}  // namespace

int moe_compute_units() {
  static int cus[MOE_MAX_DEVICES];  // per GPU; 0 = not asked yet
  const int dev = moe_current_device();
  if (cus[dev] == 0) {
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
    cus[dev] = n;
  }
  return cus[dev];
}

namespace {


// As many workgroups as are resident at once (one per compute unit), or as there are jobs.
template <int MODE, typename Cfg, typename Args>
int launch(void (*kern)(Args), bool (&attr_done)[MOE_MAX_DEVICES], const Args& a, long long jobs, hipStream_t s) {
  if (jobs <= 0) return 0;
  constexpr int LDS = lds_bytes<MODE, Cfg>();
  const int dev = moe_current_device();
  if (!attr_done[dev]) {
    hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
    if (e != hipSuccess) return (int)e;
    attr_done[dev] = true;
  }
  const long long slots = moe_compute_units();
  const unsigned grid = (unsigned)(jobs < slots ? jobs : slots);
  hipLaunchKernelGGL(kern, dim3(grid), dim3(Cfg::NT), LDS, s, a);
  return moe_launch_status();
}

long long row_slots(int64_t R, int64_t E, int tile) { return (R + tile - 1) / tile + E; }

// Which kernel a row-ragged launch takes: decided from the shapes alone (never from the routing: no host
// synchronisation).  With fewer tiles than half the compute units, by the bound on their number, every one of them can be
// halved, as long as the halves are one round (gate/up has twice the tiles for its columns; 10842 rows of 8 experts, 2496 <-> 320, 266
// halves 69 us, whole tiles and quarters 50; 13653 of 12, 1984 <-> 192, 225 halves, 34 and 35.5); what csrc/row_ring.hip takes is done there.  `forced_row_tile` (0: automatic) is a test hook.
constexpr int RING_TILE = 64, RING_TALL = 1;  // (1: the ring's tiles of 128 rows)
int forced_row_tile = 0;

// A row-ragged launch with `cols` output columns to a tile.
template <int MODE, bool BLK = false, bool TO = false, bool FROM = false>
int launch_rows(GemmArgs& a, int cols, hipStream_t s) {
  static_assert(lds_bytes<MODE, CfgHalf>() <= lds_bytes<MODE, CfgMain>(), "both row tiles fit");
  static bool attr_done[2][MOE_MAX_DEVICES];  // per GPU and instantiation
  int rc = 0;
  if (forced_row_tile <= RING_TILE &&
      moe_ring_rows((Mode)MODE, BLK, a, forced_row_tile == RING_TALL ? 128 : forced_row_tile, s, &rc))
    return rc;
  a.n_tiles = (a.N + cols - 1) / cols;
  a.by_n_tiles.set(a.n_tiles);
  const long long tiles = row_slots(a.R, a.E, ROW_TILE) * ((a.N + CfgMain::BN - 1) / CfgMain::BN);
  const bool small = forced_row_tile > RING_TILE ? forced_row_tile == CfgHalf::BM
                                                 : 2 * tiles < moe_compute_units() &&
                                                       moe_expected_tiles(a.R, a.E, CfgHalf::BM) * a.n_tiles <= moe_compute_units();
  if (small)
    return launch<MODE, CfgHalf>(small_rows_gemm_kernel<MODE, uint16_t, BLK, TO, FROM>, attr_done[0], a,
                                 a.n_tiles * row_slots(a.R, a.E, CfgHalf::BM), s);
  a.whole_only = forced_row_tile == ROW_TILE;
  // (act streamed past the caches where rows an expert are few, as it takes the weights' place in L2, gains nothing for certain: at 40 to 195 rows
  // an expert, 14 layers, ordinary -> streaming, forward passes 0.95 to 1.08 times as fast, 1.00 in the mean (1280 tokens of 32, 2624 <-> 1792,
  // 260 -> 273 us; 1280 of 64, 2048 <-> 1024, 230 -> 214), training 0.96 to 1.03, as down and the weight gradients read it next.)
  return launch<MODE, CfgMain>(rows_gemm_kernel<MODE, uint16_t, BLK, TO, FROM>, attr_done[1], a,
                               2 * a.n_tiles * row_slots(a.R, a.E, ROW_TILE), s);
}
// With few rows an expert the results come as fast as the operands do, and as streaming stores they leave the operands' lines in L2
// alone; what reads small ones afterwards would miss them (MOE_STREAMED_RESULTS).  Rows an expert and time, streaming over ordinary, three results in
// turn so that none is still cached: 64 experts of 2048 <-> 1024, bf16 and fp32: 256, 0.86 and 0.83; 512, 0.93 and 0.91; 768, 1.01 and 1.04;
// 1024, 1.00 and 1.01; 2048, 1.00 and 1.00.  128 of 1024 <-> 256, 128 to 512 rows 0.93 to 0.96 and 0.84 to 0.92; 16 of 4096 <-> 1536, 1024 rows
// 0.95 and 0.95; by Zipf's shares, 500 rows of 64 1.00 and 0.85.
// (as for wgrad_multi_kernel: rows of whole pieces of 64 bytes)
template <typename OutT>
int launch_wgrad(const WgradArgs& args, hipStream_t s) {
  WgradArgs w = args;
  long long tiles = 0, bytes = 0;
  for (int i = 0; i < w.n; ++i) bytes += (long long)w.p[i].E * w.p[i].M * w.p[i].N * (int)sizeof(OutT);
  for (int i = 0; i < w.n; ++i) {
    GemmArgs& a = w.p[i];
    a.n_tiles = (a.N + CfgMain::BN - 1) / CfgMain::BN;
    a.m_slots = (a.M + CfgMain::BM - 1) / CfgMain::BM;
    a.by_n_tiles.set(a.n_tiles), a.by_m_slots.set(a.m_slots);
    a.streaming = bytes >= MOE_STREAMED_RESULTS && a.R <= 512ll * a.E && a.N * (int)sizeof(OutT) % 64 == 0;
    const long long n = (long long)a.n_tiles * a.m_slots * a.E;
    tiles = tiles > n ? tiles : n;
  }
  static bool attr_done[3][MOE_MAX_DEVICES];
  int from = 0;  // (a's lines are where the caller has them where the experts are given, b's where the router is part of the call)
  for (int i = 0; i < w.n; ++i) {
    const int of = w.p[i].row_from ? (w.p[i].from_a ? FROM_A : FROM_B) : 0;
    if (of && from && of != from) return MOE_ERR_LIMIT;
    from |= of;
  }
  if (from == FROM_A) return launch<WGRAD, CfgMain>(wgrad_gemm_kernel<OutT, FROM_A>, attr_done[1], w, tiles, s);
  if (from == FROM_B) return launch<WGRAD, CfgMain>(wgrad_gemm_kernel<OutT, FROM_B>, attr_done[2], w, tiles, s);
  return launch<WGRAD, CfgMain>(wgrad_gemm_kernel<OutT, 0>, attr_done[0], w, tiles, s);
}

int check_common(const int32_t* offs, int64_t E, int64_t R, int64_t H, int64_t I) {
  if (!offs) return MOE_ERR_NULL;
  if (E <= 0 || R < 0 || H <= 0 || I <= 0 || (H % 8) || (I % 8)) return MOE_ERR_SHAPE;
  if (E > GEMM_MAX_E || R > (int64_t)1 << 30 || H > (1 << 16) || I > (1 << 16)) return MOE_ERR_LIMIT;
  // Row and column positions are 64-bit wherever they are multiplied by a row length; what is
  // 32-bit is the per-lane offset inside one tile's window (at most 256 rows of 65536 elements)
  // and the tile index: rows / 256 + E row slots times the column tiles of the widest output.
  const int64_t widest = H > I ? H : I;
  if ((R / 256 + E + 1) * ((widest + 127) / 128) >= ((int64_t)1 << 31)) return MOE_ERR_LIMIT;
  return 0;
}

}  // namespace

// A's rows where the tokens are.  The copies in expert order are a pass that writes k rows a token and a gate/up that reads them from memory,
// where the tokens' own rows stay in the caches; a lane's offset a row instead of a constant one costs the loop nothing (the offsets are in registers
// either way, 253 of them with the next tile's row).  Forward passes, us, copies -> this, the same bits: 64 experts, 2048 <-> 1024, 8 a token, 257 / 700
// / 1531 / 4000 / 16384 tokens 166 -> 163, 187 -> 180, 245 -> 230, 496 -> 469, 1742 -> 1639; 8192 of 128, 1024 <-> 256, 232 -> 204; 2048 of 8, 1024 <->
// 512, 42.6 -> 40.3; 3333 of 12, 1416 <-> 568, 99 -> 92; 16000, 1 of 4, 512 <-> 256, 60.6 -> 57.1; no size of 16 slower.  A lane's
// offset and a window's size have 32 bits, and one of them marks rows that there are none of: hence the limit.
bool moe_rows_from_ok(int64_t T, int64_t H) { return T * H < (int64_t)1 << 30; }

int moe_gemm_gateup_from(const uint16_t* x, const int32_t* pos_to_row, int64_t T, int64_t k, const uint16_t* w1, const uint16_t* w3,
                         const int32_t* offs, int64_t E, int64_t H, int64_t I, void* gu_blocked, uint16_t* act, void* stream) {
  const int64_t R = T * k;
  if (int rc = check_common(offs, E, R, H, I)) return rc;
  if (R == 0) return 0;
  if (!moe_rows_from_ok(T, H)) return MOE_ERR_LIMIT;
  MOE_CHECK_PTR(x); MOE_CHECK_PTR(w1); MOE_CHECK_PTR(w3); MOE_CHECK_PTR(act); MOE_CHECK_PTR(pos_to_row);
  GemmArgs a{};
  a.A0 = x; a.B0 = w1; a.B1 = w3; a.C0 = gu_blocked; a.C2 = act; a.offs = offs;
  a.E = (int)E; a.R = (int)R; a.N = (int)I; a.K = (int)H;
  a.row_from = pos_to_row; a.by_k.set((uint32_t)k); a.from_bytes = T * H * 2;
  if (gu_blocked) {
    MOE_CHECK_PTR(gu_blocked);
    return launch_rows<GATEUP, true, false, true>(a, CfgMain::BN / 2, (hipStream_t)stream);
  }
  return launch_rows<GATEUP, false, false, true>(a, CfgMain::BN / 2, (hipStream_t)stream);
}

extern "C" int moe_gemm_gateup_swiglu_fwd(const uint16_t* xp, const uint16_t* w1, const uint16_t* w3,
                                          const int32_t* offs, int64_t E, int64_t R, int64_t H,
                                          int64_t I, uint16_t* g, uint16_t* u, uint16_t* act,
                                          void* stream) {
  if (int rc = check_common(offs, E, R, H, I)) return rc;
  if (R == 0) return 0;
  MOE_CHECK_PTR(xp); MOE_CHECK_PTR(w1); MOE_CHECK_PTR(w3); MOE_CHECK_PTR(act);
  if ((g == nullptr) != (u == nullptr)) return MOE_ERR_NULL;
  GemmArgs a{};
  a.A0 = xp; a.B0 = w1; a.B1 = w3; a.C0 = g; a.C1 = u; a.C2 = act; a.offs = offs;
  a.E = (int)E; a.R = (int)R; a.N = (int)I; a.K = (int)H;
  return launch_rows<GATEUP>(a, CfgMain::BN / 2, (hipStream_t)stream);
}

// Bytes of the blocked g/u buffer: one 4 KB record per 32 x 32 block (R/32 + E bounds the number of row
// blocks whatever the routing).
extern "C" int64_t moe_gu_blocked_bytes(int64_t R, int64_t E, int64_t I) {
  if (R <= 0 || E <= 0 || I <= 0) return 0;
  return (R / 32 + E) * ((I + 31) / 32) * 4096;
}

extern "C" int moe_gemm_gateup_swiglu_fwd_blocked(const uint16_t* xp, const uint16_t* w1, const uint16_t* w3,
                                                  const int32_t* offs, int64_t E, int64_t R, int64_t H,
                                                  int64_t I, void* gu_blocked, uint16_t* act, void* stream) {
  if (int rc = check_common(offs, E, R, H, I)) return rc;
  if (R == 0) return 0;
  MOE_CHECK_PTR(xp); MOE_CHECK_PTR(w1); MOE_CHECK_PTR(w3); MOE_CHECK_PTR(act); MOE_CHECK_PTR(gu_blocked);
  GemmArgs a{};
  a.A0 = xp; a.B0 = w1; a.B1 = w3; a.C0 = gu_blocked; a.C2 = act; a.offs = offs;
  a.E = (int)E; a.R = (int)R; a.N = (int)I; a.K = (int)H;
  return launch_rows<GATEUP, true>(a, CfgMain::BN / 2, (hipStream_t)stream);
}

int moe_gemm_down_to(const uint16_t* act, const uint16_t* w2, const int32_t* offs, int64_t E, int64_t R, int64_t H, int64_t I,
                     uint16_t* y, const int32_t* row_map, void* stream) {
  if (int rc = check_common(offs, E, R, H, I)) return rc;
  if (R == 0) return 0;
  MOE_CHECK_PTR(act); MOE_CHECK_PTR(w2); MOE_CHECK_PTR(y);
  GemmArgs a{};
  a.A0 = act; a.B0 = w2; a.C0 = y; a.offs = offs;
  a.E = (int)E; a.R = (int)R; a.N = (int)H; a.K = (int)I; a.row_map = row_map;
  if (row_map) return launch_rows<DOWN, false, true>(a, CfgMain::BN, (hipStream_t)stream);
  return launch_rows<DOWN>(a, CfgMain::BN, (hipStream_t)stream);
}

extern "C" int moe_gemm_down_fwd(const uint16_t* act, const uint16_t* w2, const int32_t* offs,
                                 int64_t E, int64_t R, int64_t H, int64_t I, uint16_t* y,
                                 void* stream) {
  return moe_gemm_down_to(act, w2, offs, E, R, H, I, y, nullptr, stream);
}

// Test hook: 0 lets every row-ragged launch choose its row-tile height (the default), 64, 128 or 256 forces it, 1
// the ring's tiles of 128 rows (64 and 1: of the launches that have such tiles).  Process-wide and not synchronised: for tests that want every shape on every
// tile configuration, not for production callers.  Returns the previous setting.
extern "C" int moe_gemm_force_row_tile(int rows) {
  const int before = forced_row_tile;
  if (rows == 0 || rows == RING_TILE || rows == RING_TALL || rows == CfgHalf::BM || rows == CfgMain::BM) forced_row_tile = rows;
  return before;
}

extern "C" int64_t moe_dgate_blocks(int64_t I) {
  using Cfg = CfgMain;
  return I <= 0 ? 0 : ((I + Cfg::BN - 1) / Cfg::BN) * Cfg::WN;
}

static int dgrad_down_impl(const uint16_t* dyp, const uint16_t* w2, const uint16_t* g, const uint16_t* u,
                           const int32_t* offs, int64_t E, int64_t R, int64_t H, int64_t I,
                           uint16_t* dg, uint16_t* du, float* dgate_part, void* stream, int64_t ld_out = 0) {
  if (int rc = check_common(offs, E, R, H, I)) return rc;
  if (R == 0) return 0;
  MOE_CHECK_PTR(dyp); MOE_CHECK_PTR(w2); MOE_CHECK_PTR(g); MOE_CHECK_PTR(u);
  MOE_CHECK_PTR(dg); MOE_CHECK_PTR(du);
  GemmArgs a{};
  a.C2 = dgate_part;
  a.A0 = dyp; a.B0 = w2; a.X0 = g; a.X1 = u; a.C0 = dg; a.C1 = du; a.offs = offs;
  a.E = (int)E; a.R = (int)R; a.N = (int)I; a.K = (int)H; a.ld_c = (int)ld_out;
  return launch_rows<DGRAD_DOWN>(a, CfgMain::BN, (hipStream_t)stream);
}

extern "C" int moe_gemm_dgrad_down_swiglu_bwd(const uint16_t* dyp, const uint16_t* w2,
                                              const uint16_t* g, const uint16_t* u,
                                              const int32_t* offs, int64_t E, int64_t R, int64_t H,
                                              int64_t I, uint16_t* dg, uint16_t* du, void* stream) {
  return dgrad_down_impl(dyp, w2, g, u, offs, E, R, H, I, dg, du, nullptr, stream);
}

extern "C" int moe_gemm_dgrad_down_swiglu_bwd_dgate(const uint16_t* dyp, const uint16_t* w2,
                                                    const uint16_t* g, const uint16_t* u,
                                                    const int32_t* offs, int64_t E, int64_t R,
                                                    int64_t H, int64_t I, uint16_t* dg, uint16_t* du,
                                                    float* dgate_part, void* stream) {
  if (R > 0 && !dgate_part) return MOE_ERR_NULL;
  return dgrad_down_impl(dyp, w2, g, u, offs, E, R, H, I, dg, du, dgate_part, stream);
}

// dyp: row p is row p of it, or with pos_to_row row pos_to_row[p] / k of its `from_rows`
static int dgrad_down_blocked(const uint16_t* dyp, const int32_t* pos_to_row, int64_t from_rows, int64_t k, const uint16_t* w2,
                              const void* gu_blocked, const int32_t* offs, int64_t E, int64_t R, int64_t H, int64_t I, uint16_t* dg,
                              uint16_t* du, int64_t ld_out, float* dgate_part, void* stream) {
  if (int rc = check_common(offs, E, R, H, I)) return rc;
  if (R == 0) return 0;
  MOE_CHECK_PTR(dyp); MOE_CHECK_PTR(w2); MOE_CHECK_PTR(gu_blocked); MOE_CHECK_PTR(dg); MOE_CHECK_PTR(du);
  if (ld_out != 0 && (ld_out < I || (ld_out % 8) != 0 || ld_out > (1 << 17))) return MOE_ERR_SHAPE;
  GemmArgs a{};
  a.C2 = dgate_part;
  a.A0 = dyp; a.B0 = w2; a.X0 = (const uint16_t*)gu_blocked; a.C0 = dg; a.C1 = du; a.offs = offs;
  a.E = (int)E; a.R = (int)R; a.N = (int)I; a.K = (int)H; a.ld_c = (int)ld_out;
  if (!pos_to_row) return launch_rows<DGRAD_DOWN, true>(a, CfgMain::BN, (hipStream_t)stream);
  if (!moe_rows_from_ok(from_rows, H)) return MOE_ERR_LIMIT;
  a.row_from = pos_to_row; a.by_k.set((uint32_t)k); a.from_bytes = from_rows * H * 2;
  return launch_rows<DGRAD_DOWN, true, false, true>(a, CfgMain::BN, (hipStream_t)stream);
}

extern "C" int moe_gemm_dgrad_down_swiglu_bwd_blocked(const uint16_t* dyp, const uint16_t* w2,
                                                      const void* gu_blocked, const int32_t* offs, int64_t E,
                                                      int64_t R, int64_t H, int64_t I, uint16_t* dg,
                                                      uint16_t* du, int64_t ld_out, float* dgate_part,
                                                      void* stream) {
  return dgrad_down_blocked(dyp, nullptr, R, 1, w2, gu_blocked, offs, E, R, H, I, dg, du, ld_out, dgate_part, stream);
}

int moe_gemm_dgrad_down_from(const uint16_t* dy, const int32_t* pos_to_row, int64_t T, int64_t k, const uint16_t* w2,
                             const void* gu_blocked, const int32_t* offs, int64_t E, int64_t H, int64_t I, uint16_t* dg, uint16_t* du,
                             int64_t ld_out, float* dgate_part, void* stream) {
  if (!pos_to_row) return MOE_ERR_NULL;
  return dgrad_down_blocked(dy, pos_to_row, T, k, w2, gu_blocked, offs, E, T * k, H, I, dg, du, ld_out, dgate_part, stream);
}

// The two row gradients side by side in one buffer: dgu [R, 2I], row = [dg row | du row].  The
// weight gradients of the gate and up stacks then are ONE grouped product, dgu^T * xp, whose
// result rows 0..I-1 are dW1 and I..2I-1 dW3 (moe_gemm_wgrad_pair).
extern "C" int moe_gemm_dgrad_down_swiglu_bwd_packed(const uint16_t* dyp, const uint16_t* w2,
                                                     const uint16_t* g, const uint16_t* u,
                                                     const int32_t* offs, int64_t E, int64_t R,
                                                     int64_t H, int64_t I, uint16_t* dgu,
                                                     float* dgate_part, void* stream) {
  if (R > 0 && !dgu) return MOE_ERR_NULL;
  return dgrad_down_impl(dyp, w2, g, u, offs, E, R, H, I, dgu, dgu ? dgu + I : nullptr, dgate_part, stream, 2 * I);
}

int moe_gemm_dgrad_gateup_to(const uint16_t* dg, const uint16_t* du, int64_t ld_in, const uint16_t* w1, const uint16_t* w3,
                             const int32_t* offs, int64_t E, int64_t R, int64_t H, int64_t I, uint16_t* dxp,
                             const int32_t* row_map, void* stream) {
  if (int rc = check_common(offs, E, R, H, I)) return rc;
  if (R == 0) return 0;
  MOE_CHECK_PTR(dg); MOE_CHECK_PTR(du); MOE_CHECK_PTR(w1); MOE_CHECK_PTR(w3); MOE_CHECK_PTR(dxp);
  GemmArgs a{};
  a.A0 = dg; a.A1 = du; a.B0 = w1; a.B1 = w3; a.C0 = dxp; a.offs = offs; a.ld_a = (int)ld_in;
  a.E = (int)E; a.R = (int)R; a.N = (int)H; a.K = (int)I; a.row_map = row_map;
  if (row_map) return launch_rows<DGRAD_GATEUP, false, true>(a, CfgMain::BN, (hipStream_t)stream);
  return launch_rows<DGRAD_GATEUP>(a, CfgMain::BN, (hipStream_t)stream);
}

extern "C" int moe_gemm_dgrad_gateup_packed(const uint16_t* dgu, const uint16_t* w1, const uint16_t* w3,
                                            const int32_t* offs, int64_t E, int64_t R, int64_t H,
                                            int64_t I, uint16_t* dxp, void* stream) {
  if (R > 0 && !dgu) return MOE_ERR_NULL;
  return moe_gemm_dgrad_gateup_to(dgu, dgu ? dgu + I : nullptr, 2 * I, w1, w3, offs, E, R, H, I, dxp, nullptr, stream);
}

static int wgrad_pair_args(GemmArgs& a, const uint16_t* dgu, const uint16_t* xp, const int32_t* offs, int64_t E, int64_t R,
                           int64_t I, int64_t H, void* dw1, void* dw3, int dw_dtype, int accumulate) {
  if (int rc = check_common(offs, E, R, I, H)) return rc;  // (the stacked result has 2*I <= 131072 rows)
  // a 256-row tile of the stacked result must not straddle the two halves
  if ((I % CfgMain::BM) != 0) return MOE_ERR_SHAPE;
  MOE_CHECK_PTR(dw1); MOE_CHECK_PTR(dw3);
  if (R > 0) { MOE_CHECK_PTR(dgu); MOE_CHECK_PTR(xp); }
  if (dw_dtype != MOE_DT_BF16 && dw_dtype != MOE_DT_F32) return MOE_ERR_DTYPE;
  a = {};
  a.A0 = dgu; a.B0 = xp; a.C0 = dw1; a.C1 = dw3; a.offs = offs; a.m_split = (int)I;
  a.E = (int)E; a.R = (int)R; a.M = (int)(2 * I); a.N = (int)H; a.accumulate = accumulate;
  return 0;
}

static int wgrad_args(GemmArgs& a, const uint16_t* a_, const uint16_t* b_, const int32_t* offs, int64_t E, int64_t R, int64_t M,
                      int64_t N, void* dw, int dw_dtype, int accumulate) {
  if (int rc = check_common(offs, E, R, M, N)) return rc;
  MOE_CHECK_PTR(dw);
  if (R > 0) { MOE_CHECK_PTR(a_); MOE_CHECK_PTR(b_); }
  if (dw_dtype != MOE_DT_BF16 && dw_dtype != MOE_DT_F32) return MOE_ERR_DTYPE;
  a = {};
  a.A0 = a_; a.B0 = b_; a.C0 = dw; a.offs = offs;
  a.E = (int)E; a.R = (int)R; a.M = (int)M; a.N = (int)N; a.accumulate = accumulate;
  return 0;
}

static int run_wgrad(const WgradArgs& w, int dw_dtype, void* stream) {
  return dw_dtype == MOE_DT_F32 ? launch_wgrad<float>(w, (hipStream_t)stream) : launch_wgrad<uint16_t>(w, (hipStream_t)stream);
}

extern "C" int moe_gemm_wgrad_pair(const uint16_t* dgu, const uint16_t* xp, const int32_t* offs, int64_t E,
                                   int64_t R, int64_t I, int64_t H, void* dw1, void* dw3, int dw_dtype,
                                   int accumulate, void* stream) {
  WgradArgs w{};
  w.n = 1;
  if (int rc = wgrad_pair_args(w.p[0], dgu, xp, offs, E, R, I, H, dw1, dw3, dw_dtype, accumulate)) return rc;
  return run_wgrad(w, dw_dtype, stream);
}

int moe_gemm_wgrad_all(const MoeWgradStack* stacks, int n, const int32_t* offs, int64_t E, int64_t R, void* stream) {
  WgradArgs w{};
  if (n < 1 || n > WGRAD_PROBLEMS) return MOE_ERR_LIMIT;
  for (; w.n < n; ++w.n) {
    const MoeWgradStack& m = stacks[w.n];
    if (m.dtype != stacks[0].dtype) return MOE_ERR_DTYPE;
    const int rc = m.out2 ? wgrad_pair_args(w.p[w.n], m.a, m.b, offs, E, R, m.M / 2, m.N, m.out, m.out2, m.dtype, m.accumulate)
                          : wgrad_args(w.p[w.n], m.a, m.b, offs, E, R, m.M, m.N, m.out, m.dtype, m.accumulate);
    if (rc) return rc;
    if (m.row_from) {
      const int64_t wide = m.from_a ? m.M : m.N;
      if (!moe_rows_from_ok(m.from_rows, wide) || (m.from_a && m.out2)) return MOE_ERR_LIMIT;
      w.p[w.n].row_from = m.row_from, w.p[w.n].by_k.set((uint32_t)m.from_k), w.p[w.n].from_bytes = m.from_rows * wide * 2;
      w.p[w.n].from_a = m.from_a;
    }
  }
  return run_wgrad(w, stacks[0].dtype, stream);
}

extern "C" int moe_gemm_dgrad_gateup(const uint16_t* dg, const uint16_t* du, const uint16_t* w1,
                                     const uint16_t* w3, const int32_t* offs, int64_t E, int64_t R,
                                     int64_t H, int64_t I, uint16_t* dxp, void* stream) {
  return moe_gemm_dgrad_gateup_to(dg, du, 0, w1, w3, offs, E, R, H, I, dxp, nullptr, stream);
}

extern "C" int moe_gemm_wgrad(const uint16_t* a_, const uint16_t* b_, const int32_t* offs, int64_t E,
                              int64_t R, int64_t M, int64_t N, void* dw, int dw_dtype,
                              int accumulate, void* stream) {
  WgradArgs w{};
  w.n = 1;
  if (int rc = wgrad_args(w.p[0], a_, b_, offs, E, R, M, N, dw, dw_dtype, accumulate)) return rc;
  return run_wgrad(w, dw_dtype, stream);
}
