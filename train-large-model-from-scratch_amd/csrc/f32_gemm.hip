// Grouped (per-expert, ragged) GEMMs of the fp32 path on the matrix cores, and what is fused into them: large ones in
// six bf16 products for one of fp32 (f32_split.h says what bounds those), the others with v_mfma_f32_32x32x2_f32 (fp32 operands,
// fp32 accumulation).
//
// An fp32 MFMA takes 64 cycles for 2048 multiply-adds, sixteen times as long per flop as a bf16 one, so
// that neither LDS nor HBM bounds the kernels of fp32 products: what does is how evenly the chip's matrix pipes are
// loaded and how much of the time they wait for a wave's own loads, barriers and address arithmetic.
// Hence small workgroups (four waves), several of them on a compute unit, k-tiles requested at least two
// iterations before their use, one barrier per iteration that leaves global loads in flight, output tiles of a quarter
// of the size where the last round of tiles would leave compute units empty, and few launches: gate and up share
// one (and with it their tiles), the two halves of the input gradient another, the three weight gradients a third.
#include <cmath>

#include "f32_split.h"

namespace {

constexpr int NT = 256;                    // threads
// Operand tiles of ROWS x TK.  Of each group of eight k values the lower half of a wave multiplies the first
// four and the upper half the others (MFMA j takes k = j and j + 4; any pairing will do as long as both operands use
// the same), so that an operand that lies k-contiguous in LDS is read 16 bytes at a time.
//
// KCont: element (r, k) at base[r * ld + k]; LDS [ROWS][TK + 4], the padding keeps 16-byte reads of 32 rows
//        free of bank conflicts.
// RCont: element (r, k) at base[k * ld + r]; LDS [TK][ROWS + 4], read a value at a time.
template <int ROWS, int TK>
struct KCont {
  static constexpr int LD = TK + 4, ELEMS = ROWS * LD;
  static constexpr int CPR = TK / 4, STEP = NT / CPR, CH = ROWS * CPR / NT;
  static_assert(ROWS * CPR % NT == 0, "loader shape");
  unsigned voff[CH];
  int kc, at;
  // Row of the tile that this thread's chunk i is of.  (TK = 16: a group of eight lanes writes two rows, which lie
  // half the banks apart when they are four rows apart.)
  static __device__ __forceinline__ int row(int i) {
    const int q = threadIdx.x / CPR;
    return (CPR == 4 ? (q & ~7) | (q & 1) << 2 | (q >> 1 & 3) : q) + i * STEP;
  }
  __device__ __forceinline__ void init(int ld, int rows) {  // rows: of the tile that exist
    const int r = row(0);
    kc = threadIdx.x % CPR * 4;
    at = r * LD + kc;
#pragma unroll
    for (int i = 0; i < CH; ++i) voff[i] = r + i * STEP < rows ? (unsigned)((r + i * STEP) * ld + kc) * 4u : OUTSIDE;
  }
  static __device__ __forceinline__ long long k_elems(int k0, int) { return k0; }
  __device__ __forceinline__ f32x4 load(int i, __amdgpu_buffer_rsrc_t rs, int k_left) const {
    return window_load(rs, kc < k_left ? voff[i] : OUTSIDE);  // (K % 4 == 0)
  }
  __device__ __forceinline__ void store(int i, float* lds, f32x4 v) const {
    *reinterpret_cast<f32x4*>(lds + at + i * STEP * LD) = v;
  }
  static __device__ __forceinline__ f32x4 frag(const float* lds, int row0, int c) {
    const int lane = threadIdx.x & 63;
    return *reinterpret_cast<const f32x4*>(lds + (row0 + (lane & 31)) * LD + c * 8 + (lane >> 5) * 4);
  }
};
template <int ROWS, int TK>
struct RCont {
  static constexpr int LD = ROWS + 4, ELEMS = TK * LD;
  static constexpr int CPK = ROWS / 4, STEP = NT / CPK, CH = TK * CPK / NT;
  static_assert(TK * CPK % NT == 0, "loader shape");
  unsigned voff[CH];
  int kk, at;
  __device__ __forceinline__ void init(int ld, int rows) {
    const int r = threadIdx.x % CPK * 4;
    kk = threadIdx.x / CPK;
    at = kk * LD + r;
#pragma unroll
    for (int i = 0; i < CH; ++i) voff[i] = r < rows ? (unsigned)((kk + i * STEP) * ld + r) * 4u : OUTSIDE;  // (rows % 4 == 0)
  }
  static __device__ __forceinline__ long long k_elems(int k0, int ld) { return (long long)k0 * ld; }
  __device__ __forceinline__ f32x4 load(int i, __amdgpu_buffer_rsrc_t rs, int k_left) const {
    return window_load(rs, kk + i * STEP < k_left ? voff[i] : OUTSIDE);
  }
  __device__ __forceinline__ void store(int i, float* lds, f32x4 v) const {
    *reinterpret_cast<f32x4*>(lds + at + i * STEP * LD) = v;
  }
  static __device__ __forceinline__ f32x4 frag(const float* lds, int row0, int c) {
    const int lane = threadIdx.x & 63;
    const float* p = lds + (c * 8 + (lane >> 5) * 4) * LD + row0 + (lane & 31);
    return f32x4{p[0], p[LD], p[2 * LD], p[3 * LD]};
  }
};

// An output tile of BM x BN over k-tiles of TK.  The four waves are WM x WN x WK: each has BM/WM x BN/WN of it as
// NM x NN blocks of 32 x 32, and one of WK equal shares of every k-tile (WK > 1: fold() adds the shares up).
// PF: k-tiles held in registers on their way to LDS.
template <int BM_, int BN_, int TK_, int WM_, int WN_, int PF_>
struct Shape {
  static constexpr int BM = BM_, BN = BN_, TK = TK_, WM = WM_, WN = WN_, WK = 4 / (WM * WN), PF = PF_;
  static constexpr int NM = BM / WM / 32, NN = BN / WN / 32, CK = TK / 8 / WK;  // CK: groups of eight k values per wave
  static constexpr int WAVES = NM * NN > 1 ? 3 : 4;  // per SIMD, at least
  static_assert(WM * WN * WK == 4 && NM > 0 && NN > 0 && CK > 0 && PF % 2 == 0, "shape");
};

// The k loop: acc = A-tile x B-tile over `n` > 0 k-tiles.  k-tile t is requested (`load`) while t - 1 - PF is
// multiplied, written to LDS (two stages) while t - 1 is.  The operands go into the MFMA swapped: a lane ends up with row
// lane % 32 of a block and four consecutive columns per group of four registers (columns 8g + 4*(lane/32) .. +3).
template <typename S, typename OpA, typename OpB>
struct Loop {
  static constexpr int CH = OpA::CH + OpB::CH, STAGES = 2 * (OpA::ELEMS + OpB::ELEMS);
  static constexpr int LDS_FLOATS = S::WK > 1 && STAGES < 4 * 1024 ? 4 * 1024 : STAGES;
  typedef f32x16 Acc[S::NM][S::NN];
  struct Stage {
    f32x4 v[CH];
  };
  template <typename Load>
  static __device__ __forceinline__ void run(float* lds, const OpA& opA, const OpB& opB, int n, bool idle, int wv, Acc& acc,
                                             Load&& load) {
    if (idle) loop(std::true_type{}, lds, opA, opB, n, wv, acc, load);
    else loop(std::false_type{}, lds, opA, opB, n, wv, acc, load);
  }
  // Idle: a wave without rows only moves its share of the operands and meets the barriers
  template <typename Idle, typename Load>
  static __device__ __forceinline__ void loop(Idle, float* lds, const OpA& opA, const OpB& opB, int n, int wv, Acc& acc,
                                              Load& load) {
    const int wk = wv / (S::WM * S::WN), wm = wv / S::WN % S::WM, wn = wv % S::WN;
#pragma unroll
    for (int i = 0; i < S::NM; ++i)
#pragma unroll
      for (int j = 0; j < S::NN; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;
    const auto stage_a = [&](int b) { return lds + b * OpA::ELEMS; };
    const auto stage_b = [&](int b) { return lds + 2 * OpA::ELEMS + b * OpB::ELEMS; };
    const auto put = [&](const Stage& s, int b) {
#pragma unroll
      for (int c = 0; c < CH; ++c) {
        if (c < OpA::CH) opA.store(c, stage_a(b), s.v[c]);
        else opB.store(c - OpA::CH, stage_b(b), s.v[c]);
      }
    };
    Stage st[S::PF];
    const auto step = [&](int t, auto at) {  // at: t modulo PF
      constexpr int b = decltype(at)::value & 1, next = (decltype(at)::value + 1) % S::PF;
      f32x4 fa[S::CK][S::NM], fb[S::CK][S::NN];
      if constexpr (!Idle::value) {
#pragma unroll
        for (int c = 0; c < S::CK; ++c) {
#pragma unroll
          for (int x = 0; x < S::NM; ++x) fa[c][x] = OpA::frag(stage_a(b), (wm * S::NM + x) * 32, wk * S::CK + c);
#pragma unroll
          for (int x = 0; x < S::NN; ++x) fb[c][x] = OpB::frag(stage_b(b), (wn * S::NN + x) * 32, wk * S::CK + c);
        }
      }
      put(st[next], b ^ 1);
      load(t + 1 + S::PF, st[next]);
      if constexpr (!Idle::value) {
#pragma unroll
        for (int c = 0; c < S::CK; ++c)
#pragma unroll
          for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int x = 0; x < S::NM; ++x)
#pragma unroll
              for (int y = 0; y < S::NN; ++y)
                acc[x][y] = __builtin_amdgcn_mfma_f32_32x32x2f32(fb[c][y][j], fa[c][x][j], acc[x][y], 0, 0, 0);
      }
      lds_barrier();
    };
    const auto steps = [&](int t, int count, auto... at) { ((decltype(at)::value < count ? step(t + decltype(at)::value, at) : void()), ...); };
    const auto round = [&](int t, int count) {
      if constexpr (S::PF == 2) steps(t, count, std::integral_constant<int, 0>{}, std::integral_constant<int, 1>{});
      else steps(t, count, std::integral_constant<int, 0>{}, std::integral_constant<int, 1>{},
                 std::integral_constant<int, 2>{}, std::integral_constant<int, 3>{});
    };
    static_assert(S::PF == 2 || S::PF == 4, "rounds of two or four");
#pragma unroll
    for (int i = 0; i < S::PF; ++i) load(i, st[i]);
    put(st[0], 0);
    load(S::PF, st[0]);
    lds_barrier();
    int t = 0;
    for (; t + S::PF <= n; t += S::PF) round(t, S::PF);
    if (t < n) round(t, n - t);
  }
  // WK > 1 (one block per wave): wave w gets the sum, in the order of the shares, of group `g` of the block
  static __device__ __forceinline__ void give(float* lds, int wv, const Acc& acc) {
    static_assert(S::WK == 4 && S::NM == 1 && S::NN == 1, "one block, four shares");
    f32x4* x = reinterpret_cast<f32x4*>(lds);
#pragma unroll
    for (int g = 0; g < 4; ++g) x[(wv * 4 + g) * 64 + (threadIdx.x & 63)] = quad(acc[0][0], g);
    lds_barrier();
  }
  static __device__ __forceinline__ f32x4 taken(const float* lds, int g) {
    const f32x4* x = reinterpret_cast<const f32x4*>(lds) + g * 64 + (threadIdx.x & 63);
    return ((x[0] + x[4 * 64]) + x[8 * 64]) + x[12 * 64];
  }
  static __device__ __forceinline__ f32x4 quad(const f32x16& a, int g) {
    return f32x4{a[4 * g], a[4 * g + 1], a[4 * g + 2], a[4 * g + 3]};
  }
};

struct RowsArgs {
  const float *A0, *A1, *B0, *B1;  // A [R, K], B one stack of [E][N][K] or [E][K][N]; the second of each: see the modes
  const float *X0, *X1;            // SwiGLU backward: g and u [R, N]
  float *C0, *C1, *C2;             // [R, N]
  const int32_t* offs;
  int E, R, N, K, accumulate;
};

// PLAIN_T  C0 (+)= A0 B0^T, B0 [N][K]
// PLAIN_N  C0 (+)= A0 B0, B0 [K][N]
// GATEUP   g = A0 B0^T, u = A0 B1^T, both [N][K], half a tile of columns each: two waves hold g, two u of the same
//          columns; C2 = silu(g) * u, and C0 = g, C1 = u unless they are null
// DOWN_BWD d = A0 B0 as PLAIN_N; C0 = dg = d * u * silu'(g), C1 = du = d * silu(g)
// GATEUP_BWD C0 = A0 B0 + A1 B1 as PLAIN_N, one after the other
enum Mode { PLAIN_T, PLAIN_N, GATEUP, DOWN_BWD, GATEUP_BWD };

__device__ __forceinline__ int expert_rows(const RowsArgs& p, int e, int& first) {
  first = 0;
  if (e >= p.E) return 0;
  const int b = p.offs[e], n = p.offs[e + 1] - b;
  first = b;
  return n <= 0 || b < 0 || n > p.R - b ? 0 : n;  // (empty, or offsets that no dispatch would produce)
}


__device__ __forceinline__ float sigmoid_f32(float x) { return 1.f / (1.f + expf(-x)); }

// Which tile a workgroup computes.  The hardware hands workgroup b to XCD b % 8, each with an L2 of its own: XCD x takes
// the x-th contiguous eighth of the list, whose workgroups share a few row tiles and one or two experts' weights
// there.  The tiles after the last full round of one per compute unit are cut into four each, unless they nearly fill
// another round: 4.25 rounds of tiles then take the time of about 4.25 and not of 5.  (4096 rows of 8 experts, 1024 <-> 512:
// 89 us in whole tiles, 79 with the last quarter round cut; a chip's worth of small tiles keeps more launches of fewer
// tiles than compute units busy, too.)
struct Job {
  int tile, part;  // part: 0..3 of the tile, -1: all of it; tile < 0: none
};
// chunk > 0: the list is dealt to the XCDs by so many tiles instead (what is left after the last full deal one by one).
__device__ __forceinline__ Job job_of(int tiles, int cus, int most, int chunk = 0) {
  const int rest = tiles % cus, cut = rest * 4 <= most ? rest : 0, whole = tiles - cut;
  const int x = blockIdx.x & 7;
  int j = blockIdx.x >> 3;
  if (chunk > 0) {
    const int b = blockIdx.x, at = b - (whole + 7) / 8 * 8;
    if (j < whole / (8 * chunk) * chunk) return Job{(j / chunk * 8 + x) * chunk + j % chunk, -1};
    if (b < whole) return Job{b, -1};
    return at >= 0 && at < cut * 4 ? Job{whole + at / 4, at % 4} : Job{-1, 0};
  }
  const int q = whole / 8, r = whole % 8, mine = q + (x < r ? 1 : 0);
  if (j < mine) return Job{x * q + (x < r ? x : r) + j, -1};
  j -= mine;
  const int q4 = cut * 4 / 8, r4 = cut * 4 % 8;
  if (j >= q4 + (x < r4 ? 1 : 0)) return Job{-1, 0};  // (the grid is sized for the most there can be)
  const int at = x * q4 + (x < r4 ? x : r4) + j;
  return Job{whole + at / 4, at % 4};
}
// Workgroups for at most `tiles` tiles: each XCD may round its two shares up.
unsigned grid_of(int64_t tiles, int64_t cus) { return (unsigned)((tiles + 3 * (cus * 3 / 4) + 7) / 8 * 8 + 16); }

// How many quarters the split tiles' last round may be cut into: one workgroup is resident on a compute unit, and two rounds of quarters
// take less time than one of whole tiles for contractions past about 900 (128 tiles, operands by turns k-contiguous and not:
// 640 29 us whole; 768 33 to 36 in quarters, where whole tiles would take 33; 1024 40 to 44, and 42 to 43; 2048 69 to 73, and 78).
__host__ __device__ __forceinline__ int split_cut(int k, int cus) { return k > 900 ? 2 * cus : cus; }

template <int MODE>
constexpr bool b_kcont = MODE == PLAIN_T || MODE == GATEUP;
template <int MODE, typename S>
using RowsB = typename std::conditional<b_kcont<MODE>, KCont<S::BN, S::TK>, RCont<S::BN, S::TK>>::type;
template <int MODE, typename S>
using RowsLoop = Loop<S, KCont<S::BM, S::TK>, RowsB<MODE, S>>;
constexpr __host__ __device__ int larger(int a, int b) { return a > b ? a : b; }

// What becomes of four consecutive columns of one row (GATEUP: v of g and u of u; else u is not used)
template <int MODE>
__device__ __forceinline__ void rows_result(const RowsArgs& p, int m, int row_end, int n, f32x4 v, f32x4 u) {
  constexpr bool DUAL = MODE == GATEUP;
  if (m >= row_end || n >= p.N) return;  // (N % 4 == 0: the four columns are inside or outside together)
  const long long at = (long long)m * p.N + n;
  if constexpr (DUAL) {
    f32x4 a;
#pragma unroll
    for (int c = 0; c < 4; ++c) a[c] = v[c] * sigmoid_f32(v[c]) * u[c];
    if (p.C0) {
      *reinterpret_cast<f32x4*>(p.C0 + at) = v;
      *reinterpret_cast<f32x4*>(p.C1 + at) = u;
    }
    *reinterpret_cast<f32x4*>(p.C2 + at) = a;
  } else if constexpr (MODE == DOWN_BWD) {  // silu'(g) = s * (1 + g * (1 - s)), s = sigmoid(g)
    const f32x4 gv = *reinterpret_cast<const f32x4*>(p.X0 + at), uv = *reinterpret_cast<const f32x4*>(p.X1 + at);
    f32x4 dg, du;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const float s = sigmoid_f32(gv[c]);
      dg[c] = v[c] * uv[c] * (s * (1.f + gv[c] * (1.f - s)));
      du[c] = v[c] * (gv[c] * s);
    }
    *reinterpret_cast<f32x4*>(p.C0 + at) = dg;
    *reinterpret_cast<f32x4*>(p.C1 + at) = du;
  } else {
    if (p.accumulate) v += *reinterpret_cast<const f32x4*>(p.C0 + at);
    *reinterpret_cast<f32x4*>(p.C0 + at) = v;
  }
}

// The tile of Shape S at rows row0.. (of the expert's up to row_end), columns n0..
template <int MODE, typename S>
__device__ __forceinline__ void rows_tile(const RowsArgs& p, float* lds, int e, int row0, int row_end, int n0) {
  constexpr bool B_KCONT = b_kcont<MODE>, DUAL = MODE == GATEUP;
  using OpA = KCont<S::BM, S::TK>;
  using OpB = RowsB<MODE, S>;
  using L = RowsLoop<MODE, S>;
  const int lane = threadIdx.x & 63, wv = uniform((int)(threadIdx.x >> 6));
  const int ldb = B_KCONT ? p.K : p.N;
  OpA opA;
  OpB opB;
  opA.init(p.K, row_end - row0);
  opB.init(ldb, p.N - n0);
  // GATEUP: each 32 columns of the product are 16 of g and 16 of u, so that a lane holds both of a place
  const auto is_up = [&](int c) {  // (the same for a whole wave)
    if constexpr (DUAL) {
      static_assert(16 % (64 / OpB::CPR) == 0, "a wave's chunks lie in 16 rows");
      return ((wv * (64 / OpB::CPR) + c * OpB::STEP) & 16) != 0;
    }
    return false;
  };
  if constexpr (DUAL) {
#pragma unroll
    for (int i = 0; i < OpB::CH; ++i) {
      const int rr = OpB::row(i), r = rr / 32 * 16 + (rr & 15);
      opB.voff[i] = r < p.N - n0 ? (unsigned)(r * p.K + opB.kc) * 4u : OUTSIDE;
    }
  }
  const long long wofs = (long long)e * p.N * p.K + (long long)n0 * (B_KCONT ? p.K : 1);
  const float *A0 = p.A0 + (long long)row0 * p.K, *B0 = p.B0 + wofs;
  const float *A1 = p.A1 + (long long)row0 * p.K, *B1 = p.B1 + wofs;  // (null and unused outside the two-operand modes)
  const int per_seg = (p.K + S::TK - 1) / S::TK;
  auto load = [&](int t, typename L::Stage& s) {
    int k0 = t * S::TK;
    const bool second = MODE == GATEUP_BWD && t >= per_seg;
    if (second) k0 -= per_seg * S::TK;
    const __amdgpu_buffer_rsrc_t ra = window(second ? A1 : A0, OpA::k_elems(k0, p.K));
#pragma unroll
    for (int c = 0; c < OpA::CH; ++c) s.v[c] = opA.load(c, ra, p.K - k0);
#pragma unroll
    for (int c = 0; c < OpB::CH; ++c)
      s.v[OpA::CH + c] = opB.load(c, window(second || is_up(c) ? B1 : B0, OpB::k_elems(k0, ldb)), p.K - k0);
  };
  typename L::Acc acc;
  const int wm = wv / S::WN % S::WM, wn = wv % S::WN;
  const bool idle = uniform((int)(row0 + wm * S::NM * 32 >= row_end)) != 0;
  L::run(lds, opA, opB, MODE == GATEUP_BWD ? 2 * per_seg : per_seg, idle, wv, acc, load);

  const auto emit = [&](int m, int n, f32x4 v, f32x4 u) { rows_result<MODE>(p, m, row_end, n, v, u); };
  const int l32 = lane & 31, lh = lane >> 5;
  if constexpr (S::WK > 1) {
    L::give(lds, wv, acc);
    if (DUAL && wv >= 2) return;
    const f32x4 v = L::taken(lds, wv), u = DUAL ? L::taken(lds, wv + 2) : v;
    emit(row0 + l32, n0 + 8 * wv + 4 * lh, v, u);
  } else if (!idle) {
#pragma unroll
    for (int bi = 0; bi < S::NM; ++bi)
#pragma unroll
      for (int bj = 0; bj < S::NN; ++bj)
#pragma unroll
        for (int g = 0; g < (DUAL ? 2 : 4); ++g)
          emit(row0 + (wm * S::NM + bi) * 32 + l32, n0 + (wn * S::NN + bj) * (DUAL ? 16 : 32) + 8 * g + 4 * lh,
               L::quad(acc[bi][bj], g), L::quad(acc[bi][bj], DUAL ? g + 2 : g));
  }
}

// The same on the bf16 matrix cores (f32_split.h)
template <int MODE, typename S>
using SplitB = typename std::conditional<b_kcont<MODE>, SplitInner<S::BN, S::TK, S::NT>, SplitOuter<S::BN, S::TK, S::NT>>::type;
template <int MODE, typename S>
using SplitRowsLoop = SplitLoop<S, SplitInner<S::BM, S::TK, S::NT>, SplitB<MODE, S>>;

template <int MODE, typename S>
__device__ __forceinline__ void split_rows_tile(const RowsArgs& p, char* lds, int e, int row0, int row_end, int n0) {
  constexpr bool B_KCONT = b_kcont<MODE>, DUAL = MODE == GATEUP;
  using OpA = SplitInner<S::BM, S::TK, S::NT>;
  using OpB = SplitB<MODE, S>;
  using L = SplitRowsLoop<MODE, S>;
  const int lane = lane_id(), wv = uniform((int)(threadIdx.x >> 6));
  const int ldb = B_KCONT ? p.K : p.N;
  OpA opA;
  OpB opB;
  opA.init(p.K, row_end - row0);
  opB.init(ldb, p.N - n0);
  bool up[OpB::CH];  // GATEUP: each 32 columns of the product are 16 of g and 16 of u (the same for a whole wave)
#pragma unroll
  for (int i = 0; i < OpB::CH; ++i) up[i] = false;
  if constexpr (DUAL) {
    static_assert(16 % (64 / OpB::CPR) == 0, "a wave's chunks lie in 16 rows");
#pragma unroll
    for (int i = 0; i < OpB::CH; ++i) {
      const int rr = OpB::row(i), r = rr / 32 * 16 + (rr & 15);
      opB.voff[i] = r < p.N - n0 ? (unsigned)(r * p.K + opB.kc) * 4u : OUTSIDE;
      up[i] = ((wv * (64 / OpB::CPR) + i * OpB::STEP) & 16) != 0;
    }
  }
  const long long wofs = (long long)e * p.N * p.K + (long long)n0 * (B_KCONT ? p.K : 1);
  const float *A0 = p.A0 + (long long)row0 * p.K, *B0 = p.B0 + wofs;
  const float *A1 = p.A1 + (long long)row0 * p.K, *B1 = p.B1 + wofs;  // (null and unused outside the two-operand modes)
  const int per_seg = (p.K + S::TK - 1) / S::TK;
  const auto load = [&](int t, typename L::Stage& s) __attribute__((always_inline)) {
    int k0 = t * S::TK;
    const bool second = MODE == GATEUP_BWD && t >= per_seg;
    if (second) k0 -= per_seg * S::TK;
    const __amdgpu_buffer_rsrc_t ra = window(second ? A1 : A0, OpA::k_elems(k0, p.K));
#pragma unroll
    for (int c = 0; c < OpA::CH; ++c)
#pragma unroll
      for (int h = 0; h < 2; ++h) s.v[c][h] = opA.load(c, h, ra, p.K - k0);
#pragma unroll
    for (int c = 0; c < OpB::CH; ++c) {
      const __amdgpu_buffer_rsrc_t rb = window(second || up[c] ? B1 : B0, OpB::k_elems(k0, ldb));
#pragma unroll
      for (int h = 0; h < 2; ++h) s.v[OpA::CH + c][h] = opB.load(c, h, rb, p.K - k0);
    }
  };
  const int l32 = lane & 31, lh = lane >> 5;
  const auto again = [&](int r0, int c0, int share, f32x16& acc) {  // the block of rows r0.., columns c0.. of the tile
    const int quarter = p.K / 4, k1 = share == 3 ? p.K : (share + 1) * quarter;
    const int c = c0 + l32, col = DUAL ? c / 32 * 16 + (c & 15) : c;
    for (int seg = 0; seg < (MODE == GATEUP_BWD ? 2 : 1); ++seg) {
      const float *A = seg ? A1 : A0, *B = seg || (DUAL && (c & 16)) ? B1 : B0;
      for (int k = share * quarter; k < k1; k += 2)
        acc = __builtin_amdgcn_mfma_f32_32x32x2f32(OpB::value(B, ldb, p.N - n0, k1, col, k + lh),
                                                   OpA::value(A, p.K, row_end - row0, k1, r0 + l32, k + lh), acc, 0, 0, 0);
    }
  };
  typename L::Out out;
  L::run(lds, MODE == GATEUP_BWD ? 2 * per_seg : per_seg, wv, out, load, again);

  const int wn = wv % S::WN, wm = wv / S::WN % S::WM, wk = wv / (S::WN * S::WM);
#pragma unroll
  for (int o = 0; o < S::OWN; ++o) {
    const int item = wk * S::OWN + o, block = item / 2, g = item & 1;
    const int m = row0 + (wm * S::NM + block / S::NN) * 32 + l32, at = wn * S::NN + block % S::NN;
    if constexpr (DUAL) {
      rows_result<MODE>(p, m, row_end, n0 + at * 16 + 8 * g + 4 * lh, out.lo[o], out.hi[o]);
    } else {
      rows_result<MODE>(p, m, row_end, n0 + at * 32 + 8 * g + 4 * lh, out.lo[o], out.lo[o]);
      rows_result<MODE>(p, m, row_end, n0 + at * 32 + 8 * g + 16 + 4 * lh, out.hi[o], out.hi[o]);
    }
  }
}

// Tiles of BM x TN are numbered row tile by row tile (an expert's last one may be short), column tiles fastest.  The
// workgroup's: false if it has none.
template <int BM, int TN>
__device__ __forceinline__ bool rows_job(const RowsArgs& p, int cus, int most, int& e, int& row0, int& row_end, int& n0, int& part) {
  const int lane = threadIdx.x & 63, n_col = (p.N + TN - 1) / TN;
  int tiles = 0;
  for (int e0 = 0; e0 < p.E; e0 += MOE_WAVE) {
    int first;
    const int nt = (expert_rows(p, e0 + lane, first) + BM - 1) / BM;
    tiles += uniform(__shfl(wave_inclusive(nt), MOE_WAVE - 1, MOE_WAVE));
  }
  const Job job = job_of(tiles * n_col, cus, most);
  if (job.tile < 0) return false;
  const int row_tile = job.tile / n_col;
  n0 = job.tile % n_col * TN, e = 0, row0 = 0, row_end = 0, part = job.part;
  for (int e0 = 0, seen = 0; e0 < p.E; e0 += MOE_WAVE) {
    int first;
    const int n = expert_rows(p, e0 + lane, first), nt = (n + BM - 1) / BM, incl = seen + wave_inclusive(nt);
    const unsigned long long past = __ballot(incl > row_tile);
    if (past) {
      const int l = __builtin_ctzll(past);
      e = e0 + l;
      row0 = uniform(__shfl(first + (row_tile - (incl - nt)) * BM, l, MOE_WAVE));
      row_end = uniform(__shfl(first + n, l, MOE_WAVE));
      break;
    }
    seen = uniform(__shfl(incl, MOE_WAVE - 1, MOE_WAVE));
  }
  return true;
}

// S is a whole tile, Q a quarter of one.
template <int MODE, typename S, typename Q>
__global__ __launch_bounds__(NT, S::WAVES) void f32_rows_kernel(const RowsArgs p, int cus) {
  static_assert(S::BM == 2 * Q::BM && S::BN == 2 * Q::BN, "a quarter");
  constexpr int TN = MODE == GATEUP ? S::BN / 2 : S::BN;  // columns of a tile
  __shared__ __align__(16) float lds[larger(RowsLoop<MODE, S>::LDS_FLOATS, RowsLoop<MODE, Q>::LDS_FLOATS)];
  int e, row0, row_end, n0, part;
  if (!rows_job<S::BM, TN>(p, cus, cus * 3, e, row0, row_end, n0, part)) return;
  if (part < 0) {
    rows_tile<MODE, S>(p, lds, e, row0, row_end, n0);
  } else {
    row0 += (part >> 1) * Q::BM;
    n0 += (part & 1) * (TN / 2);
    if (row0 < row_end && n0 < p.N) rows_tile<MODE, Q>(p, lds, e, row0, row_end, n0);
  }
}

template <int MODE, typename S, typename Q>
__global__ __launch_bounds__(S::NT, S::NT / 256) void f32_split_rows_kernel(const RowsArgs p, int cus) {
  static_assert(S::BM == 2 * Q::BM && S::BN == 2 * Q::BN && S::NT == Q::NT, "a quarter");
  constexpr int TN = MODE == GATEUP ? S::BN / 2 : S::BN;  // columns of a tile
  extern __shared__ __align__(16) char split_lds[];
  int e, row0, row_end, n0, part;
  if (!rows_job<S::BM, TN>(p, cus, split_cut(MODE == GATEUP_BWD ? 2 * p.K : p.K, cus), e, row0, row_end, n0, part)) return;
  if (part < 0) {
    split_rows_tile<MODE, S>(p, split_lds, e, row0, row_end, n0);
  } else {
    row0 += (part >> 1) * Q::BM;
    n0 += (part & 1) * (TN / 2);
    if (row0 < row_end && n0 < p.N) split_rows_tile<MODE, Q>(p, split_lds, e, row0, row_end, n0);
  }
}

// Weight gradients: per stack C_e[m, n] (+)= sum over the rows r of expert e of A[r, m] * B[r, n], up to three stacks in
// one launch: the workgroups that an XCD runs side by side walk the rows of a few experts together and find them in its
// L2.  An expert without rows gets zeros (or is left alone when accumulating).
struct F32Stack {
  const float *a, *b;  // [R, M], [R, N]
  float* c;            // [E, M, N]
  int M, N, accumulate;
};
struct WgradArgs {
  F32Stack s[3];
  const int32_t* offs;
  int n, E, R;
};

__device__ __forceinline__ void wgrad_result(const F32Stack& s, float* C, int m, int n, f32x4 v) {
  if (m >= s.M || n >= s.N) return;
  f32x4* dst = reinterpret_cast<f32x4*>(C + (long long)m * s.N + n);
  if (s.accumulate) v += *dst;
  *dst = v;
}

template <typename S>
using WgradLoop = Loop<S, RCont<S::BM, S::TK>, RCont<S::BN, S::TK>>;
template <typename S>
__device__ __forceinline__ void wgrad_tile(const F32Stack& s, float* lds, int e, int b, int end, int m0, int n0) {
  using OpA = RCont<S::BM, S::TK>;
  using OpB = RCont<S::BN, S::TK>;
  using L = WgradLoop<S>;
  const int lane = threadIdx.x & 63, wv = uniform((int)(threadIdx.x >> 6));
  OpA opA;
  OpB opB;
  opA.init(s.M, s.M - m0);
  opB.init(s.N, s.N - n0);
  const float *A = s.a + (long long)b * s.M + m0, *B = s.b + (long long)b * s.N + n0;
  auto load = [&](int t, typename L::Stage& st) {
    const int left = end - b - t * S::TK;
    const __amdgpu_buffer_rsrc_t ra = window(A, OpA::k_elems(t * S::TK, s.M)), rb = window(B, OpB::k_elems(t * S::TK, s.N));
#pragma unroll
    for (int c = 0; c < OpA::CH; ++c) st.v[c] = opA.load(c, ra, left);
#pragma unroll
    for (int c = 0; c < OpB::CH; ++c) st.v[OpA::CH + c] = opB.load(c, rb, left);
  };
  typename L::Acc acc;
  const int n = (end - b + S::TK - 1) / S::TK;  // (without rows: one k-tile of zeros)
  L::run(lds, opA, opB, n > 0 ? n : 1, false, wv, acc, load);
  if (end == b && s.accumulate) return;
  float* C = s.c + (long long)e * s.M * s.N;
  const auto emit = [&](int m, int n, f32x4 v) { wgrad_result(s, C, m, n, v); };
  const int l32 = lane & 31, lh = lane >> 5, wm = wv / S::WN % S::WM, wn = wv % S::WN;
  if constexpr (S::WK > 1) {
    L::give(lds, wv, acc);
    emit(m0 + l32, n0 + 8 * wv + 4 * lh, L::taken(lds, wv));
  } else {
#pragma unroll
    for (int bi = 0; bi < S::NM; ++bi)
#pragma unroll
      for (int bj = 0; bj < S::NN; ++bj)
#pragma unroll
        for (int g = 0; g < 4; ++g)
          emit(m0 + (wm * S::NM + bi) * 32 + l32, n0 + (wn * S::NN + bj) * 32 + 8 * g + 4 * lh, L::quad(acc[bi][bj], g));
  }
}

template <typename S>
using SplitWgradLoop = SplitLoop<S, SplitOuter<S::BM, S::TK, S::NT>, SplitOuter<S::BN, S::TK, S::NT>>;
template <typename S>
__device__ __forceinline__ void split_wgrad_tile(const F32Stack& s, char* lds, int e, int b, int end, int m0, int n0) {
  using OpA = SplitOuter<S::BM, S::TK, S::NT>;
  using OpB = SplitOuter<S::BN, S::TK, S::NT>;
  using L = SplitWgradLoop<S>;
  const int lane = lane_id(), wv = uniform((int)(threadIdx.x >> 6));
  OpA opA;
  OpB opB;
  opA.init(s.M, s.M - m0);
  opB.init(s.N, s.N - n0);
  const float *A = s.a + (long long)b * s.M + m0, *B = s.b + (long long)b * s.N + n0;
  const auto load = [&](int t, typename L::Stage& st) __attribute__((always_inline)) {
    const int left = end - b - t * S::TK;
    const __amdgpu_buffer_rsrc_t ra = window(A, OpA::k_elems(t * S::TK, s.M)), rb = window(B, OpB::k_elems(t * S::TK, s.N));
#pragma unroll
    for (int c = 0; c < OpA::CH; ++c)
#pragma unroll
      for (int h = 0; h < 2; ++h) st.v[c][h] = opA.load(c, h, ra, left);
#pragma unroll
    for (int c = 0; c < OpB::CH; ++c)
#pragma unroll
      for (int h = 0; h < 2; ++h) st.v[OpA::CH + c][h] = opB.load(c, h, rb, left);
  };
  const int l32 = lane & 31, lh = lane >> 5;
  const auto again = [&](int r0, int c0, int share, f32x16& acc) {
    const int quarter = (end - b) / 4, k1 = share == 3 ? end - b : (share + 1) * quarter;
    for (int k = share * quarter; k < k1; k += 2)
      acc = __builtin_amdgcn_mfma_f32_32x32x2f32(OpB::value(B, s.N, s.N - n0, k1, c0 + l32, k + lh),
                                                 OpA::value(A, s.M, s.M - m0, k1, r0 + l32, k + lh), acc, 0, 0, 0);
  };
  typename L::Out out;
  const int n = (end - b + S::TK - 1) / S::TK;  // (without rows: one k-tile of zeros)
  L::run(lds, n > 0 ? n : 1, wv, out, load, again);
  if (end == b && s.accumulate) return;
  float* C = s.c + (long long)e * s.M * s.N;
  const int wn = wv % S::WN, wm = wv / S::WN % S::WM, wk = wv / (S::WN * S::WM);
#pragma unroll
  for (int o = 0; o < S::OWN; ++o) {
    const int item = wk * S::OWN + o, block = item / 2, g = item & 1;
    const int m = m0 + (wm * S::NM + block / S::NN) * 32 + l32, n = n0 + (wn * S::NN + block % S::NN) * 32 + 8 * g + 4 * lh;
    wgrad_result(s, C, m, n, out.lo[o]);
    wgrad_result(s, C, m, n + 16, out.hi[o]);
  }
}

// The e-th largest of up to 64 values >= 0, each lane's own (a lane without one has -1), equal ones in the order of the
// lanes: its lane.  The value bit by bit from the top, by how many are at least as large.  (Every ballot is of all lanes.)
__device__ __forceinline__ int lane_of_rank(int n, int largest, int e) {
  int value = 0;
  for (int bit = 1 << (31 - __builtin_clz(largest | 1)); bit; bit >>= 1)
    if (__builtin_popcountll(__ballot(n >= (value | bit))) > e) value |= bit;
  const unsigned long long same = __ballot(n == value);
  const int before = (int)__builtin_amdgcn_mbcnt_hi((unsigned)(same >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)same, 0));
  const int place = e - __builtin_popcountll(__ballot(n > value));
  return __builtin_ctzll(__ballot(n == value & before == place));
}

// Tiles go stack by stack and expert by expert, an eighth of the list for each XCD, which gives it the tiles of 3/8 of the
// experts.  A tile costs what its expert has rows, so that an XCD with a heavy expert keeps the others waiting: where
// it gets more by that than 1/8 of its share, the tiles go expert by expert, up to 64 experts the largest first,
// and are dealt to all XCDs, an eighth of a stack's at a time.  (Shares with a heavy expert from there on gain: 1/8
// to 3/8 more 1.09 to 1.12 times as fast, more 1.2 to 1.6; below it what dealing costs the L2s is more than it gives,
// 0.93 to 0.98.  4096 rows of 8 experts by Zipf's shares, three stacks of 1024 x 512: 221 -> 111 us; even 107 and 107.)
// DEAL: without it the offsets of all experts are not looked at, which costs a workgroup a trip to memory before it
// can begin (2000 rows of 128 experts, 256 x 256: 32 us without and 40 with).
struct WgradJob {
  int w, e, b, end, m0, n0, part;  // stack w, rows b .. end of expert e; part as in Job
};
template <int BM, int BN, bool DEAL>
__device__ __forceinline__ bool wgrad_job(const WgradArgs& p, int cus, int most, WgradJob& out) {
  int per_e[3], n_col[3], per = 0;
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    n_col[i] = i < p.n ? (p.s[i].N + BN - 1) / BN : 0;
    per_e[i] = i < p.n ? n_col[i] * ((p.s[i].M + BM - 1) / BM) : 0;
    per += per_e[i];
  }
  const auto rows_of = [&](int e, int& first) {  // 0: none, or offsets that no dispatch would produce; -1: no such expert
    first = 0;
    if (e >= p.E) return -1;
    const int b = p.offs[e], end = p.offs[e + 1];
    if (b < 0 || end > p.R || end <= b) return 0;
    first = b;
    return end - b;
  };
  int first = 0, rows = 0;  // DEAL: of the lane's expert
  bool uneven = false;
  if constexpr (DEAL) {
    const int lane = threadIdx.x & 63;
    const auto heavy = [&](int n) { return 64ll * ((long long)n * p.E - p.R) > (long long)p.n * p.E * p.R; };
    rows = rows_of(lane, first);
    uneven = __ballot(heavy(rows)) != 0;
    for (int e0 = MOE_WAVE; e0 < p.E; e0 += MOE_WAVE) {
      int at;
      uneven |= __ballot(heavy(rows_of(e0 + lane, at))) != 0;
    }
  }
  const Job job = job_of(per * p.E, cus, most, uneven ? larger(per_e[0] / 8, 1) : 0);
  if (job.tile < 0) return false;
  int w = 0, nc = n_col[0], pe = per_e[0], tile = uneven ? job.tile % per : job.tile;
  const int share = uneven ? 1 : p.E;  // experts whose tiles of a stack follow each other
#pragma unroll
  for (int i = 1; i < 3; ++i)
    if (w == i - 1 && tile >= per_e[i - 1] * share) {
      tile -= per_e[i - 1] * share;
      w = i, nc = n_col[i], pe = per_e[i];
    }
  int e = uneven ? job.tile / per : tile / pe;
  tile %= pe;
  if (DEAL && p.E <= MOE_WAVE) {
    if (uneven) e = lane_of_rank(rows, p.R, e);
    first = read_lane(first, e);
    rows = read_lane(rows, e);
  } else {
    rows = rows_of(e, first);
  }
  const int b = uniform(first);
  out = WgradJob{w, e, b, b + uniform(rows), tile / nc * BM, tile % nc * BN, job.part};
  return true;
}

template <typename S, typename Q, bool DEAL>
__global__ __launch_bounds__(NT, S::WAVES) void f32_wgrad_kernel(const WgradArgs p, int cus) {
  __shared__ __align__(16) float lds[larger(WgradLoop<S>::LDS_FLOATS, WgradLoop<Q>::LDS_FLOATS)];
  WgradJob j;
  if (!wgrad_job<S::BM, S::BN, DEAL>(p, cus, cus * 3, j)) return;
  const F32Stack s = p.s[j.w];
  if (j.part < 0) {
    wgrad_tile<S>(s, lds, j.e, j.b, j.end, j.m0, j.n0);
  } else {
    j.m0 += (j.part >> 1) * Q::BM;
    j.n0 += (j.part & 1) * Q::BN;
    if (j.m0 < s.M && j.n0 < s.N) wgrad_tile<Q>(s, lds, j.e, j.b, j.end, j.m0, j.n0);
  }
}
template <typename S, typename Q, bool DEAL>
__global__ __launch_bounds__(S::NT, S::NT / 256) void f32_split_wgrad_kernel(const WgradArgs p, int cus) {
  extern __shared__ __align__(16) char split_lds[];
  WgradJob j;
  if (!wgrad_job<S::BM, S::BN, DEAL>(p, cus, split_cut(p.R / p.E, cus), j)) return;
  const F32Stack s = p.s[j.w];
  if (j.part < 0) {
    split_wgrad_tile<S>(s, split_lds, j.e, j.b, j.end, j.m0, j.n0);
  } else {
    j.m0 += (j.part >> 1) * Q::BM;
    j.n0 += (j.part & 1) * Q::BN;
    if (j.m0 < s.M && j.n0 < s.N) split_wgrad_tile<Q>(s, split_lds, j.e, j.b, j.end, j.m0, j.n0);
  }
}

using Small = Shape<64, 64, 32, 2, 2, 2>;    // four of them on a compute unit by their LDS
using Quarter = Shape<32, 32, 32, 1, 1, 4>;  // of Small: the four waves share the contraction
using Large = Shape<128, 128, 16, 2, 2, 2>;  // three by their registers
using LargeQuarter = Shape<64, 64, 16, 2, 2, 2>;

using SplitTile = SplitShape<128, 128, 32, 2, 2, 2>;   // eight waves
using SplitQuarter = SplitShape<64, 64, 64, 1, 2, 4>;

int forced_tile = 0;
template <typename K>
int set_lds(K kern, bool (&done)[MOE_MAX_DEVICES], int bytes) {
  const int dev = moe_current_device();
  if (!done[dev]) {
    const hipError_t err = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    if (err != hipSuccess) return (int)err;
    done[dev] = true;
  }
  return 0;
}
// The large tile has half the operand traffic and LDS reads per flop (32768 rows of 8 experts, 2048 <-> 1024, gate and up: 1.99
// against 2.17 ms, 138 TFLOP/s), but few of them share a compute unit less evenly (8192 rows of 16 experts, 1024 <-> 1024, five
// rounds of large tiles: 335 against 295 us; three rounds: equal): from eight rounds on.  So, too, for weight gradients,
// where a tile takes as long as its expert has rows.  From three to eight rounds the large one is faster by a tenth
// where a router with random weights deals the rows (4096 rows of 8 experts, three stacks of 1024 x 512, three rounds: 120 us
// against 126), and slower where it does not: with logits off by 0.3 from expert to expert 0.90 to 1.03 times as fast on
// average and down to 0.42 (16384 rows of 128 experts, 256 x 128: 220 us against 92), with Zipf's shares 0.67 to 0.81 and
// down to 0.31.  From eight rounds on: 1.04, 1.08 and 1.03 times as fast.  Rounds by the bound, which has a tile for every
// expert: row launches whose experts do not fill half of one stay with the small tile (1020 rows of 128 experts, 2584 <-> 288, down and
// dgrad-gate/up 173, 315 us in large tiles, 105 and 171 in small ones).
bool large_tiles(int64_t tiles128) {
  if (forced_tile) return forced_tile == 128;
  return tiles128 >= 8 * (int64_t)moe_compute_units();
}

// Split tiles (f32_split.h) keep a whole compute unit busy; fp32 ones of 64 x 64 share it.  Both launches' times follow, to 8 %, from
// their tiles and the contraction's length k, us: a round of split tiles `start` + 0.038 k, one of quarters 7 + 0.0115 k; fp32
// tiles 5 + 0.0025 k and, of 256 compute units, `each` + 0.0645 k a thousand.  Split where that is 5 % less, experts fill half a tile
// (weight gradients: have some rows, and tiles for every compute unit, as one heavy expert's would keep few of them), half of what
// is computed is wanted (weight gradients, which have no other remainder: 0.7), and there is work to gain by.  DOWN_BWD, whose
// epilogue reads two more operands, needs more of it.  900 drawn layers, 4 to 128 experts, 64 to 32768 rows, even to skewed, widths
// 256 to 4096 and 128 to 2048: of 4500 launches 1111 are taken, gate/up 1.26, down 1.22, down's input gradient 1.16, gate/up's
// 1.19, weight gradients 1.22 times as fast as in fp32 tiles in the mean, 27 of them slower by more than 3 %.
constexpr int SPLIT = 1;
bool split_pays(double tiles128, double tiles64, double k, double start, double each) {
  const double cus = moe_compute_units(), whole = std::floor(tiles128 / cus), rest = tiles128 - whole * cus;
  const bool cut = rest * 4 <= split_cut((int)k, (int)cus);
  const double split = (cut ? whole : whole + 1) * (start + 0.038 * k) + (cut ? std::ceil(rest * 4 / cus) * (7 + 0.0115 * k) : 0);
  return split < 0.95 * (5 + 0.0025 * k + tiles64 / 1000 * 256 / cus * (each + 0.0645 * k));
}
bool split_rows(Mode mode, int64_t E, int64_t R, int64_t N, int64_t K) {
  if (forced_tile) return forced_tile == SPLIT;
  const auto tiles = [&](int t) { return moe_expected_tiles(R, E, t) * ((N + t - 1) / t); };
  const bool bwd = mode == DOWN_BWD;
  const double work = (double)R * N * K / (1 << 30);
  return R >= 64 * E && K >= (bwd ? 512 : 256) && work >= (bwd ? 1.5 : 1) && R * N * 2 >= tiles(128) * 128 * 128 &&
         split_pays(tiles(128), tiles(64), (double)K, bwd ? 14 : mode == GATEUP ? 8 : 6, bwd ? 11 : mode == GATEUP ? 4.7 : 2.5);
}
bool split_wgrad(int64_t E, int64_t R, int64_t elements, int64_t tiles128, int64_t tiles64) {  // elements, tiles: of all stacks
  if (forced_tile) return forced_tile == SPLIT;
  return R >= 224 * E && tiles128 >= moe_compute_units() && elements >= ((int64_t)1 << 30) / R && 10 * E * elements >= 7 * tiles128 * 128 * 128 &&
         split_pays((double)tiles128, (double)tiles64, (double)R / E, 9, 3.4);
}

int check_rows(int64_t E, int64_t R, int64_t N, int64_t K) {
  for (int64_t width : {N, K})
    if (width <= 0 || width % 4 != 0) return MOE_ERR_SHAPE;
  if (E <= 0 || R < 0) return MOE_ERR_SHAPE;
  if (E > 1024 || R > (int64_t)1 << 30 || N > 65536 || K > 65536) return MOE_ERR_LIMIT;
  if ((R / 64 + E) * ((N + 31) / 32) > 0x70000000ll) return MOE_ERR_LIMIT;
  return 0;
}

template <int MODE>
int launch_rows(RowsArgs a, int64_t E, int64_t R, int64_t N, int64_t K, hipStream_t s) {
  a.E = (int)E, a.R = (int)R, a.N = (int)N, a.K = (int)K;
  const int cus = moe_compute_units();
  const auto tiles = [&](int64_t t) { return (R / t + E) * ((N * (MODE == GATEUP ? 2 : 1) + t - 1) / t); };  // at most
  if (split_rows((Mode)MODE, E, R, N * (MODE == GATEUP ? 2 : 1), K * (MODE == GATEUP_BWD ? 2 : 1))) {
    constexpr int LDS = larger(SplitRowsLoop<MODE, SplitTile>::LDS_BYTES, SplitRowsLoop<MODE, SplitQuarter>::LDS_BYTES);
    static bool done[MOE_MAX_DEVICES];
    const auto kern = f32_split_rows_kernel<MODE, SplitTile, SplitQuarter>;
    if (int rc = set_lds(kern, done, LDS)) return rc;
    hipLaunchKernelGGL(kern, dim3(grid_of(tiles(128), cus)), dim3(SplitTile::NT), LDS, s, a, cus);
    return moe_launch_status();
  }
  if (large_tiles(tiles(128)) && (R >= 64 * E || forced_tile))
    hipLaunchKernelGGL((f32_rows_kernel<MODE, Large, LargeQuarter>), dim3(grid_of(tiles(128), cus)), dim3(NT), 0, s, a, cus);
  else
    hipLaunchKernelGGL((f32_rows_kernel<MODE, Small, Quarter>), dim3(grid_of(tiles(64), cus)), dim3(NT), 0, s, a, cus);
  return moe_launch_status();
}

}  // namespace

extern "C" int moe_f32_gemm_rows(const float* a, const float* b, const int32_t* offs, int64_t E, int64_t R, int64_t N,
                                 int64_t K, int b_k_contiguous, float* c, int accumulate, void* stream) {
  if (int rc = check_rows(E, R, N, K)) return rc;
  if (R == 0) return 0;
  MOE_CHECK_PTR(a);
  MOE_CHECK_PTR(b);
  MOE_CHECK_PTR(c);
  if (!offs) return MOE_ERR_NULL;
  RowsArgs p{};
  p.A0 = a, p.B0 = b, p.C0 = c, p.offs = offs, p.accumulate = accumulate;
  return b_k_contiguous ? launch_rows<PLAIN_T>(p, E, R, N, K, (hipStream_t)stream)
                        : launch_rows<PLAIN_N>(p, E, R, N, K, (hipStream_t)stream);
}

// (g and u null: not stored)
int moe_f32_gateup(const float* xp, const float* w1, const float* w3, const int32_t* offs, int64_t E, int64_t R, int64_t H,
                   int64_t I, float* g, float* u, float* act, void* stream) {
  if (int rc = check_rows(E, R, I, H)) return rc;
  if (R == 0) return 0;
  for (const float* q : {xp, w1, w3, (const float*)act}) MOE_CHECK_PTR(q);
  if (!offs) return MOE_ERR_NULL;
  RowsArgs p{};
  p.A0 = xp, p.B0 = w1, p.B1 = w3, p.C0 = g, p.C1 = u, p.C2 = act, p.offs = offs;
  return launch_rows<GATEUP>(p, E, R, I, H, (hipStream_t)stream);
}

extern "C" int moe_f32_gemm_gateup_swiglu(const float* xp, const float* w1, const float* w3, const int32_t* offs, int64_t E,
                                          int64_t R, int64_t H, int64_t I, float* g, float* u, float* act, void* stream) {
  if (R > 0) {
    MOE_CHECK_PTR(g);
    MOE_CHECK_PTR(u);
  }
  return moe_f32_gateup(xp, w1, w3, offs, E, R, H, I, g, u, act, stream);
}

extern "C" int moe_f32_gemm_down_swiglu_bwd(const float* dyp, const float* w2, const float* g, const float* u,
                                            const int32_t* offs, int64_t E, int64_t R, int64_t H, int64_t I, float* dg,
                                            float* du, void* stream) {
  if (int rc = check_rows(E, R, I, H)) return rc;
  if (R == 0) return 0;
  for (const float* q : {dyp, w2, g, u, (const float*)dg, (const float*)du}) MOE_CHECK_PTR(q);
  if (!offs) return MOE_ERR_NULL;
  RowsArgs p{};
  p.A0 = dyp, p.B0 = w2, p.X0 = g, p.X1 = u, p.C0 = dg, p.C1 = du, p.offs = offs;
  return launch_rows<DOWN_BWD>(p, E, R, I, H, (hipStream_t)stream);
}

extern "C" int moe_f32_gemm_gateup_bwd(const float* dg, const float* du, const float* w1, const float* w3,
                                       const int32_t* offs, int64_t E, int64_t R, int64_t H, int64_t I, float* dxp,
                                       void* stream) {
  if (int rc = check_rows(E, R, H, I)) return rc;
  if (R == 0) return 0;
  for (const float* q : {dg, du, w1, w3, (const float*)dxp}) MOE_CHECK_PTR(q);
  if (!offs) return MOE_ERR_NULL;
  RowsArgs p{};
  p.A0 = dg, p.A1 = du, p.B0 = w1, p.B1 = w3, p.C0 = dxp, p.offs = offs;
  return launch_rows<GATEUP_BWD>(p, E, R, H, I, (hipStream_t)stream);
}

static int wgrads(const F32Stack* s, int n, const int32_t* offs, int64_t E, int64_t R, hipStream_t st) {
  if (n < 0 || n > 3) return MOE_ERR_SHAPE;
  if (n == 0) return 0;
  if (!offs) return MOE_ERR_NULL;
  WgradArgs p{};
  p.offs = offs, p.n = n, p.E = (int)E, p.R = (int)R;
  const auto tiles = [&](int64_t t) {
    int64_t b = 0;
    for (int i = 0; i < n; ++i) b += E * ((s[i].M + t - 1) / t) * ((s[i].N + t - 1) / t);
    return b;
  };
  for (int i = 0; i < n; ++i) {
    if (int rc = check_rows(E, R, s[i].M, s[i].N)) return rc;
    MOE_CHECK_PTR(s[i].c);
    if (R > 0) {
      MOE_CHECK_PTR(s[i].a);
      MOE_CHECK_PTR(s[i].b);
    }
    p.s[i] = s[i];
  }
  if (tiles(64) > 0x70000000ll) return MOE_ERR_LIMIT;
  const int cus = moe_compute_units();
  int64_t elements = 0;
  for (int i = 0; i < n; ++i) elements += s[i].M * (int64_t)s[i].N;
  const bool large = large_tiles(tiles(128)), split = R > 0 && split_wgrad(E, R, elements, tiles(128), tiles(64));
  const auto go = [&](auto deal) {
    constexpr bool DEAL = decltype(deal)::value;
    if (split) {
      constexpr int LDS = larger(SplitWgradLoop<SplitTile>::LDS_BYTES, SplitWgradLoop<SplitQuarter>::LDS_BYTES);
      static bool done[MOE_MAX_DEVICES];
      const auto kern = f32_split_wgrad_kernel<SplitTile, SplitQuarter, DEAL>;
      if (int rc = set_lds(kern, done, LDS)) return rc;
      hipLaunchKernelGGL(kern, dim3(grid_of(tiles(128), cus)), dim3(SplitTile::NT), LDS, st, p, cus);
      return 0;
    }
    if (large)
      hipLaunchKernelGGL((f32_wgrad_kernel<Large, LargeQuarter, DEAL>), dim3(grid_of(tiles(128), cus)), dim3(NT), 0, st, p, cus);
    else
      hipLaunchKernelGGL((f32_wgrad_kernel<Small, Quarter, DEAL>), dim3(grid_of(tiles(64), cus)), dim3(NT), 0, st, p, cus);
    return 0;
  };
  // Times as fast with a look at the offsets as without, up to 64 experts, even loads and loads with a heavy expert: tiles of
  // 64, below 32 rows an expert 0.86 to 0.91, 0.87 to 1.0; 64 to 128 rows 0.94, 1.25; 128 to 256 rows 0.98, 1.35; more 0.99,
  // 1.45.  Tiles of 128: below 64 rows 0.91 to 0.97, 1.03 to 1.13; 64 to 128 rows 0.98, 1.19; more 0.99, 1.3.  Of 128 experts,
  // which are not sorted, 128 rows each: 0.95, 1.1.
  if (R >= (E > MOE_WAVE ? 256 : large || split ? 64 : 128) * E) {
    if (int rc = go(std::true_type{})) return rc;
  } else if (int rc = go(std::false_type{})) {
    return rc;
  }
  return moe_launch_status();
}

// (a null result is not computed)
int moe_f32_wgrads(const float* dg, const float* du, const float* dyp, const float* xp, const float* act, const int32_t* offs,
                   int64_t E, int64_t R, int64_t H, int64_t I, float* dw1, float* dw3, float* dw2, void* stream) {
  if (H > 65536 || I > 65536) return MOE_ERR_LIMIT;
  const F32Stack all[3] = {{dg, xp, dw1, (int)I, (int)H, 0}, {du, xp, dw3, (int)I, (int)H, 0}, {dyp, act, dw2, (int)H, (int)I, 0}};
  F32Stack wanted[3];
  int n = 0;
  for (const F32Stack& s : all)
    if (s.c) wanted[n++] = s;
  return wgrads(wanted, n, offs, E, R, (hipStream_t)stream);
}

extern "C" int moe_f32_gemm_wgrads(const float* dg, const float* du, const float* dyp, const float* xp, const float* act,
                                   const int32_t* offs, int64_t E, int64_t R, int64_t H, int64_t I, float* dw1, float* dw3,
                                   float* dw2, void* stream) {
  for (const float* q : {dw1, dw3, dw2}) MOE_CHECK_PTR(q);
  return moe_f32_wgrads(dg, du, dyp, xp, act, offs, E, R, H, I, dw1, dw3, dw2, stream);
}

extern "C" int moe_f32_gemm_wgrad(const float* a, const float* b, const int32_t* offs, int64_t E, int64_t R, int64_t M,
                                  int64_t N, float* dw, int accumulate, void* stream) {
  if (M > 65536 || N > 65536) return MOE_ERR_LIMIT;
  const F32Stack s{a, b, dw, (int)M, (int)N, accumulate};
  return wgrads(&s, 1, offs, E, R, (hipStream_t)stream);
}

// Test hook: 0 lets every fp32 GEMM launch choose its tile (the default), 64 or 128 forces it, 1 the split tiles.
// Process-wide and not synchronised: for tests, not for production callers.  Returns the previous
// setting.
extern "C" int moe_f32_gemm_force_tile(int t) {
  const int before = forced_tile;
  if (t == 0 || t == SPLIT || t == 64 || t == 128) forced_tile = t;
  return before;
}
