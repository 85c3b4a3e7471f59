// The grouped products over an expert's rows (gate/up, down and their input gradients) for launches of few tiles.
//
// With a tile or two to a compute unit nothing but a tile's own length counts: a trip to memory for the offsets, one for the
// first k-tile, the contraction, the epilogue.  Hence small tiles of 64 x 128 (gate and up: 64 columns of each), four waves
// of 32 rows x 64 columns, and k-tiles of 64 that go straight into a ring of three LDS stages, two on their way;
// two such workgroups share a compute unit.  A k-tile takes 1050 cycles alone and 700 shared (576 of LDS traffic: 24 KB
// arriving, 48 KB read), where the eight waves of a 128 x 256 tile take 2000 and have their loads one k-tile ahead.
// 1024 rows of 8 experts, 1024 <-> 512, gate/up, down, dgrad-down and dgrad-gate/up: 18.6, 10.6, 22.0, 17.0 us in
// tiles of 128 x 256, 11.8, 6.0, 13.3, 10.7 here; 768 rows of 12 experts, 1416 <-> 568: 25.8, 12.8, 29.7, 20.5 and 17.6,
// 10.6, 18.5, 15.2.  (64 x 128 in five stages, one workgroup to a compute unit: 12.6, 6.7, 13.9, 11.9; 128 x 128 in
// three: 14.2, 7.9, 17.5, 13.7; the next k-tile's first fragments read before the last products: 12.2, 6.5, 13.6, 11.0.)
#include <cmath>

#include "row_ring.h"

namespace {

constexpr int MAX_E = 2 * MOE_WAVE;

// A lane's experts `lane` and `lane + 64`: their rows, and the row tiles up to and including theirs.
struct Experts {
  int first[2], end[2], upto[2], total;
  __device__ __forceinline__ void init(const int32_t* offs, int E, int bm) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int e = h * MOE_WAVE + lane_id();
      first[h] = e < E ? offs[e] : 0;
      end[h] = e < E ? offs[e + 1] : 0;
    }
    total = 0;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      upto[h] = total + wave_inclusive((end[h] - first[h] + bm - 1) / bm);
      total = read_lane(upto[h], MOE_WAVE - 1);
    }
  }
};

template <int MODE, bool BLK, int FM, bool TO, bool FROM>
__global__ __launch_bounds__(256, 2) void ring_rows_kernel(const GemmArgs p) {
  using O = RingTile<MODE, FM, 4>;
  constexpr int BM = O::BM;
  extern __shared__ __attribute__((aligned(1024))) char ring[];
  // ---- this workgroup's tile: XCD x takes the x-th contiguous eighth of the list, in which the row tiles of an expert
  // over the same columns follow each other
  Experts ex;
  ex.init(p.offs, p.E, BM);
  const int total = ex.total * p.n_tiles, x = blockIdx.x & 7, j = blockIdx.x >> 3, q = total >> 3, r = total & 7;
  if (j >= q + (x < r ? 1 : 0)) return;
  const int tile = x * q + (x < r ? x : r) + j;
  int e = __popcll(__ballot(ex.upto[0] * p.n_tiles <= tile));
  const bool high = e == MOE_WAVE;
  if (high) e += __popcll(__ballot(ex.upto[1] * p.n_tiles <= tile));
  const int l = e & (MOE_WAVE - 1);
  const int first = read_lane(high ? ex.first[1] : ex.first[0], l), row_end = read_lane(high ? ex.end[1] : ex.end[0], l);
  const int nt = (row_end - first + BM - 1) / BM;
  const int in = tile - (read_lane(high ? ex.upto[1] : ex.upto[0], l) - nt) * p.n_tiles;
  ring_tile<MODE, BLK, FM, 4, TO, FROM>(p, ring, e, first, row_end, in % nt * BM, in / nt * O::BNC);
}

// Tiles side by side.  (dgrad-down's sums cover the columns in steps of 256)
template <int MODE>
int columns(int N) {
  constexpr int BNC = RingTile<MODE, 1, 4>::BNC;
  return MODE == DGRAD_DOWN ? (N + 255) / 256 * 2 : (N + BNC - 1) / BNC;
}

// Launches of at most `most` tiles (by the bound that R and E give), or of any number.
template <int MODE, bool BLK, int FM, bool TO, bool FROM>
bool launch(GemmArgs a, long long most, bool any, hipStream_t s, int* rc) {
  using O = RingTile<MODE, FM, 4>;
  a.n_tiles = columns<MODE>(a.N);
  const long long tiles = ((a.R + O::BM - 1) / O::BM + (long long)a.E) * a.n_tiles;
  if (tiles > (any ? 0x7fffff00ll : most)) return false;
  const auto kern = ring_rows_kernel<MODE, BLK, FM, TO, FROM>;
  static bool attr_done[MOE_MAX_DEVICES];
  const int dev = moe_current_device();
  if (!attr_done[dev]) {
    const hipError_t err = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, O::LDS);
    if (err != hipSuccess) return *rc = (int)err, true;
    attr_done[dev] = true;
  }
  hipLaunchKernelGGL(kern, dim3((unsigned)((tiles + 7) / 8 * 8)), dim3(256), O::LDS, s, a);
  return *rc = moe_launch_status(), true;
}

// Whether tiles of 64 rows are the faster ones where there are more of them than run at once.  With few rows an expert the
// weights bound a launch, larger tiles are padding and an expert has one of them: their launch lasts as many whole rounds
// of one to a compute unit as E experts' tiles fill.  Tiles of 64 rows, two to a compute unit, are dealt out as they end
// and take their share of a round each, about 0.8 of it where the contraction is short and 1 at 4096, and from some 30
// rows an expert on more and more experts have two (by chance and by the router).  Over 11 layers, 4 to 128 experts,
// 8 to 500 rows an expert dealt evenly and unevenly, this takes 2.2 % longer than the faster one everywhere, 40 rows an
// expert as the line 3.3 %.  Larger tiles -> this, us: 24 experts, 3000 <-> 1200, 50 rows each (1.1 rounds) down 61 -> 48,
// dgrad-gate/up 99 -> 84; 48 experts, 1536 <-> 640, 50 rows (1.1) 30 -> 22, 50 -> 40; 64 experts, 2048 <-> 1024 (2 rounds) 31 rows
// down 55 -> 49, 50 rows, not taken, gate/up 154 -> 164, dgrad-gate/up 107 -> 116; 16 experts, 4096 <-> 2048, 37 rows (1
// round), not taken, gate/up 89 -> 95, dgrad-gate/up 92 -> 99.  What it gets wrong: 16 experts, 2880 <-> 1440, 32 rows, gate/up
// 45 -> 48; 32 experts, 2048 <-> 1024, 50 rows, down takes 33 and could take 28; 128 experts, 1024 <-> 256, 50 rows dealt
// unevenly, gate/up takes 40 and could take 27.
template <int MODE>
bool small_tiles_pay(const GemmArgs& a) {
  constexpr int LARGE = MODE == GATEUP ? 128 : 256, SMALL = MODE == GATEUP ? 64 : 128;  // columns of a tile
  const double cus = moe_compute_units(), rows = (double)a.R / a.E, k = (double)a.K * (MODE == DGRAD_GATEUP ? 2 : 1);
  if (rows > 80) return false;
  const double second = rows > 30 ? (rows - 30) / 40 : 0;
  const double large = std::ceil(a.E * (double)((a.N + LARGE - 1) / LARGE) / cus);
  return a.E * (double)((a.N + SMALL - 1) / SMALL) / (2 * cus) * (1 + second) * (0.75 + 0.07 * k / 1024) < large;
}

// Up to two tiles for each compute unit, all resident at once.  (Tiles of 64 rows, this and the kernels of larger tiles in
// us: gate/up 320, 14.8 and 19.2; 512, 18.0 and 19.2; 576, 23.3 and 20.5; dgrad-down 288, 18.1 and 23.8; 404, 19.7 and
// 24.8; 544, 29.2 and 25.3.)
// Down and dgrad-gate/up, whose epilogues are short, have tiles of 128 rows and two stages for what is too much for 64
// rows (tiles of 128 rows; down and dgrad-gate/up us: 320 12.4, 19.8 -> 11.2, 17.6; 440 14.5, 22.6 -> 12.5, 19.6; 576
// 19.0, 29.2 -> 19.5, 31.8).
// The bound has a tile too many for every other expert.  Past it, gate/up and dgrad-down are taken all the same where their tiles
// are expected to fit (with room for a twentieth more: unless a router deals evenly there are more, and a second round of a few tiles
// takes as long as the first); so are, where experts have 64 rows, launches in tiles of 128 whose contraction is at most 1280, gate/up's,
// whose larger kernels have less LDS traffic in tiles of 128 x 256, 640 (1024: 18.6 -> 16.8 us by itself, but a forward pass of 2048
// tokens of 8 experts 45.3 -> 46.2), dgrad-down's, whose narrow results larger tiles pad no more, 768 (17836 rows of 12, 1024 <-> 192,
// not taken, 24.9 -> 26.5), or at most 320 and two rounds: there a tile's end is as long as its contraction, and two workgroups to a
// compute unit cover each other's.  With fewer rows an expert the rule behind is the better one (240 rows of 64, 320 <-> 1664,
// dgrad-down, 8.0 -> 11.1).  Before -> this, us: 6492 rows of 8 experts, 256 <-> 576, gate/up 16.2 -> 9.8; 18388 of 64, 576 <->
// 192, down 18.4 -> 12.1; 3784 of 16, 384 <-> 896, dgrad-down 16.3 -> 12.0 (in tiles of 64).  Of 472 launches of 300 drawn layers
// with a launch past the bound, weights cold, gate/up take 0.94, down 0.955, dgrad-down 0.96 and dgrad-gate/up 0.985 of the time in the
// mean, one in thirty is slower by more than 3 % (up to 1.10, by heavy experts).
template <int MODE, bool BLK, bool TO = false, bool FROM = false>
bool choose(const GemmArgs& a, int forced, hipStream_t s, int* rc) {
  const long long slots = 2ll * moe_compute_units();
  if (forced == 128) return launch<MODE, BLK, 2, TO, FROM>(a, slots, true, s, rc);
  if (launch<MODE, BLK, 1, TO, FROM>(a, slots, forced != 0, s, rc)) return true;
  constexpr bool FUSED = MODE == GATEUP || MODE == DGRAD_DOWN;
  if (!FUSED && launch<MODE, BLK, 2, TO, FROM>(a, slots, false, s, rc)) return true;
  constexpr int LONGEST = MODE == GATEUP ? 640 : MODE == DGRAD_DOWN ? 768 : 1280;
  const double cols = columns<MODE>(a.N), k = (double)a.K * (MODE == DGRAD_GATEUP ? 2 : 1);
  const double most = 0.95 * slots;
  if (FUSED && moe_expected_tiles(a.R, a.E, 64) * cols <= most) return launch<MODE, BLK, 1, TO, FROM>(a, slots, true, s, rc);
  const double tall = moe_expected_tiles(a.R, a.E, 128) * cols;
  if (a.R >= 64ll * a.E &&
      ((tall <= most && k <= LONGEST) || (tall <= 2 * most && k <= 320 && MODE != DGRAD_GATEUP)))
    return launch<MODE, BLK, 2, TO, FROM>(a, slots, true, s, rc);
  return small_tiles_pay<MODE>(a) && launch<MODE, BLK, 1, TO, FROM>(a, slots, true, s, rc);
}

}  // namespace

bool moe_ring_rows(Mode mode, bool blocked, const GemmArgs& a, int forced, hipStream_t s, int* rc) {
  if (a.E > MAX_E) return false;
  switch (mode) {
    case GATEUP:
      if (blocked) return a.row_from ? choose<GATEUP, true, false, true>(a, forced, s, rc) : choose<GATEUP, true>(a, forced, s, rc);
      if (a.C0) return false;  // (g and u in rows: not here)
      return a.row_from ? choose<GATEUP, false, false, true>(a, forced, s, rc) : choose<GATEUP, false>(a, forced, s, rc);
    case DOWN: return a.row_map ? choose<DOWN, false, true>(a, forced, s, rc) : choose<DOWN, false>(a, forced, s, rc);
    case DGRAD_DOWN:
      if (!blocked) return false;
      return a.row_from ? choose<DGRAD_DOWN, true, false, true>(a, forced, s, rc) : choose<DGRAD_DOWN, true>(a, forced, s, rc);
    default: return a.row_map ? choose<DGRAD_GATEUP, false, true>(a, forced, s, rc) : choose<DGRAD_GATEUP, false>(a, forced, s, rc);
  }
}
