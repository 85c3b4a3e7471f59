// fp32 products on the bf16 matrix cores.  An fp32 value is the sum of three bf16 values, exactly: x = h + m + l, each the nearest to
// what the ones before it leave (8 significant bits each: h leaves 16 at most, m then 7).  bf16 has the
// exponents of fp32, so this holds for each value by itself, whatever the sizes of its neighbours.  Of the nine products of two
// such sums six are added up in the matrix cores' fp32 accumulators, small ones first (lh, hl, mm, mh, hm, hh); the rest
// (ml, lm, ll) is at most 2^-24 of the product, mostly far below.  Six instructions at sixteen times the rate of the fp32 one.
// Relative 2-norm error against fp64, normal operands, 4 / 16 / 64 / 256 / 1024 / 4096 products: 3.2e-8 / 3.4e-8 / 5.5e-8 / 1.2e-7 /
// 2.4e-7 / 5.0e-7 in quarters of a tile, the fp32 instruction 4.0e-8 / 6.0e-8 / 8.5e-8 / 1.5e-7 / 2.9e-7 / 5.7e-7 there.
// (Two fp16 parts need half the products, and lose what a scale shared with larger neighbours takes from small values.)
//
// Values are multiplied by 2^24 on the way, so that no part of one is denormal (the smallest fp32 bit, 2^-149, becomes 2^-125),
// and sums by 2^-48 at the end.  What does not fit then (values from 2^104 on, sums from 2^80 on), infinities and NaN make
// an element's sum infinite or NaN: such an element, and no other, is the fp32 instruction's.
#pragma once
#include "internal.h"
#include "tile_ops.h"

namespace {

constexpr unsigned OUTSIDE = 0xfffffff0u;  // a byte offset that no window reaches: reads as zero

// Operand chunks are read through buffer resources, whose hardware bounds check makes an out-of-range
// chunk a zero without a branch: chunks past the tile's rows or past the end of the contraction get the offset OUTSIDE.
// A window is moved along k by its base, a scalar addition.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t window(const float* base, long long elems) {
  return __builtin_amdgcn_make_buffer_rsrc((void*)(base + elems), 0, 0x7fffffff, 0x00020000);
}
__device__ __forceinline__ f32x4 window_load(__amdgpu_buffer_rsrc_t rs, unsigned off) {
  return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, (int)off, 0, 0));
}

// f(0), f(1), .. f(N - 1) with constants for arguments: what they index stays in registers, however long the code
template <typename F, int... I>
__device__ __forceinline__ void each_of(F&& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void each(F&& f) {
  each_of(f, std::make_integer_sequence<int, N>{});
}

constexpr float SPLIT_SCALE = 16777216.f;  // 2^24, and what undoes it twice
constexpr int SPLIT_EXP = -48;

// The next part of two values, packed; what it leaves of them.
__device__ __forceinline__ uint32_t next_part(float& x, float& y) {
  uint32_t w = pack_bf16x2(x, y);
  asm("" : "+v"(w));  // (the compiler would convert each once more on its own to have it unpacked)
  x -= bf16lo(w), y -= bf16hi(w);
  return w;
}

// Operand tiles of ROWS x TK in LDS, one plane a part.  A thread moves chunks of eight values.
//
// SplitInner: element (r, k) at base[r * ld + k]; a plane is [ROWS][TK], chunks permuted against bank conflicts; a fragment is
//             one 16-byte read.
// SplitOuter: element (r, k) at base[k * ld + r]; a plane is [TK][ROWS], chunks permuted; fragments come
//             through the transposing read (see OpOuter).
template <int ROWS, int TK, int NT>
struct SplitInner {
  static constexpr int PLANE = ROWS * TK * 2, CPR = TK / 8, STEP = NT / CPR, CH = ROWS * CPR / NT;
  static_assert(ROWS * CPR % NT == 0 && (CPR == 4 || CPR == 8), "loader shape");
  unsigned voff[CH];
  int kc;
  static __device__ __forceinline__ int row(int i) { return (int)threadIdx.x / CPR + i * STEP; }
  // The lanes of a 16-byte read meet in groups of four consecutive ones: 0, 3, 5 and 6; 1, 2, 4 and 7; and so on.
  static __device__ __forceinline__ int swizzle(int r) { return CPR == 8 ? r >> 1 & 7 : (r >> 2 ^ r >> 3) & 3; }
  __device__ __forceinline__ void init(int ld, int rows) {  // rows: of the tile that exist
    kc = (int)threadIdx.x % CPR * 8;
#pragma unroll
    for (int i = 0; i < CH; ++i) voff[i] = row(i) < rows ? (unsigned)(row(i) * ld + kc) * 4u : OUTSIDE;
  }
  static __device__ __forceinline__ long long k_elems(int k0, int) { return k0; }
  // half 0, 1: the chunk's first and last four values (K % 4 == 0)
  __device__ __forceinline__ f32x4 load(int i, int half, __amdgpu_buffer_rsrc_t rs, int k_left) const {
    return window_load(rs, kc + half * 4 < k_left && voff[i] != OUTSIDE ? voff[i] + half * 16 : OUTSIDE);
  }
  static __device__ __forceinline__ int place(int i) {  // byte offset of chunk i in a plane
    const int r = row(i), c = (int)threadIdx.x % CPR;
    return r * TK * 2 + ((c ^ swizzle(r)) << 4);
  }
  struct Lane {
    int at, chunk;
  };
  static __device__ __forceinline__ Lane lane(int row0) {
    const int l = lane_id(), r = row0 + (l & 31);
    return Lane{r * TK * 2, (l >> 5) ^ swizzle(r)};
  }
  static __device__ __forceinline__ bf16x8 frag(const char* plane, const Lane& l, int rows, int ks) {
    return *reinterpret_cast<const bf16x8*>(plane + (l.at + rows * TK * 2 + ((l.chunk ^ (ks * 2)) << 4)));
  }
  // one value, anywhere
  static __device__ __forceinline__ float value(const float* base, int ld, int rows, int k_end, int r, int k) {
    return r < rows && k < k_end ? base[(long long)r * ld + k] : 0.f;
  }
};
template <int ROWS, int TK, int NT>
struct SplitOuter {
  static constexpr int PLANE = ROWS * TK * 2, CPL = ROWS / 8, STEP = NT / CPL, CH = TK * CPL / NT;
  static_assert(TK * CPL % NT == 0 && (ROWS == 64 || ROWS == 128), "loader shape");
  unsigned voff[CH];
  int kk, second;
  static __device__ __forceinline__ int line(int i) { return (int)threadIdx.x / CPL + i * STEP; }
  // Half a wave's transposing read covers 64 bytes of each of four lines: they lie in different quarters of the 64 banks.
  static __device__ __forceinline__ int swizzle(int line) { return ROWS == 64 ? 4 * ((line >> 1) & 1) : 4 * (line & 3); }
  __device__ __forceinline__ void init(int ld, int rows) {
    const int r = (int)threadIdx.x % CPL * 8;
    kk = line(0);
    second = r + 4 < rows;
#pragma unroll
    for (int i = 0; i < CH; ++i) voff[i] = r < rows ? (unsigned)(line(i) * ld + r) * 4u : OUTSIDE;  // (rows % 4 == 0)
  }
  static __device__ __forceinline__ long long k_elems(int k0, int ld) { return (long long)k0 * ld; }
  __device__ __forceinline__ f32x4 load(int i, int half, __amdgpu_buffer_rsrc_t rs, int k_left) const {
    return window_load(rs, kk + i * STEP < k_left && voff[i] != OUTSIDE && (half == 0 || second) ? voff[i] + half * 16 : OUTSIDE);
  }
  static __device__ __forceinline__ int place(int i) {
    const int c = (int)threadIdx.x % CPL;
    return line(i) * ROWS * 2 + ((c ^ swizzle(line(i))) << 4);
  }
  struct Lane {
    int at, chunk;
  };
  static __device__ __forceinline__ Lane lane(int row0) {
    const int l = lane_id(), i = l & 15, b = l >> 4;
    return Lane{((b >> 1) * 8 + (i >> 2)) * ROWS * 2 + (i & 1) * 8, (row0 / 8 + 2 * (b & 1) + ((i & 3) >> 1)) ^ swizzle(i >> 2)};
  }
  static __device__ __forceinline__ bf16x8 frag(const char* plane, const Lane& l, int rows, int ks) {
    const char* at = plane + (l.at + ((l.chunk ^ (rows / 8)) << 4) + ks * 16 * ROWS * 2);
    const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)at);
    const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(at + 4 * ROWS * 2));
    typedef __attribute__((ext_vector_type(8))) short s16x8;
    const s16x8 r = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    return __builtin_bit_cast(bf16x8, r);
  }
  static __device__ __forceinline__ float value(const float* base, int ld, int rows, int k_end, int r, int k) {
    return r < rows && k < k_end ? base[(long long)k * ld + r] : 0.f;
  }
};

// An output tile of BM x BN over k-tiles of TK.  The waves are WM x WN x WK: each has BM/WM x BN/WN of it as
// NM x NN blocks of 32 x 32, and one of WK equal shares of every k-tile; the shares are added up at the end.
template <int BM_, int BN_, int TK_, int WM_, int WN_, int WK_>
struct SplitShape {
  static constexpr int BM = BM_, BN = BN_, TK = TK_, WM = WM_, WN = WN_, WK = WK_, NT = 64 * WM * WN * WK;
  static constexpr int NM = BM / WM / 32, NN = BN / WN / 32;
  static_assert(TK == 16 * WK && NM > 0 && NN > 0, "a wave multiplies 16 k values of a k-tile");
  static constexpr int ITEMS = NM * NN * 2, OWN = ITEMS / WK;  // half blocks (groups g and g + 2), and those a wave ends up with
  static_assert(ITEMS % WK == 0, "whole items");
};

template <typename S, typename OpA, typename OpB>
struct SplitLoop {
  static constexpr int CH = OpA::CH + OpB::CH, STAGE = 3 * (OpA::PLANE + OpB::PLANE);
  static constexpr int SWAP = S::WM * S::WN * S::ITEMS * (S::WK - 1) * 2048;
  static constexpr int LDS_BYTES = 2 * STAGE > SWAP ? 2 * STAGE : SWAP;
  static constexpr int PF = 4;  // k-tiles in registers on their way to LDS
  typedef f32x16 Acc[S::NM][S::NN];
  struct Stage {
    f32x4 v[CH][2];
  };
  struct Frags {  // of the parts h, m, l
    bf16x8 a[S::NM][3], b[S::NN][3];
  };
  // What a wave ends up with: item i is the quads g and g + 2 of block (bm, bn), lane l row l % 32 of the block, columns
  // 8 * quad + 4 * (l / 32) .. + 3
  struct Out {
    f32x4 lo[S::OWN], hi[S::OWN];
  };
  static __device__ __forceinline__ f32x4 quad(const f32x16& a, int g) {
    return f32x4{a[4 * g], a[4 * g + 1], a[4 * g + 2], a[4 * g + 3]};
  }

  // acc = A-tile x B-tile over `n` > 0 k-tiles.  While k-tile t is multiplied, the fragments of t + 1 are read, t + 2 is split and
  // written to the LDS stage that t has left, and t + 2 + PF is requested: one barrier a k-tile, and nothing between two of them that
  // waits for one another.  What bounds it is the matrix unit, at the clock that its power leaves, with little to spare: a k-tile of 32
  // has 1536 cycles of products, 700 of LDS writes, 375 of reads and 830 of vector work.  16384 rows of 8 experts, 1024 -> 2 x 512,
  // four tiles of 128 x 128 to a compute unit: 211 us (fp32 instruction: 281), where the products alone take 161 at the rate of a
  // large bf16 product.  224 to 232 registers: h alone is in them twice (below), with all parts twice there would be none left.
  // `load(t, stage)` requests a k-tile, `again(row, column, share, acc)` adds up a quarter of the fp32 products of a
  // block.
  template <typename Load, typename Again>
  static __device__ __forceinline__ void run(char* lds, int n, int wv, Out& out, Load&& load, Again&& again) {
    const int wn = wv % S::WN, wm = wv / S::WN % S::WM, wk = wv / (S::WN * S::WM);
    Acc acc;
#pragma unroll
    for (int i = 0; i < S::NM; ++i)
#pragma unroll
      for (int j = 0; j < S::NN; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;
    const typename OpA::Lane la = OpA::lane(wm * S::NM * 32);
    const typename OpB::Lane lb = OpB::lane(wn * S::NN * 32);
    const auto read_a = [&](int b, Frags& f, int x, int p) {
      f.a[x][p] = OpA::frag(lds + b * STAGE + p * OpA::PLANE, la, x * 32, wk);
    };
    const auto read_b = [&](int b, Frags& f, int x, int p) {
      f.b[x][p] = OpB::frag(lds + b * STAGE + 3 * OpA::PLANE + p * OpB::PLANE, lb, x * 32, wk);
    };
    u32x4 parts[3];
    float x, y;
    // step i of chunk c: a part of two of its values; the last one also writes the chunk
    const auto put = [&](const Stage& s, int b, auto chunk, auto step) __attribute__((always_inline)) {
      constexpr int c = decltype(chunk)::value, q = decltype(step)::value / 3, p = decltype(step)::value % 3;
      if constexpr (p == 0) x = s.v[c][q >> 1][(q & 1) * 2] * SPLIT_SCALE, y = s.v[c][q >> 1][(q & 1) * 2 + 1] * SPLIT_SCALE;
      if constexpr (p < 2) parts[p][q] = next_part(x, y);
      else parts[p][q] = pack_bf16x2(x, y);
      if constexpr (q == 3 && p == 2) {
        char* to = c < OpA::CH ? lds + b * STAGE + OpA::place(c) : lds + b * STAGE + 3 * OpA::PLANE + OpB::place(c - OpA::CH);
#pragma unroll
        for (int i = 0; i < 3; ++i) *reinterpret_cast<u32x4*>(to + i * (c < OpA::CH ? OpA::PLANE : OpB::PLANE)) = parts[i];
      }
    };
    constexpr int STEPS = 12;  // of a chunk
    const auto put_all = [&](const Stage& s, int b) __attribute__((always_inline)) {
      each<CH * STEPS>([&](auto q) __attribute__((always_inline)) {
        put(s, b, std::integral_constant<int, decltype(q)::value / STEPS>{}, std::integral_constant<int, decltype(q)::value % STEPS>{});
      });
    };
    Stage st[PF];
    Frags fr[2];
    const auto step = [&](int t, auto at) __attribute__((always_inline)) {  // at: t modulo PF
      constexpr int b = decltype(at)::value & 1, held = (decltype(at)::value + 2) % PF;
      constexpr int BLOCKS = S::NM * S::NN, MFMAS = BLOCKS * 6, READS = S::NM + S::NN;
      constexpr int PART_A[6] = {2, 0, 1, 1, 0, 0}, PART_B[6] = {0, 2, 1, 0, 1, 0};
      const Frags& f = fr[b];
      Frags& next = fr[b ^ 1];
      each<MFMAS>([&](auto slot) __attribute__((always_inline)) {
        constexpr int s = decltype(slot)::value, term = s / BLOCKS, bm = s % BLOCKS / S::NN, bn = s % S::NN;
        acc[bm][bn] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f.b[bn][PART_B[term]], f.a[bm][PART_A[term]], acc[bm][bn], 0, 0, 0);
        // n things done by slots begin .. end - 1: those of slot s
        const auto share = [&](auto n_, auto begin_, auto end_, auto&& what) __attribute__((always_inline)) {
          constexpr int n = decltype(n_)::value, begin = decltype(begin_)::value, end = decltype(end_)::value;
          constexpr auto upto = [](int at) { return at < begin ? 0 : at >= end ? n : (at - begin) * n / (end - begin); };
          constexpr int from = upto(s), to = upto(s + 1);
          each<to - from>([&](auto i) __attribute__((always_inline)) { what(std::integral_constant<int, from + decltype(i)::value>{}); });
        };
        // The parts of t + 1, each where those of t have been used for the last time or soon will: h alone is there twice.
        const auto read = [&](auto part, auto begin, auto end) __attribute__((always_inline)) {
          share(std::integral_constant<int, READS>{}, begin, end, [&](auto i) __attribute__((always_inline)) {
            constexpr int r = decltype(i)::value;
            if constexpr (r < S::NM) read_a(b ^ 1, next, r, decltype(part)::value);
            else read_b(b ^ 1, next, r - S::NM, decltype(part)::value);
          });
        };
        using std::integral_constant;
        read(integral_constant<int, 2>{}, integral_constant<int, 2 * BLOCKS>{}, integral_constant<int, 3 * BLOCKS>{});
        read(integral_constant<int, 0>{}, integral_constant<int, 3 * BLOCKS>{}, integral_constant<int, 4 * BLOCKS>{});
        read(integral_constant<int, 1>{}, integral_constant<int, 4 * BLOCKS>{}, integral_constant<int, 5 * BLOCKS + BLOCKS / 2>{});
        share(integral_constant<int, CH * STEPS>{}, integral_constant<int, 0>{}, integral_constant<int, MFMAS * 5 / 6>{},
              [&](auto q) __attribute__((always_inline)) {
          put(st[held], b, integral_constant<int, decltype(q)::value / STEPS>{}, integral_constant<int, decltype(q)::value % STEPS>{});
        });
        if constexpr (s + 1 < MFMAS) __builtin_amdgcn_sched_barrier(0);
      });
      load(t + 2 + PF, st[held]);
      lds_barrier();
    };
    each<PF>([&](auto i) __attribute__((always_inline)) { load(decltype(i)::value, st[decltype(i)::value]); });
    put_all(st[0], 0);
    load(PF, st[0]);
    put_all(st[1], 1);
    load(PF + 1, st[1]);
    lds_barrier();
#pragma unroll
    for (int p = 0; p < 3; ++p) {
#pragma unroll
      for (int i = 0; i < S::NM; ++i) read_a(0, fr[0], i, p);
#pragma unroll
      for (int i = 0; i < S::NN; ++i) read_b(0, fr[0], i, p);
    }
    lds_barrier();  // (k-tile 2 takes the place of k-tile 0)
    static_assert(PF == 4, "rounds of four");
    for (int t = 0;; t += 4) {
      step(t, std::integral_constant<int, 0>{});
      if (t + 1 >= n) break;
      step(t + 1, std::integral_constant<int, 1>{});
      if (t + 2 >= n) break;
      step(t + 2, std::integral_constant<int, 2>{});
      if (t + 3 >= n) break;
      step(t + 3, std::integral_constant<int, 3>{});
      if (t + 4 >= n) break;
    }

    // ---- the shares of the k-tiles are added up, in their order
    const int pos = wm * S::WN + wn;
    f32x4* swap = reinterpret_cast<f32x4*>(lds) + lane_id();
    const auto slot = [&](int item, int owner, int from) {
      return ((pos * S::ITEMS + item) * (S::WK - 1) + (from < owner ? from : from - 1)) * 128;
    };
    if constexpr (S::WK > 1) {
#pragma unroll
      for (int i = 0; i < S::ITEMS; ++i) {
        const int owner = i / S::OWN, g = i & 1;
        if (owner != wk) {
          swap[slot(i, owner, wk)] = quad(acc[i / 2 / S::NN][i / 2 % S::NN], g);
          swap[slot(i, owner, wk) + 64] = quad(acc[i / 2 / S::NN][i / 2 % S::NN], g + 2);
        }
      }
    }
    lds_barrier();
#pragma unroll
    for (int i = 0; i < S::ITEMS; ++i) {
      const int owner = i / S::OWN, g = i & 1;
      if (owner == wk) {
        f32x4 lo = {0.f, 0.f, 0.f, 0.f}, hi = lo;
#pragma unroll
        for (int from = 0; from < S::WK; ++from) {
          const f32x4 l = from == owner ? quad(acc[i / 2 / S::NN][i / 2 % S::NN], g) : swap[slot(i, owner, from)];
          const f32x4 h = from == owner ? quad(acc[i / 2 / S::NN][i / 2 % S::NN], g + 2) : swap[slot(i, owner, from) + 64];
          if (from == 0) lo = l, hi = h;
          else lo += l, hi += h;
        }
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          out.lo[i % S::OWN][c] = __builtin_ldexpf(lo[c], SPLIT_EXP);
          out.hi[i % S::OWN][c] = __builtin_ldexpf(hi[c], SPLIT_EXP);
        }
      }
    }
    // Elements that are not finite.  (Rare: not worth LDS.  A wave computes the blocks of its items.)
    const auto odd = [](float v) { return __builtin_fabsf(v) >= __builtin_inff() || v != v; };
    bool any = false;
#pragma unroll
    for (int k = 0; k < S::OWN; ++k)
#pragma unroll
      for (int c = 0; c < 4; ++c) any |= odd(out.lo[k][c]) || odd(out.hi[k][c]);
    if (__ballot(any) == 0) return;
#pragma unroll 1
    for (int o = 0; o < S::OWN; ++o) {
      const int item = wk * S::OWN + o, block = item / 2, g = item & 1;
      f32x16 a;
#pragma unroll 1
      for (int share = 0; share < 4; ++share) {  // (as the smallest fp32 tiles have it)
        f32x16 q;
#pragma unroll
        for (int v = 0; v < 16; ++v) q[v] = 0.f;
        again((wm * S::NM + block / S::NN) * 32, (wn * S::NN + block % S::NN) * 32, share, q);
        a = share ? a + q : q;
      }
      const f32x4 lo = g ? quad(a, 1) : quad(a, 0), hi = g ? quad(a, 3) : quad(a, 2);
#pragma unroll
      for (int k = 0; k < S::OWN; ++k)
        if (k == o) {
#pragma unroll
          for (int c = 0; c < 4; ++c) {
            if (odd(out.lo[k][c])) out.lo[k][c] = lo[c];
            if (odd(out.hi[k][c])) out.hi[k][c] = hi[c];
          }
        }
    }
  }
};

}  // namespace
