// fp32 products on the fp16 matrix cores.  A value times a power of two is the sum of two fp16 values, x = h + l with h the
// nearest one and l the nearest to what is left, to 2^-24 of it.  Of the four products of two such sums three are added
// up in the matrix cores' fp32 accumulators (hl, lh, hh; ll is below 2^-24 of the product and mostly far below): three
// instructions at sixteen times the rate of the fp32 one, and closer to the exact sum, since an accumulator is rounded 3 times for
// every 16 products instead of 8 times.  Relative 2-norm error against fp64, normal operands, 64 / 256 / 1024 / 4096 products:
// 1.2e-7 / 1.9e-7 / 3.6e-7 / 7.1e-7, the fp32 instruction 1.4e-7 / 2.9e-7 / 5.7e-7 / 1.1e-6 (16 products: 8.7e-8, 7.3e-8).
// (Three bf16 parts need no scale, but six products: 2.3e-7 .. 1.0e-6, and 205 us where this takes 168.)
//
// The power of two brings the largest value of the first two k-tiles to 2^12 .. 2^13, so that what is lost of smaller ones is
// below 2^-37 of it: of a row where the operand is rows of activations or their gradients, of the tile where it is weights,
// or the contraction is along rows.  A k-tile whose values no longer fit, or are all below 4, gets another one, and
// what was added up so far is multiplied by the ratio: what is lost is always below 2^-27 of the k-tile's largest value.  Infinities and NaN give sums that are not finite: such a tile is computed again with the fp32
// instruction, and every result is the one it gives.
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

typedef __attribute__((ext_vector_type(8))) _Float16 f16x8;
typedef __attribute__((ext_vector_type(2))) _Float16 f16x2;

// f(0), f(1), .. f(N - 1) with constants for arguments: what they index stays in registers, however long the code
template <typename F, int... I>
__device__ __forceinline__ void each_of(F&& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void each(F&& f) {
  each_of(f, std::make_integer_sequence<int, N>{});
}

// Two values times `scale`, in their two parts, packed.
__device__ __forceinline__ uint32_t high_parts(float x, float y, float scale) {
  const f16x2 h = {(_Float16)(x * scale), (_Float16)(y * scale)};
  uint32_t w = __builtin_bit_cast(uint32_t, h);
  asm("" : "+v"(w));  // (the compiler would convert each once more on its own to have it unpacked)
  return w;
}
__device__ __forceinline__ uint32_t low_parts(float x, float y, float scale, uint32_t high) {
  const f16x2 h = __builtin_bit_cast(f16x2, high);
  const f16x2 l = {(_Float16)__builtin_fmaf(x, scale, -(float)h[0]), (_Float16)__builtin_fmaf(y, scale, -(float)h[1])};
  return __builtin_bit_cast(uint32_t, l);
}
// max(big, |x|, |y|), where a NaN counts for nothing (fmaxf would quiet every operand first)
__device__ __forceinline__ void larger_of(float& big, float x, float y) {
  asm("v_max3_f32 %0, %0, |%1|, |%2|" : "+v"(big) : "v"(x), "v"(y));
}

// The largest of the wave's values >= 0, which integers order as floats (in the vector unit alone, as wave_inclusive).
__device__ __forceinline__ float wave_largest(float f) {
  int v = __builtin_bit_cast(int, f);
  const auto larger = [&](int w) { v = v > w ? v : w; };
  larger(__builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, true));  // row_shr:1, 2, 4, 8: inside the rows of 16
  larger(__builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, true));
  larger(__builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, true));
  larger(__builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, true));
  larger(__builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false));  // row_bcast:15 to rows 1 and 3
  larger(__builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false));  // row_bcast:31 to rows 2 and 3
  return __builtin_bit_cast(float, read_lane(v, MOE_WAVE - 1));
}

// Operand tiles of ROWS x TK in LDS, one plane a part.  A thread moves chunks of eight values.
//
// SplitInner: element (r, k) at base[r * ld + k]; a plane is [ROWS][TK], chunks permuted against bank conflicts; a fragment is
//             one 16-byte read.
// SplitOuter: element (r, k) at base[k * ld + r]; a plane is [TK][ROWS], chunks permuted; fragments come
//             through the transposing read (see OpOuter).
template <int ROWS, int TK, int NT>
struct SplitInner {
  static constexpr bool INNER = true;
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
  static __device__ __forceinline__ f16x8 frag(const char* plane, const Lane& l, int rows, int ks) {
    return *reinterpret_cast<const f16x8*>(plane + (l.at + rows * TK * 2 + ((l.chunk ^ (ks * 2)) << 4)));
  }
  // the largest value of a row's chunks (the lanes that hold them), which integers order as floats
  static __device__ __forceinline__ float row_largest(float f) {
    int v = __builtin_bit_cast(int, f), w = __builtin_amdgcn_mov_dpp(v, 0xb1, 0xf, 0xf, true);  // quad_perm 1 0 3 2
    v = v > w ? v : w;
    w = __builtin_amdgcn_mov_dpp(v, 0x4e, 0xf, 0xf, true);  // quad_perm 2 3 0 1
    v = v > w ? v : w;
    if constexpr (CPR == 8) {
      w = __builtin_amdgcn_mov_dpp(v, 0x141, 0xf, 0xf, true);  // row_half_mirror
      v = v > w ? v : w;
    }
    return __builtin_bit_cast(float, v);
  }
  // one value, anywhere
  static __device__ __forceinline__ float value(const float* base, int ld, int rows, int k_end, int r, int k) {
    return r < rows && k < k_end ? base[(long long)r * ld + k] : 0.f;
  }
};
template <int ROWS, int TK, int NT>
struct SplitOuter {
  static constexpr bool INNER = false;
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
  static __device__ __forceinline__ f16x8 frag(const char* plane, const Lane& l, int rows, int ks) {
    const char* at = plane + (l.at + ((l.chunk ^ (rows / 8)) << 4) + ks * 16 * ROWS * 2);
    const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)at);
    const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(at + 4 * ROWS * 2));
    typedef __attribute__((ext_vector_type(8))) short s16x8;
    const s16x8 r = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    return __builtin_bit_cast(f16x8, r);
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
  static constexpr int CH = OpA::CH + OpB::CH, STAGE = 2 * (OpA::PLANE + OpB::PLANE);
  static constexpr int SWAP = S::WM * S::WN * S::ITEMS * (S::WK - 1) * 2048, WORDS = 128;
  // An operand A that lies k-contiguous is scaled row by row: then no row's values matter to another one's result
  static constexpr bool BY_ROW = OpA::INNER;
  static constexpr int ROW_WORDS = BY_ROW ? 5 * S::BM * 4 : 0;
  static_assert(!BY_ROW || OpA::CH == 1, "a thread's values of A are of one row");
  static constexpr int LDS_BYTES = (2 * STAGE > SWAP ? 2 * STAGE : SWAP) + WORDS + ROW_WORDS;
  static constexpr int PF = 4;  // k-tiles in registers on their way to LDS
  typedef f32x16 Acc[S::NM][S::NN];
  struct Stage {
    f32x4 v[CH][2];
  };
  struct Frags {
    f16x8 a[S::NM][2], b[S::NN][2];
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
  // written to the LDS stage that t has left, and t + 6 is requested: one barrier a k-tile, and nothing between two of them that
  // waits for one another.  16384 rows of 8 experts, 1024 -> 2 x 512, four tiles of 128 x 128 to a compute unit: 168 us (fp32 instruction: 285), where the
  // products alone take 76 and a tile's start and end 35; each k-tile of 32 has 768 cycles of products, 470 of LDS
  // writes (70 bytes a cycle; reads 240), 450 of vector work.  Splitting after the LDS instead (fp32 values straight
  // from memory into the ring, twice the vector work) takes a tenth longer: vector and matrix work of two waves hardly overlap.
  // `load(t, stage)` requests a k-tile, `again(row, column, acc)` computes a block with fp32 products.
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
      f.b[x][p] = OpB::frag(lds + b * STAGE + 2 * OpA::PLANE + p * OpB::PLANE, lb, x * 32, wk);
    };
    u32x4 parts[2];
    float scale_a, scale_b;  // powers of two: a row's (BY_ROW) or all threads', all threads'
    // step i of chunk c: a part of two of its values; the last one also writes the chunk
    const auto put = [&](const Stage& s, int b, auto chunk, auto step) __attribute__((always_inline)) {
      constexpr int c = decltype(chunk)::value, q = decltype(step)::value / 2, p = decltype(step)::value % 2;
      const float x = s.v[c][q >> 1][(q & 1) * 2], y = s.v[c][q >> 1][(q & 1) * 2 + 1], scale = c < OpA::CH ? scale_a : scale_b;
      if constexpr (p == 0) parts[0][q] = high_parts(x, y, scale);
      else parts[1][q] = low_parts(x, y, scale, parts[0][q]);
      if constexpr (q == 3 && p == 1) {
        char* to = c < OpA::CH ? lds + b * STAGE + OpA::place(c) : lds + b * STAGE + 2 * OpA::PLANE + OpB::place(c - OpA::CH);
        *reinterpret_cast<u32x4*>(to) = parts[0];
        *reinterpret_cast<u32x4*>(to + (c < OpA::CH ? OpA::PLANE : OpB::PLANE)) = parts[1];
      }
    };
    // the largest values of a k-tile's chunks
    const auto largest = [&](const Stage& s, float& a, float& b) __attribute__((always_inline)) {
      each<CH * 4>([&](auto i) __attribute__((always_inline)) {
        constexpr int c = decltype(i)::value / 4, q = decltype(i)::value % 4;
        larger_of(c < OpA::CH ? a : b, s.v[c][q >> 1][(q & 1) * 2], s.v[c][q >> 1][(q & 1) * 2 + 1]);
      });
    };
    // [8][2] largest values; [2] "values do not fit"; [2][2] the last k-tile that was large enough
    int* words = reinterpret_cast<int*>(lds + LDS_BYTES - WORDS - ROW_WORDS);
    float* row_grown = reinterpret_cast<float*>(lds + LDS_BYTES - ROW_WORDS);  // [4][BM] for k-tile t % 4, as `grown`
    int* row_exp = reinterpret_cast<int*>(row_grown + 4 * S::BM);               // [BM] at the end
    const auto largest_of_all = [&](float& a, float& b) {  // (two barriers)
      a = wave_largest(a), b = wave_largest(b);
      if (lane_id() == 0) words[2 * wv] = __builtin_bit_cast(int, a), words[2 * wv + 1] = __builtin_bit_cast(int, b);
      lds_barrier();
      int ia = 0, ib = 0;  // (as integers: an infinity is the largest, a NaN was left out)
#pragma unroll
      for (int w = 0; w < S::NT / 64; ++w) {
        ia = ia > words[2 * w] ? ia : words[2 * w];
        ib = ib > words[2 * w + 1] ? ib : words[2 * w + 1];
      }
      a = __builtin_bit_cast(float, uniform(ia)), b = __builtin_bit_cast(float, uniform(ib));
      lds_barrier();
    };
    int exp_a, exp_b, least_a, least_b;  // least: the smallest so far
    float limit_a, limit_b, low_a, low_b;
    // What the sums are multiplied by before k-tile t, t + 1, t + 2 (BY_ROW: times row_grown; 0: nothing)
    float grown[3] = {0.f, 0.f, 0.f};
    // The largest of so many values becomes 2^12 to 2^13: 7 times more fits, and parts below 2^-38 of it are lost.
    const auto exponent_for = [](float big) {
      const int e = 12 + 127 - (__builtin_bit_cast(int, big) >> 23);
      return e > 126 ? 126 : e < -114 ? -114 : e;
    };
    const auto power = [](int e) { return __builtin_bit_cast(float, (127 + e) << 23); };
    const auto set_scales = [&](int ea, int eb) {
      exp_a = ea, exp_b = eb;
      scale_a = power(ea), scale_b = power(eb);
      limit_a = 60000.f * power(-ea), limit_b = 60000.f * power(-eb);
      low_a = 4.f * power(-ea), low_b = 4.f * power(-eb);
    };
    const auto too_large = [](float big, float limit) { return big > limit && big < __builtin_inff(); };
    const auto too_small = [](float big, float low) { return big > 0.f && big < low; };
    const auto report = [&](int t, int word, float a, float b) __attribute__((always_inline)) {  // the largest values of k-tile t
      bool misfit = too_large(b, limit_b);
      if constexpr (BY_ROW) {
        a = OpA::row_largest(a);
        misfit |= too_large(a, limit_a) | too_small(a, low_a);
      } else {
        misfit |= too_large(a, limit_a);
        if (__ballot(a >= low_a)) words[18 + 2 * word] = t;
      }
      if (__ballot(misfit)) words[16 + word] = 1;
      if (__ballot(b >= low_b)) words[19 + 2 * word] = t;
    };
    const auto rescale = [&](const Stage& s, int t, int word) {  // for k-tile t, which s holds
      float a = 0.f, b = 0.f, all_a;
      largest(s, a, b);
      all_a = a;
      largest_of_all(all_a, b);
      if constexpr (BY_ROW) a = OpA::row_largest(a);
      else a = all_a;
      // (2^30 more than the least: the sums, below 2^42 then, stay finite)
      const auto fitting = [&](float big, float low, float limit, int e, int least) {
        const int want = too_large(big, limit) || too_small(big, low) ? exponent_for(big) : e;
        return want < least + 30 ? want : least + 30;
      };
      const int ea = fitting(a, low_a, limit_a, exp_a, least_a), eb = fitting(b, low_b, limit_b, exp_b, least_b);
      const auto ratio = [&](int d) { return power(d < -126 ? -126 : d); };  // (what is lost so is far below the rest)
      grown[2] = ratio(eb - exp_b);
      if constexpr (BY_ROW) {
        if (threadIdx.x % OpA::CPR == 0) row_grown[(t & 3) * S::BM + OpA::row(0)] = ratio(ea - exp_a);
      } else {
        grown[2] = ratio(ea - exp_a + eb - exp_b);
      }
      least_a = least_a < ea ? least_a : ea, least_b = least_b < eb ? least_b : eb;
      set_scales(ea, eb);
      words[16 + word] = 0;
    };
    const auto put_all = [&](const Stage& s, int b) __attribute__((always_inline)) {
      each<CH * 8>([&](auto q) __attribute__((always_inline)) {
        put(s, b, std::integral_constant<int, decltype(q)::value / 8>{}, std::integral_constant<int, decltype(q)::value % 8>{});
      });
    };
    Stage st[PF];
    Frags fr[2];
    const auto step = [&](int t, auto at) __attribute__((always_inline)) {  // at: t modulo PF
      constexpr int b = decltype(at)::value & 1, held = (decltype(at)::value + 2) % PF, after = (decltype(at)::value + 3) % PF;
      constexpr int READS = (S::NM + S::NN) * 2, BLOCKS = S::NM * S::NN, MFMAS = BLOCKS * 3, PUTS = CH * 8;
      const Frags& f = fr[b];
      Frags& next = fr[b ^ 1];
      const int misfit = words[16 + b], large_a = BY_ROW ? t + 2 : words[18 + 2 * b], large_b = words[19 + 2 * b];  // of k-tile t + 2
      if (grown[0] != 0.f) {
#pragma unroll
        for (int i = 0; i < S::NM; ++i) {
          float by = grown[0];
          if constexpr (BY_ROW) by *= row_grown[(t & 3) * S::BM + (wm * S::NM + i) * 32 + (lane_id() & 31)];
#pragma unroll
          for (int j = 0; j < S::NN; ++j) acc[i][j] *= by;
        }
      }
      float seen_a = 0.f, seen_b = 0.f;  // of k-tile t + 3
      each<MFMAS>([&](auto slot) __attribute__((always_inline)) {
        constexpr int s = decltype(slot)::value, term = s / BLOCKS, bm = s % BLOCKS / S::NN, bn = s % S::NN;  // small products first
        acc[bm][bn] = __builtin_amdgcn_mfma_f32_32x32x16_f16(f.b[bn][term == 0], f.a[bm][term == 1], acc[bm][bn], 0, 0, 0);
        constexpr auto upto = [](int at, int n, int begin, int end) {
          const int v = (at - begin) * n / (end - begin);
          return at < begin ? 0 : v < n ? v : n;
        };
        constexpr int CHECK = MFMAS / 6, R0 = upto(s, READS, 0, MFMAS * 2 / 3), R1 = upto(s + 1, READS, 0, MFMAS * 2 / 3);
        constexpr int Q0 = upto(s, PUTS, CHECK, MFMAS * 5 / 6), Q1 = upto(s + 1, PUTS, CHECK, MFMAS * 5 / 6);
        if constexpr (s == CHECK) {
          if (uniform(misfit | (large_a ^ (t + 2)) | (large_b ^ (t + 2))) && t + 2 < n) rescale(st[held], t + 2, b);
          grown[0] = grown[1], grown[1] = grown[2], grown[2] = 0.f;
        }
        each<R1 - R0>([&](auto i) __attribute__((always_inline)) {
          constexpr int r = R0 + decltype(i)::value, rb = r - S::NM * 2;
          if constexpr (r < S::NM * 2) read_a(b ^ 1, next, r % S::NM, r / S::NM);
          else read_b(b ^ 1, next, rb % S::NN, rb / S::NN);
        });
        each<Q1 - Q0>([&](auto i) __attribute__((always_inline)) {
          constexpr int q = Q0 + decltype(i)::value;
          put(st[held], b, std::integral_constant<int, q / 8>{}, std::integral_constant<int, q % 8>{});
        });
        constexpr int L0 = upto(s, CH * 4, MFMAS / 2, MFMAS), L1 = upto(s + 1, CH * 4, MFMAS / 2, MFMAS);
        each<L1 - L0>([&](auto i) __attribute__((always_inline)) {
          constexpr int l = L0 + decltype(i)::value, c = l / 4, q = l % 4;
          larger_of(c < OpA::CH ? seen_a : seen_b, st[after].v[c][q >> 1][(q & 1) * 2], st[after].v[c][q >> 1][(q & 1) * 2 + 1]);
        });
        if constexpr (s + 1 < MFMAS) __builtin_amdgcn_sched_barrier(0);
      });
      load(t + 2 + PF, st[held]);
      report(t + 3, b ^ 1, seen_a, seen_b);
      lds_barrier();
    };
    static_assert(PF == 4, "rounds of four");
    if (threadIdx.x < 2) words[16 + threadIdx.x] = 0;
    load(0, st[0]);
    load(1, st[1]);
    load(2, st[2]);
    load(3, st[3]);
    {
      float a = 0.f, b = 0.f;
      largest(st[0], a, b);
      largest(st[1], a, b);
      float all_a = a;
      largest_of_all(all_a, b);
      if constexpr (BY_ROW) a = OpA::row_largest(a);
      else a = all_a;
      set_scales(exponent_for(a), exponent_for(b));
      least_a = exp_a, least_b = exp_b;
    }
    put_all(st[0], 0);
    load(PF, st[0]);
    put_all(st[1], 1);
    load(PF + 1, st[1]);
    {
      float a = 0.f, b = 0.f;
      largest(st[2], a, b);
      report(2, 0, a, b);
    }
    lds_barrier();
#pragma unroll
    for (int p = 0; p < 2; ++p) {
#pragma unroll
      for (int x = 0; x < S::NM; ++x) read_a(0, fr[0], x, p);
#pragma unroll
      for (int x = 0; x < S::NN; ++x) read_b(0, fr[0], x, p);
    }
    lds_barrier();  // (k-tile 2 takes the place of k-tile 0)
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

    // ---- the shares of the k-tiles are added up, in their order, and the tile's range is looked at
    f32x4 zeros = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < S::NM; ++i)
#pragma unroll
      for (int j = 0; j < S::NN; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v) zeros[v & 3] = __builtin_fmaf(acc[i][j][v], 0.f, zeros[v & 3]);
    const float zero = (zeros[0] + zeros[1]) + (zeros[2] + zeros[3]);
    const bool finite = __ballot(zero != 0.f) == 0;
    if (lane_id() == 0) words[wv] = !finite;
    if constexpr (BY_ROW) {
      if (threadIdx.x % OpA::CPR == 0) row_exp[OpA::row(0)] = exp_a;
    }
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
    int again_all = 0;
#pragma unroll
    for (int i = 0; i < S::NT / 64; ++i) again_all |= words[i];
    if (uniform(again_all)) {
      // (rare: not worth LDS.  A wave computes the blocks of its items.)
#pragma unroll 1
      for (int o = 0; o < S::OWN; ++o) {
        const int item = wk * S::OWN + o, block = item / 2, g = item & 1;
        f32x16 a;
#pragma unroll
        for (int v = 0; v < 16; ++v) a[v] = 0.f;
        again((wm * S::NM + block / S::NN) * 32, (wn * S::NN + block % S::NN) * 32, a);
#pragma unroll
        for (int k = 0; k < S::OWN; ++k)
          if (k == o) out.lo[k] = g ? quad(a, 1) : quad(a, 0), out.hi[k] = g ? quad(a, 3) : quad(a, 2);
      }
      return;
    }
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
        const int e = (BY_ROW ? row_exp[(wm * S::NM + i / 2 / S::NN) * 32 + (lane_id() & 31)] : exp_a) + exp_b;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          out.lo[i % S::OWN][c] = __builtin_ldexpf(lo[c], -e);
          out.hi[i % S::OWN][c] = __builtin_ldexpf(hi[c], -e);
        }
      }
    }
  }
};

}  // namespace
