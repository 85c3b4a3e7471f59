// Operand tiles that go from memory straight into a ring of LDS stages (buffer_load .. lds), for workgroups of WAVES
// waves: no staging registers, no LDS stores, and as many steps on their way as the ring has stages.  A wave-wide load
// fills 1 KB of consecutive LDS, so a stage has no padding; 16-byte chunks are permuted on the way instead, so that
// the fragment reads find different banks (no conflicts by SQ_LDS_BANK_CONFLICT).
#pragma once
#include "tile_ops.h"

namespace {

// The window's resource from byte_off on; not `live`: empty, everything reads as zero.
__device__ __forceinline__ u32x4 ring_rsrc(const View& w, long long byte_off, bool live) {
  const uint64_t at = (uint64_t)((const char*)w.base + byte_off);
  return u32x4{(uint32_t)at, (uint32_t)(at >> 32) & 0xffffu, live ? window_size(w.bytes - byte_off) : 0u, 0x00020000u};
}
// 16 bytes per lane from `off` into LDS at lds_byte + 16 * lane.  In assembly because the compiler would wait for every
// such load before any LDS read that follows; the waits are ring_wait's.  The load takes its LDS address from m0, which is
// written here and declared so: the compiler, which reserves m0, writes it anew for an instruction of its own that reads it.
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"  // (a reserved register on the list, which is the point)
__device__ __forceinline__ void ring_load(uint32_t lds_byte, u32x4 rsrc, uint32_t off) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, 0 offen lds" ::"v"(off), "s"(rsrc), "s"(lds_byte)
               : "m0");
}
// 4 bytes per lane, to lds_byte + 4 * lane.
__device__ __forceinline__ void ring_load_word(uint32_t lds_byte, u32x4 rsrc, uint32_t off) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tbuffer_load_dword %0, %1, 0 offen lds" ::"v"(off), "s"(rsrc), "s"(lds_byte) : "m0");
}
#pragma clang diagnostic pop
// All but the wave's N youngest loads have arrived and its LDS reads are done; then meet the other waves, for whose loads
// and reads the same holds.
template <int N>
__device__ __forceinline__ void ring_wait() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}
__device__ __forceinline__ uint32_t lds_address(const char* p) {
  return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const char*)p;
}

// Source is k-contiguous: element (r, kk) at view[r * ld + k0 + kk].  A stage holds ROWS rows of BK elements; fragments are
// 16-byte reads.
template <int ROWS_, int BK, int WAVES = 4>
struct RingInner {
  static constexpr int ROWS = ROWS_;
  static constexpr int CPR = BK / 8;  // 16-byte chunks per row
  static constexpr int BYTES = ROWS * BK * 2;
  static constexpr int RPP = 64 / CPR;  // rows per wave-wide load
  static constexpr int PER_WAVE = BYTES / (WAVES * 1024);
  static_assert(BYTES % (WAVES * 1024) == 0 && CPR == 8, "whole loads, rows of 128 bytes");
  static __device__ __forceinline__ int swizzle(int row) { return (row >> 1) & 7; }
  uint32_t off[PER_WAVE];  // byte offsets of this lane's chunks in the view
  int kc;                  // first k of its chunks
  __device__ __forceinline__ void init(int ld, int wv) {
    const int lane = lane_id(), r = lane / CPR;
    kc = ((lane % CPR) ^ swizzle(wv * RPP + r)) * 8;
#pragma unroll
    for (int i = 0; i < PER_WAVE; ++i) off[i] = (uint32_t)(((i * WAVES + wv) * RPP + r) * ld + kc) * 2;
  }
  // Rows from anywhere: at(r) is the byte offset of the tile's row r.
  template <typename At>
  __device__ __forceinline__ void set_rows(int wv, At at) {
#pragma unroll
    for (int i = 0; i < PER_WAVE; ++i) off[i] = at((i * WAVES + wv) * RPP + lane_id() / CPR) + (uint32_t)kc * 2;
  }
  // k past the end of the contraction lies in the next row: such chunks get an offset past any view (k_left: valid k)
  __device__ __forceinline__ void load(uint32_t stage, int wv, u32x4 rsrc, int k_left) const {
    const uint32_t past = kc >= k_left ? 0xffffffffu : 0u;
#pragma unroll
    for (int i = 0; i < PER_WAVE; ++i) ring_load(stage + (i * WAVES + wv) * 1024, rsrc, off[i] | past);
  }
  struct Place {
    uint32_t at, chunk;
  };
  static __device__ __forceinline__ Place place(int row0) {
    const int lane = lane_id(), r = row0 + (lane & 31);
    return {(uint32_t)(r * BK * 2), (uint32_t)((lane >> 5) ^ swizzle(r))};
  }
  static __device__ __forceinline__ bf16x8 frag(const char* stage, const Place& p, int rows, int ks) {
    return *reinterpret_cast<const bf16x8*>(stage + (p.at + rows * BK * 2 + ((p.chunk ^ (uint32_t)(ks * 2)) << 4)));
  }
};

// Source is row-contiguous: element (r, kk) at view[(k0 + kk) * ld + r].  A stage holds BK lines of ROWS elements as they
// lie in memory; fragments come through the transposing read (see OpOuter).
template <int ROWS_, int BK, int WAVES = 4>
struct RingOuter {
  static constexpr int ROWS = ROWS_;
  static constexpr int CPL = ROWS / 8;  // 16-byte chunks per line
  static constexpr int BYTES = ROWS * BK * 2;
  static constexpr int LPP = 64 / CPL;  // lines per wave-wide load
  static constexpr int PER_WAVE = BYTES / (WAVES * 1024);
  static_assert(BYTES % (WAVES * 1024) == 0 && ROWS % 128 == 0 && ROWS <= 256, "whole loads, lines of 16 or 32 chunks");
  // Half a wave's transposing read covers 64 bytes of each of four lines: they lie in different quarters of the 64 banks.
  static __device__ __forceinline__ int swizzle(int line) { return 4 * (line & 3); }
  uint32_t off[PER_WAVE];  // byte offsets of this lane's chunks in the view
  __device__ __forceinline__ void init(int ld, int wv) {
    const int lane = lane_id();
#pragma unroll
    for (int i = 0; i < PER_WAVE; ++i) {
      const int line = (i * WAVES + wv) * LPP + lane / CPL;
      off[i] = (uint32_t)(line * ld + ((lane % CPL) ^ swizzle(line)) * 8) * 2;
    }
  }
  __device__ __forceinline__ void load(uint32_t stage, int wv, u32x4 rsrc) const {
#pragma unroll
    for (int i = 0; i < PER_WAVE; ++i) ring_load(stage + (i * WAVES + wv) * 1024, rsrc, off[i]);
  }
  // A lane's place in the fragments of rows row0 .. row0 + 31, + 32, ...
  struct Place {
    uint32_t at, chunk;
  };
  static __device__ __forceinline__ Place place(int row0) {
    const int lane = lane_id(), i = lane & 15, b = lane >> 4;
    return {(uint32_t)(((b >> 1) * 8 + (i >> 2)) * ROWS * 2 + (i & 1) * 8),
            (uint32_t)((row0 / 8 + 2 * (b & 1) + ((i & 3) >> 1)) ^ swizzle(i >> 2))};
  }
  // (rows: 0, 32, .. past row0, in bits that row0 does not have)
  static __device__ __forceinline__ bf16x8 frag(const char* stage, const Place& p, int rows, int ks) {
    const char* at = stage + (p.at + ((p.chunk ^ (uint32_t)(rows / 8)) << 4) + ks * 16 * ROWS * 2);
    const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)at);
    const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(at + 4 * ROWS * 2));
    typedef __attribute__((ext_vector_type(8))) short s16x8;
    const s16x8 r = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    return __builtin_bit_cast(bf16x8, r);
  }
};

}  // namespace
