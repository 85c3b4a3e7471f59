// What the tiled matrix kernels share: windows of global memory read through buffer resources, the two LDS layouts
// of an operand tile with their loaders and fragment reads, and the workgroup barrier that leaves global loads
// in flight.
#pragma once
#include "common.h"

namespace {

typedef __attribute__((ext_vector_type(4))) short s16x4;
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;

// A window of global memory read through a buffer resource: reads at or past `bytes`
// return zero.  Only the per-lane offset takes part in the hardware bounds check (a scalar
// offset does not), so a window is advanced along k by moving its base and shrinking its
// size, both scalar operations.
struct View {
  const uint16_t* base;
  long long bytes;
};
__device__ __forceinline__ View make_view(const uint16_t* base, long long valid_elems) {
  return View{base, valid_elems > 0 ? valid_elems * 2 : 0};
}
// What a window has left, as a resource's size: none past its end, and no more than the 32 bits hold.  In the scalar unit: there is no
// 64-bit comparison there, and the vector unit's, whose results travel back, are what a k-tile's first products waited for.
__device__ __forceinline__ uint32_t window_size(long long left) {
  int high = (int)(left >> 32);
  asm("" : "+s"(high));  // (or the two halves become one 64-bit comparison again)
  return high < 0 ? 0u : high > 0 ? 0xffffffffu : (uint32_t)left;
}
// The window from a byte on, in scalar registers.
struct Window {
  const char* at;
  uint32_t size;
  __device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc() const {
    return __builtin_amdgcn_make_buffer_rsrc((void*)at, 0, (int)size, 0x00020000);
  }
  // Worked out where the program says so, not where it is first needed.
  __device__ __forceinline__ void stay_here() { asm volatile("" : "+s"(at), "+s"(size)); }
};
__device__ __forceinline__ Window window(const View& w, long long byte_off) {
  return {(const char*)w.base + byte_off, window_size(w.bytes - byte_off)};
}

// A byte offset outside any window that rows are read from anywhere of (less than 2 GB).
constexpr uint32_t NO_ROW = 1u << 31;

// ---- operand staging ----------------------------------------------------------------------
// Two LDS layouts, one per memory order of the operand, each with the fragment read that
// hands an MFMA lane its 8 consecutive k values for row (lane % 32):
//
// OpInner  source is k-contiguous: element (r, kk) at view[r * ld + k0 + kk].
//          LDS holds [ROWS][BK + 8] (16 bytes of padding per row); a fragment is one
//          16-byte LDS read.
// OpOuter  source is row-contiguous: element (r, kk) at view[(k0 + kk) * ld + r].
//          LDS holds the tile as it lies in memory, [BK][ROWS + 32] (64 bytes of padding
//          per k line); a fragment is two ds_read_b64_tr_b16, the gfx950 transposing LDS
//          read: a group of 16 lanes addresses a block of 4 k lines x 16 columns (lane i
//          points at line i/4, columns 4*(i%4)..+3) and lane i gets back column i of that
//          block, i.e. 4 consecutive k of its own row.
template <int ROWS_, int BK, int NT>
struct OpInner {
  static constexpr int ROWS = ROWS_;
  static constexpr int LDK = BK + 8;
  static constexpr int LDS_ELEMS = ROWS * LDK;
  static constexpr int CPR = BK / 8;          // 16-byte chunks per row
  static constexpr int CH = ROWS * CPR / NT;  // chunks per thread
  static constexpr int RSTEP = NT / CPR;      // rows between a thread's consecutive chunks
  static_assert((ROWS * CPR) % NT == 0 && NT % CPR == 0, "loader shape");
  int voff[CH];  // byte offsets of this thread's chunks inside the view at k0 = 0
  int lds_w;     // element offset of its first chunk in the LDS tile
  int kc;        // first k of its chunks inside the tile
  __device__ __forceinline__ void init(int ld) {
    const int r = threadIdx.x / CPR;
    kc = (threadIdx.x % CPR) * 8;
#pragma unroll
    for (int i = 0; i < CH; ++i) voff[i] = ((r + i * RSTEP) * ld + kc) * 2;
    lds_w = r * LDK + kc;
  }
  // Rows from anywhere: lane l has the byte offset of row own_row(l), of which the wave's lanes read CH * RPW.
  static constexpr int RPW = MOE_WAVE / CPR;  // rows of a wave's chunk
  static_assert(CH * RPW <= MOE_WAVE, "a lane a row");
  static __device__ __forceinline__ int own_row(int wv, int lane) { return wv * RPW + lane % RPW + lane / RPW * RSTEP; }
  __device__ __forceinline__ void set_rows(uint32_t at) {
#pragma unroll
    for (int i = 0; i < CH; ++i) voff[i] = (int)(__shfl(at, lane_id() / CPR + i * RPW, MOE_WAVE) + (uint32_t)kc * 2);
  }
  static __device__ __forceinline__ long long k_bytes(int k0, int /*ld*/) { return (long long)k0 * 2; }
  __device__ __forceinline__ u32x4 load_one(int i, __amdgpu_buffer_rsrc_t rs) const {
    return __builtin_amdgcn_raw_buffer_load_b128(rs, voff[i], 0, 0);
  }
  // k beyond the end of the contraction lies in the next row of a k-contiguous source, so
  // the hardware bound cannot catch it: such chunks are cleared by hand (k_left = valid k)
  __device__ __forceinline__ bool past_k(int k_left) const { return kc >= k_left; }
  __device__ __forceinline__ void store_one(int i, uint16_t* lds, u32x4 v) const {
    *reinterpret_cast<u32x4*>(lds + lds_w + i * RSTEP * LDK) = v;
  }
  static __device__ __forceinline__ int lane_off(int lane) { return (lane & 31) * LDK + (lane >> 5) * 8; }
  static __device__ __forceinline__ bf16x8 frag(const uint16_t* lds, int lane_offset, int row_base, int ks) {
    return *reinterpret_cast<const bf16x8*>(lds + lane_offset + row_base * LDK + ks * 16);
  }
};

template <int ROWS_, int BK, int NT>
struct OpOuter {
  static constexpr int ROWS = ROWS_;
  static constexpr int LDN = ROWS + 32;
  static constexpr int LDS_ELEMS = BK * LDN;
  static constexpr int CPK = ROWS / 8;        // 16-byte chunks per k line
  static constexpr int CH = BK * CPK / NT;
  static constexpr int KSTEP = NT / CPK;      // k lines between a thread's consecutive chunks
  static_assert((BK * CPK) % NT == 0 && NT % CPK == 0, "loader shape");
  int voff[CH];
  int lds_w;
  __device__ __forceinline__ void init(int ld) {
    const int kk = threadIdx.x / CPK, rc = (threadIdx.x % CPK) * 8;
#pragma unroll
    for (int i = 0; i < CH; ++i) voff[i] = ((kk + i * KSTEP) * ld + rc) * 2;
    lds_w = kk * LDN + rc;
  }
  // Lines from anywhere: lane l has the byte offset of line own_line(l), of which the wave's lanes read CH * LPW.
  static constexpr int LPW = MOE_WAVE / CPK;  // lines of a wave's chunk
  static_assert(LPW > 0 && CH * LPW <= MOE_WAVE, "a lane a line");
  static __device__ __forceinline__ int own_line(int wv, int lane) { return wv * LPW + lane % LPW + lane / LPW % CH * KSTEP; }
  __device__ __forceinline__ void set_lines(uint32_t at) {
    const uint32_t rc = threadIdx.x % CPK * 16;
#pragma unroll
    for (int i = 0; i < CH; ++i) voff[i] = (int)(__shfl(at, lane_id() / CPK + i * LPW, MOE_WAVE) + rc);
  }
  static __device__ __forceinline__ long long k_bytes(int k0, int ld) { return (long long)k0 * ld * 2; }
  __device__ __forceinline__ u32x4 load_one(int i, __amdgpu_buffer_rsrc_t rs) const {
    return __builtin_amdgcn_raw_buffer_load_b128(rs, voff[i], 0, 0);
  }
  // the k bound of this layout is the end of the view: the hardware zero-fills
  __device__ __forceinline__ bool past_k(int) const { return false; }
  __device__ __forceinline__ void store_one(int i, uint16_t* lds, u32x4 v) const {
    *reinterpret_cast<u32x4*>(lds + lds_w + i * KSTEP * LDN) = v;
  }
  // lane l = 16*b + i: k line (b/2)*8 + i/4, columns 16*(b%2) + 4*(i%4) .. +3
  static __device__ __forceinline__ int lane_off(int lane) {
    const int i = lane & 15, b = lane >> 4;
    return ((b >> 1) * 8 + (i >> 2)) * LDN + (b & 1) * 16 + (i & 3) * 4;
  }
  static __device__ __forceinline__ bf16x8 frag(const uint16_t* lds, int lane_offset, int row_base, int ks) {
    const uint16_t* p = lds + lane_offset + ks * 16 * LDN + row_base;
    const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(p));
    const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(p + 4 * LDN));
    typedef __attribute__((ext_vector_type(8))) short s16x8;
    const s16x8 r = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    return __builtin_bit_cast(bf16x8, r);
  }
};

// Wait for this wave's LDS traffic, then meet the other waves.  Global loads stay in flight.
__device__ __forceinline__ void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

}  // namespace
