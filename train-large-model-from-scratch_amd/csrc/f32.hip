// The expert path in fp32, for callers that run the layer without autocast on fp32 tensors: the
// reference then computes its three bmm's, SwiGLU, gate weighting and k-sum in fp32
// (model/modules/mlp.py:133-169 with fp32 operands), and so does this file.  Same routing and
// dispatch kernels as the bf16 path; what differs is the row type of the expert-contiguous
// buffers (fp32 [R,H] / [R,I]).  The products are in f32_gemm.hip.
#include "common.h"
#include "internal.h"

namespace {

// ---- row movers and element-wise kernels (one workgroup per row, 16-byte accesses)

// xp[pos, :] = x[pos_to_row[pos] / k, :]   (mlp.py:104-131: repeat_interleave + the two sorts)
__global__ __launch_bounds__(256) void f32_gather_rows_kernel(const float* __restrict__ x,
                                                              const int32_t* __restrict__ pos_to_row, int T,
                                                              int H, int k, float* __restrict__ xp) {
  const long long pos = blockIdx.x;
  const int row = pos_to_row[pos];
  const int t = row / k;
  const bool ok = row >= 0 && t < T;
  for (int h = threadIdx.x * 4; h < H; h += 256 * 4) {
    f32x4 v = {0.f, 0.f, 0.f, 0.f};
    if (ok) v = *reinterpret_cast<const f32x4*>(x + (long long)t * H + h);
    *reinterpret_cast<f32x4*>(xp + pos * H + h) = v;
  }
}

// out[t, :] = sum_j gates[t*k+j] * y[row_to_pos[t*k+j], :], j ascending  (mlp.py:160-169);
// gates == nullptr: all ones (with k = 1 a pure un-permute)
__global__ __launch_bounds__(256) void f32_combine_fwd_kernel(const float* __restrict__ y,
                                                              const float* __restrict__ gates,
                                                              const int32_t* __restrict__ row_to_pos, int R,
                                                              int H, int k, float* __restrict__ out) {
  const long long t = blockIdx.x;
  for (int h = threadIdx.x * 4; h < H; h += 256 * 4) {
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    for (int j = 0; j < k; ++j) {
      const int pos = row_to_pos[t * k + j];
      if (pos < 0 || pos >= R) continue;
      const float g = gates ? gates[t * k + j] : 1.f;
      const f32x4 v = *reinterpret_cast<const f32x4*>(y + (long long)pos * H + h);
      acc += g * v;
    }
    *reinterpret_cast<f32x4*>(out + t * H + h) = acc;
  }
}

// Backward of the above: dyp[pos, :] = gate * dy[t, :], dgates[row] = <dy[t, :], y[pos, :]>
// (row = pos_to_row[pos], t = row / k).  The dot product is reduced in a fixed tree.
__global__ __launch_bounds__(256) void f32_combine_bwd_kernel(const float* __restrict__ dy,
                                                              const float* __restrict__ y,
                                                              const float* __restrict__ gates,
                                                              const int32_t* __restrict__ pos_to_row, int T,
                                                              int H, int k, float* __restrict__ dyp,
                                                              float* __restrict__ dgates) {
  __shared__ float part[4];
  const long long pos = blockIdx.x;
  const int row = pos_to_row[pos];
  const int t = row / k;
  const bool ok = row >= 0 && t < T;
  const float g = ok ? (gates ? gates[row] : 1.f) : 0.f;
  float dot = 0.f;
  for (int h = threadIdx.x * 4; h < H; h += 256 * 4) {
    f32x4 d = {0.f, 0.f, 0.f, 0.f};
    if (ok) d = *reinterpret_cast<const f32x4*>(dy + (long long)t * H + h);
    *reinterpret_cast<f32x4*>(dyp + pos * H + h) = g * d;
    if (dgates) {
      const f32x4 v = *reinterpret_cast<const f32x4*>(y + pos * H + h);
      dot += d[0] * v[0] + d[1] * v[1] + d[2] * v[2] + d[3] * v[3];
    }
  }
  if (!dgates) return;  // (uniform: every thread leaves)
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) dot += __shfl_xor(dot, o, MOE_WAVE);
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = dot;
  __syncthreads();
  if (threadIdx.x == 0 && ok) dgates[row] = (part[0] + part[1]) + (part[2] + part[3]);
}

// dx[t, :] = sum_j dxp[row_to_pos[t*k+j], :], j ascending  (backward of the replication)
__global__ __launch_bounds__(256) void f32_permute_bwd_kernel(const float* __restrict__ dxp,
                                                              const int32_t* __restrict__ row_to_pos, int R,
                                                              int H, int k, float* __restrict__ dx) {
  const long long t = blockIdx.x;
  for (int h = threadIdx.x * 4; h < H; h += 256 * 4) {
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    for (int j = 0; j < k; ++j) {
      const int pos = row_to_pos[t * k + j];
      if (pos < 0 || pos >= R) continue;
      acc += *reinterpret_cast<const f32x4*>(dxp + (long long)pos * H + h);
    }
    *reinterpret_cast<f32x4*>(dx + t * H + h) = acc;
  }
}

// The same with the router's backward in it, where the router product is part of the layer: from the gate gradients the softmax
// Jacobian over the token's k winners (as router_topk_bwd_kernel, the k-term sum ascending), dsel = its k nonzero logit gradients,
// left by position for the weight gradient, and dx += sum_j dsel[j] * wr[ids[t*k+j], :] (dx NULL: not wanted).  In its place were a
// launch for the rows of dlogits, the library's product with them, and an addition of two [T, H].  Bound by memory, k rows of wr a token
// from L2 on top of the other kernel's.  With the next kernel, whole passes, us: 2048 tokens, 2 of 8 experts, 1024 <-> 512, 381 -> 362; 4717,
// 2 of 64, 768 <-> 384, 690 -> 624; 11981, 1 of 128, 320 <-> 1472, 1536 -> 1422; 939, 8 of 16, 3136 <-> 256, 1014 -> 1000; where the host bounds
// them, two library products and two nodes less: 686, 2 of 4, 1136 <-> 160, 221 -> 161; 239, 3 of 64, 816 <-> 168, 227 -> 201.
__global__ __launch_bounds__(256) void f32_permute_bwd_router_kernel(
    const float* __restrict__ dxp, const int32_t* __restrict__ row_to_pos, const float* __restrict__ gates,
    const float* __restrict__ dgates, const int32_t* __restrict__ ids, const float* __restrict__ wr, int R, int H, int k,
    float* __restrict__ dsel_by_pos, float* __restrict__ dx) {
  const long long t = blockIdx.x;
  const int lane = lane_id();
  float g = 0.f, dg = 0.f;
  int id = 0, pos = -1;
  if (lane < k) {
    g = gates[t * k + lane];
    dg = dgates[t * k + lane];
    id = ids[t * k + lane];
    pos = row_to_pos[t * k + lane];
  }
  float s = 0.f;
  for (int j = 0; j < k; ++j) s += read_lane_f(g, j) * read_lane_f(dg, j);
  const float dsel = g * (dg - s);
  if (threadIdx.x < (unsigned)k && pos >= 0 && pos < R) dsel_by_pos[pos] = dsel;
  if (!dx) return;
  for (int h = threadIdx.x * 4; h < H; h += 256 * 4) {
    f32x4 acc = {0.f, 0.f, 0.f, 0.f}, router = {0.f, 0.f, 0.f, 0.f};
    for (int j = 0; j < k; ++j) {
      const int p = read_lane(pos, j);
      router += read_lane_f(dsel, j) * *reinterpret_cast<const f32x4*>(wr + (long long)read_lane(id, j) * H + h);
      if (p < 0 || p >= R) continue;
      acc += *reinterpret_cast<const f32x4*>(dxp + (long long)p * H + h);
    }
    *reinterpret_cast<f32x4*>(dx + t * H + h) = acc + router;
  }
}

// dwr[e, :] = sum over the expert's rows of dsel * xp[row, :]: what dlogits^T x comes to, whose other entries are zero, in one
// pass over the rows that the experts' products read anyway.  256 columns a workgroup, a row a wave, eight of them requested at
// once, the waves' sums added in order.  Workgroup y of a column is segment y of the rows: an expert of more than L rows is cut into
// parts, whose sums the next kernel adds up.
constexpr int RW_WAVES = 8, RW_COLS = 4 * MOE_WAVE;
struct RowCut {
  const int32_t* offs;
  int E, L;
  // (an expert without rows is a part too: its gradient is zero)
  __device__ __forceinline__ int parts(int rows) const { return rows <= L ? 1 : (int)(((long long)rows + L - 1) / L); }
  __device__ __forceinline__ int rows(int e) const { return e < E ? offs[e + 1] - offs[e] : 0; }
  // Number of segments of the experts before e, by a whole wave; e past the last: those of all.
  __device__ __forceinline__ int before(int e) const {
    int n = 0;
    for (int b = 0; b < e; b += MOE_WAVE) {
      const int at = b + lane_id();
      n += read_lane(wave_inclusive(at < e ? parts(rows(at)) : 0), MOE_WAVE - 1);
    }
    return n;
  }
};
__global__ __launch_bounds__(RW_WAVES* MOE_WAVE) void f32_router_wgrad_kernel(const float* __restrict__ xp,
                                                                            const float* __restrict__ dsel, const RowCut cut,
                                                                            int H, float* __restrict__ partial,
                                                                            float* __restrict__ dwr) {
  constexpr int AHEAD = 8;
  __shared__ f32x4 part[RW_WAVES][MOE_WAVE];
  const int lane = lane_id(), wv = uniform((int)(threadIdx.x / MOE_WAVE)), col = blockIdx.x * RW_COLS + lane * 4;
  const int seg = blockIdx.y;
  int e = -1, parts = 0, j = 0;
  for (int b = 0, carry = 0; b < cut.E; b += MOE_WAVE) {
    const int p = b + lane < cut.E ? cut.parts(cut.rows(b + lane)) : 0, upto = carry + wave_inclusive(p);
    const unsigned long long past = __ballot(upto > seg);
    if (past) {
      const int f = __builtin_ctzll(past);
      e = b + f, parts = read_lane(p, f), j = seg - (read_lane(upto, f) - parts);
      break;
    }
    carry = read_lane(upto, MOE_WAVE - 1);
  }
  if (e < 0) return;
  const int first = cut.offs[e];
  const long long n = cut.offs[e + 1] - first;
  const int lo = first + (int)(n * j / parts), hi = first + (int)(n * (j + 1) / parts);
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  for (int r = lo + wv; r < hi; r += RW_WAVES * AHEAD) {
    f32x4 v[AHEAD];
    float d[AHEAD];
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) {
      const int row = r + i * RW_WAVES;
      const bool in = row < hi;
      d[i] = in ? dsel[row] : 0.f;
      v[i] = in && col < H ? *reinterpret_cast<const f32x4*>(xp + (long long)row * H + col) : f32x4{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) acc += d[i] * v[i];
  }
  part[wv][lane] = acc;
  __syncthreads();
  if (wv || col >= H) return;
#pragma unroll
  for (int w = 1; w < RW_WAVES; ++w) acc += part[w][lane];
  float* out = parts > 1 ? partial + (long long)seg * H : dwr + (long long)e * H;
  *reinterpret_cast<f32x4*>(out + col) = acc;
}
// dwr[e, :] of the experts that were cut: four waves, each every fourth part in ascending order, and the four sums in order.
constexpr int RS_WAVES = 4;
__global__ __launch_bounds__(RS_WAVES* MOE_WAVE) void f32_router_wgrad_sum_kernel(const float* __restrict__ partial,
                                                                                const RowCut cut, int H,
                                                                                float* __restrict__ dwr) {
  __shared__ f32x4 part[RS_WAVES][MOE_WAVE];
  const int e = blockIdx.y, parts = uniform(cut.parts(cut.rows(e)));
  if (parts == 1) return;
  const int lane = lane_id(), wv = uniform((int)(threadIdx.x / MOE_WAVE)), col = blockIdx.x * RW_COLS + lane * 4;
  const float* from = partial + (long long)cut.before(e) * H + col;
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  if (col < H) {
#pragma unroll 8
    for (int j = wv; j < parts; j += RS_WAVES) acc += *reinterpret_cast<const f32x4*>(from + (long long)j * H);
  }
  part[wv][lane] = acc;
  __syncthreads();
  if (wv || col >= H) return;
#pragma unroll
  for (int w = 1; w < RS_WAVES; ++w) acc += part[w][lane];
  *reinterpret_cast<f32x4*>(dwr + (long long)e * H + col) = acc;
}

__device__ __forceinline__ float sigmoid_f32(float x) { return 1.f / (1.f + expf(-x)); }

// act = silu(g) * u   (mlp.py:156)
__global__ __launch_bounds__(256) void f32_swiglu_fwd_kernel(const float* __restrict__ g,
                                                             const float* __restrict__ u, long long n4,
                                                             float* __restrict__ act) {
  const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
  if (i >= n4) return;
  const f32x4 gv = reinterpret_cast<const f32x4*>(g)[i], uv = reinterpret_cast<const f32x4*>(u)[i];
  f32x4 a;
#pragma unroll
  for (int x = 0; x < 4; ++x) a[x] = gv[x] * sigmoid_f32(gv[x]) * uv[x];
  reinterpret_cast<f32x4*>(act)[i] = a;
}

// dg = dact * u * silu'(g), du = dact * silu(g);  silu'(g) = s * (1 + g * (1 - s)), s = sigmoid(g)
__global__ __launch_bounds__(256) void f32_swiglu_bwd_kernel(const float* __restrict__ dact,
                                                             const float* __restrict__ g,
                                                             const float* __restrict__ u, long long n4,
                                                             float* __restrict__ dg, float* __restrict__ du) {
  const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
  if (i >= n4) return;
  const f32x4 dv = reinterpret_cast<const f32x4*>(dact)[i];
  const f32x4 gv = reinterpret_cast<const f32x4*>(g)[i], uv = reinterpret_cast<const f32x4*>(u)[i];
  f32x4 a, b;
#pragma unroll
  for (int x = 0; x < 4; ++x) {
    const float s = sigmoid_f32(gv[x]);
    a[x] = dv[x] * uv[x] * (s * (1.f + gv[x] * (1.f - s)));
    b[x] = dv[x] * (gv[x] * s);
  }
  reinterpret_cast<f32x4*>(dg)[i] = a;
  reinterpret_cast<f32x4*>(du)[i] = b;
}

int check_rows(int64_t rows, int64_t width) {
  if (rows < 0 || width <= 0 || width % 4 != 0) return MOE_ERR_SHAPE;
  if (rows > (int64_t)1 << 30 || width > 65536) return MOE_ERR_LIMIT;
  return 0;
}

}  // namespace

extern "C" int moe_f32_gather_rows(const float* x, const int32_t* pos_to_row, int64_t T, int64_t R, int64_t H,
                                   int64_t k, float* xp, void* stream) {
  if (int rc = check_rows(R, H)) return rc;
  if (T < 0 || k <= 0) return MOE_ERR_SHAPE;
  if (T > (int64_t)1 << 30 || k > MOE_MAX_TOPK) return MOE_ERR_LIMIT;
  if (R == 0) return 0;
  MOE_CHECK_PTR(x);
  MOE_CHECK_PTR(xp);
  if (!pos_to_row) return MOE_ERR_NULL;
  hipLaunchKernelGGL(f32_gather_rows_kernel, dim3((unsigned)R), dim3(256), 0, (hipStream_t)stream, x, pos_to_row,
                     (int)T, (int)H, (int)k, xp);
  return moe_launch_status();
}

extern "C" int moe_f32_combine_fwd(const float* y, const float* gates, const int32_t* row_to_pos, int64_t T,
                                   int64_t H, int64_t k, float* out, void* stream) {
  if (int rc = check_rows(T, H)) return rc;
  if (k <= 0) return MOE_ERR_SHAPE;
  if (k > MOE_MAX_TOPK || T * k > (int64_t)1 << 30) return MOE_ERR_LIMIT;
  if (T == 0) return 0;
  MOE_CHECK_PTR(y);
  MOE_CHECK_PTR(out);
  if (!row_to_pos) return MOE_ERR_NULL;
  hipLaunchKernelGGL(f32_combine_fwd_kernel, dim3((unsigned)T), dim3(256), 0, (hipStream_t)stream, y, gates,
                     row_to_pos, (int)(T * k), (int)H, (int)k, out);
  return moe_launch_status();
}

extern "C" int moe_f32_combine_bwd(const float* dy, const float* y, const float* gates,
                                   const int32_t* pos_to_row, int64_t T, int64_t R, int64_t H, int64_t k,
                                   float* dyp, float* dgates, void* stream) {
  if (int rc = check_rows(R, H)) return rc;
  if (T < 0 || k <= 0) return MOE_ERR_SHAPE;
  if (T > (int64_t)1 << 30 || k > MOE_MAX_TOPK) return MOE_ERR_LIMIT;
  if (R == 0) return 0;
  MOE_CHECK_PTR(dy);
  MOE_CHECK_PTR(dyp);
  if (!pos_to_row) return MOE_ERR_NULL;
  if (dgates) MOE_CHECK_PTR(y);
  hipLaunchKernelGGL(f32_combine_bwd_kernel, dim3((unsigned)R), dim3(256), 0, (hipStream_t)stream, dy, y, gates,
                     pos_to_row, (int)T, (int)H, (int)k, dyp, dgates);
  return moe_launch_status();
}

extern "C" int moe_f32_permute_bwd(const float* dxp, const int32_t* row_to_pos, int64_t T, int64_t H, int64_t k,
                                   float* dx, void* stream) {
  if (int rc = check_rows(T, H)) return rc;
  if (k <= 0) return MOE_ERR_SHAPE;
  if (k > MOE_MAX_TOPK || T * k > (int64_t)1 << 30) return MOE_ERR_LIMIT;
  if (T == 0) return 0;
  MOE_CHECK_PTR(dxp);
  MOE_CHECK_PTR(dx);
  if (!row_to_pos) return MOE_ERR_NULL;
  hipLaunchKernelGGL(f32_permute_bwd_kernel, dim3((unsigned)T), dim3(256), 0, (hipStream_t)stream, dxp, row_to_pos,
                     (int)(T * k), (int)H, (int)k, dx);
  return moe_launch_status();
}

int moe_f32_permute_bwd_router(const float* dxp, const int32_t* row_to_pos, const float* gates, const float* dgates,
                               const int32_t* ids, const float* wr, int64_t T, int64_t H, int64_t k, float* dsel, float* dx,
                               void* stream) {
  if (int rc = check_rows(T, H)) return rc;
  if (k <= 0) return MOE_ERR_SHAPE;
  if (k > MOE_MAX_TOPK || T * k > (int64_t)1 << 30) return MOE_ERR_LIMIT;
  if (T == 0) return 0;
  if (dx) {
    MOE_CHECK_PTR(dxp);
    MOE_CHECK_PTR(wr);
    MOE_CHECK_PTR(dx);
  }
  if (!row_to_pos || !gates || !dgates || !ids || !dsel) return MOE_ERR_NULL;
  hipLaunchKernelGGL(f32_permute_bwd_router_kernel, dim3((unsigned)T), dim3(256), 0, (hipStream_t)stream, dxp, row_to_pos, gates,
                     dgates, ids, wr, (int)(T * k), (int)H, (int)k, dsel, dx);
  return moe_launch_status();
}

// The most rows of a segment: two workgroups for every compute unit, but eight rows for every wave.  (By rows, not so many parts
// an expert: the longest expert's rows are what a workgroup walks one after the other.  Every expert cut alike by the mean, and here, whole
// passes, us: 16384 tokens all with 1 of 128 experts, 1024 <-> 64, 1688 -> 1413; evenly 512 -> 507; 8192 all with 2 of 64, 2048 <-> 128, 1208 ->
// 1097; 4717, 2 of 64, 768 <-> 384, two thirds with two, 877 -> 843, evenly 622 and 629, the same kernels' times.)
static int router_segment_rows(int64_t R, int64_t H, int64_t E) {
  const int64_t cols = (H + RW_COLS - 1) / RW_COLS, cus = moe_compute_units();
  const int64_t want = 2 * cus / cols > 0 ? 2 * cus / cols : 1;
  int64_t L = (R + want - 1) / want;
  if (E * cols >= cus && L < 2 * (R / E)) L = 2 * (R / E);  // (the experts alone are enough workgroups: none of about the mean is cut)
  return (int)(L < 8 * RW_WAVES ? 8 * RW_WAVES : L);
}

int64_t moe_f32_router_wgrad_floats(int64_t R, int64_t H, int64_t E) {
  const int64_t L = router_segment_rows(R, H, E);
  return R > L ? (R / L + E) * H : 0;
}

// `partial`: moe_f32_router_wgrad_floats floats.
int moe_f32_router_wgrad(const float* xp, const float* dsel, const int32_t* offs, int64_t R, int64_t H, int64_t E, float* partial,
                         float* dwr, void* stream) {
  if (int rc = check_rows(R, H)) return rc;
  if (E <= 0) return MOE_ERR_SHAPE;
  if (E > MOE_MAX_EXPERTS) return MOE_ERR_LIMIT;
  MOE_CHECK_PTR(xp);
  MOE_CHECK_PTR(dwr);
  if (!dsel || !offs) return MOE_ERR_NULL;
  const RowCut cut{offs, (int)E, router_segment_rows(R, H, E)};
  const bool any = R > cut.L;  // (else no expert can have more)
  if (any) MOE_CHECK_PTR(partial);
  const hipStream_t s = (hipStream_t)stream;
  const unsigned cols = (unsigned)((H + RW_COLS - 1) / RW_COLS);
  hipLaunchKernelGGL(f32_router_wgrad_kernel, dim3(cols, (unsigned)(R / cut.L + E)), dim3(RW_WAVES * MOE_WAVE), 0, s, xp, dsel, cut,
                     (int)H, partial, dwr);
  if (!any) return moe_launch_status();
  if (const int rc = moe_launch_status()) return rc;
  hipLaunchKernelGGL(f32_router_wgrad_sum_kernel, dim3(cols, (unsigned)E), dim3(RS_WAVES * MOE_WAVE), 0, s, partial, cut, (int)H, dwr);
  return moe_launch_status();
}

extern "C" int moe_f32_swiglu_fwd(const float* g, const float* u, int64_t n, float* act, void* stream) {
  if (n < 0 || n % 4 != 0) return MOE_ERR_SHAPE;
  if (n == 0) return 0;
  if (n / 4 > (int64_t)0x7fffffff * 256) return MOE_ERR_LIMIT;
  MOE_CHECK_PTR(g);
  MOE_CHECK_PTR(u);
  MOE_CHECK_PTR(act);
  const long long n4 = n / 4;
  hipLaunchKernelGGL(f32_swiglu_fwd_kernel, dim3((unsigned)((n4 + 255) / 256)), dim3(256), 0, (hipStream_t)stream,
                     g, u, n4, act);
  return moe_launch_status();
}

extern "C" int moe_f32_swiglu_bwd(const float* dact, const float* g, const float* u, int64_t n, float* dg,
                                  float* du, void* stream) {
  if (n < 0 || n % 4 != 0) return MOE_ERR_SHAPE;
  if (n == 0) return 0;
  if (n / 4 > (int64_t)0x7fffffff * 256) return MOE_ERR_LIMIT;
  MOE_CHECK_PTR(dact);
  MOE_CHECK_PTR(g);
  MOE_CHECK_PTR(u);
  MOE_CHECK_PTR(dg);
  MOE_CHECK_PTR(du);
  const long long n4 = n / 4;
  hipLaunchKernelGGL(f32_swiglu_bwd_kernel, dim3((unsigned)((n4 + 255) / 256)), dim3(256), 0, (hipStream_t)stream,
                     dact, g, u, n4, dg, du);
  return moe_launch_status();
}
