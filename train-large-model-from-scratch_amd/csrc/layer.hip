// The layer body behind single calls.
//
// Forward only: the whole pass behind one call: routing, dispatch, row gather, the two
// grouped GEMMs and the combine (model/modules/mlp.py:101-167) enqueued back to back on the
// caller's stream, with every intermediate in a workspace the caller provides.  For callers that
// only want the output (inference, evaluation, a forward under no_grad): one crossing of the FFI
// boundary and two buffers instead of six crossings and a dozen.  Nothing here touches the GPU
// itself.  Above 64 tokens the kernels are the ones the separate entry points launch, in the same
// order, so the output holds the same bits; at most 64 tokens go to kernels of their own
// (moe_few_ok), which add the same products in another order: a token's output then depends on
// whether it came in a batch of 64 or of 65, by what another order of fp32 sums makes of it.
//
// Training: moe_layer_forward / moe_layer_backward enqueue one direction each (two dozen kernels
// between them).  What they replace is host work: a step of 512 tokens of a narrow layer has 0.1 ms of
// kernels, and took the host 0.42 ms when every launch was its own call from Python with its own
// allocations.
#include "common.h"
#include "internal.h"

namespace {

moe_launch_observer_fn g_observer = nullptr;

// Enqueues one step and tells the observer about it; leaves the calling function on an error.
#define MOE_STEP(name, call)    \
  do {                          \
    moe_observe(name, 0);       \
    const int rc_ = (call);     \
    moe_observe(name, 1);       \
    if (rc_) return rc_;        \
  } while (0)

constexpr int64_t ALIGN = 256;
int64_t up(int64_t n) { return (n + ALIGN - 1) / ALIGN * ALIGN; }

struct Carve {
  int64_t ids, gates, counts, offs, pos_to_row, row_to_pos, xp, act, y, dispatch, total;
};

// Room for the counts that selection and places, or histograms and scans, work on.
int64_t order_bytes(int64_t T, int64_t E, int64_t k) {
  const int64_t general = moe_dispatch_workspace_bytes(T * k, E);
  const int64_t place = moe_place_ok(T, E, k) ? moe_count_bytes(T, E) : 0;
  return place > general ? place : general;
}

Carve carve(int64_t T, int64_t H, int64_t E, int64_t I, int64_t k, bool with_xp = true) {
  const int64_t R = T * k;
  Carve c;
  int64_t at = 0;
  auto take = [&](int64_t bytes) {
    const int64_t here = at;
    at += up(bytes > 0 ? bytes : 1);
    return here;
  };
  c.ids = take(R * 4);
  c.gates = take(R * 4);
  c.counts = take(E * 4);
  c.offs = take((E + 1) * 4);
  c.pos_to_row = take(R * 4);
  c.row_to_pos = take(R * 4);
  c.xp = take(with_xp ? R * H * 2 : 0);
  c.act = take(R * I * 2);
  c.y = take(R * H * 2);
  c.dispatch = take(order_bytes(T, E, k));
  c.total = at;
  return c;
}

bool sizes_ok(int64_t T, int64_t H, int64_t E, int64_t I, int64_t k) {
  return T >= 0 && H > 0 && E > 0 && I > 0 && k > 0 && k <= MOE_MAX_TOPK && k <= E && E <= MOE_MAX_EXPERTS &&
         H <= 65536 && I <= 65536 && T <= ((int64_t)1 << 30) / k;
}

// Gate/up reads a token's row where it is, k times, and nobody else wants copies in expert order.
bool forward_in_place(int64_t T, int64_t H, int64_t E, int64_t I, int64_t k, int x_dtype) {
  return !moe_few_ok(T, H, E, I, k, x_dtype) && x_dtype == MOE_DT_BF16 && moe_rows_from_ok(T, H);
}

}  // namespace

extern "C" int64_t moe_ffn_forward_workspace_bytes(int64_t T, int64_t H, int64_t E, int64_t I, int64_t k) {
  if (!sizes_ok(T, H, E, I, k)) return 0;
  return carve(T, H, E, I, k).total;
}
int64_t moe_forward_only_scratch(int64_t T, int64_t H, int64_t E, int64_t I, int64_t k, int x_dtype) {
  if (!sizes_ok(T, H, E, I, k)) return 0;
  return carve(T, H, E, I, k, !forward_in_place(T, H, E, I, k, x_dtype)).total;
}

// The pass itself.  With `router` its product is part of it (see router.h), without it the logits are given.  `room`: what the workspace has to have.
static int forward_only(int64_t room, const void* x, int x_dtype, const void* logits, int logits_dtype, const MoeRouter* router,
                        const float* bias, const uint16_t* w1, const uint16_t* w3, const uint16_t* w2, int64_t T, int64_t H, int64_t E, int64_t I, int64_t k, void* out,
                        int out_dtype, void* workspace, int64_t workspace_bytes, void* stream) {
  if (T < 0 || H <= 0 || E <= 0 || I <= 0 || k <= 0 || H % 8 != 0 || I % 8 != 0) return MOE_ERR_SHAPE;
  if (!sizes_ok(T, H, E, I, k)) return MOE_ERR_LIMIT;
  if (x_dtype != MOE_DT_BF16 && x_dtype != MOE_DT_F32) return MOE_ERR_DTYPE;
  if (logits_dtype != MOE_DT_BF16 && logits_dtype != MOE_DT_F32) return MOE_ERR_DTYPE;
  if (out_dtype != MOE_DT_BF16 && out_dtype != MOE_DT_F32) return MOE_ERR_DTYPE;
  if (T == 0) return 0;
  MOE_CHECK_PTR(x);
  const bool few_logits = router && moe_router_few_ok(T, H, E, k);
  if (router) {
    MOE_CHECK_PTR(router->wr);
    MOE_CHECK_PTR(router->logits);
    if (few_logits ? x_dtype != MOE_DT_BF16 || router->wr_dtype != MOE_DT_BF16 : !moe_router_select_ok(T, H, E, k, router->wr_dtype))
      return few_logits ? MOE_ERR_DTYPE : MOE_ERR_LIMIT;
  } else {
    MOE_CHECK_PTR(logits);
  }
  MOE_CHECK_PTR(w1);
  MOE_CHECK_PTR(w3);
  MOE_CHECK_PTR(w2);
  MOE_CHECK_PTR(out);
  MOE_CHECK_PTR(workspace);
  const bool in_place = forward_in_place(T, H, E, I, k, x_dtype);
  const Carve c = carve(T, H, E, I, k, !in_place);
  if (workspace_bytes < room || workspace_bytes < c.total) return MOE_ERR_WORKSPACE;
  char* ws = (char*)workspace;
  const int64_t R = T * k;
  int32_t* ids = (int32_t*)(ws + c.ids);
  float* gates = (float*)(ws + c.gates);
  int32_t* counts = (int32_t*)(ws + c.counts);
  int32_t* offs = (int32_t*)(ws + c.offs);
  int32_t* pos_to_row = (int32_t*)(ws + c.pos_to_row);
  int32_t* row_to_pos = (int32_t*)(ws + c.row_to_pos);
  uint16_t* xp = (uint16_t*)(ws + c.xp);
  uint16_t* act = (uint16_t*)(ws + c.act);
  uint16_t* y = (uint16_t*)(ws + c.y);
  hipStream_t st = (hipStream_t)stream;
  if (few_logits) MOE_STEP("moe_router_few", moe_router_few((const uint16_t*)x, (const uint16_t*)router->wr, T, H, E, router->logits, st));
  if (router) {
    logits = router->logits;
    logits_dtype = MOE_DT_BF16;
    bias = router->bias;
  }
  if (moe_gateup_one_ok(T, E, k)) {
    MOE_STEP("moe_gateup_one", moe_gateup_one(x, x_dtype, logits, logits_dtype, bias, w1, w3, H, E, I, k, ids, gates, act, st));
    MOE_STEP("moe_down_one", moe_down_one(act, ids, gates, w2, H, E, I, k, out, out_dtype, st));
    return 0;
  }
  const bool few = moe_few_ok(T, H, E, I, k, x_dtype), place = !few && moe_place_ok(T, E, k);
  const bool selects = few && moe_gateup_few_selects(T, E, I, k);  // gate/up does the selection
  uint16_t* rows = in_place ? nullptr : xp;
  const bool selected = router && !few_logits, at_once = place && !selected && moe_select_place_ok(logits, T, E, k);
  if (selected)
    MOE_STEP("moe_router_select", moe_router_select(*router, T, H, E, k, ids, gates, place ? ws + c.dispatch : nullptr, st));
  else if (at_once)
    MOE_STEP("moe_select_place", moe_select_place(x, x_dtype, logits, logits_dtype, bias, T, H, E, k, ids, gates, counts, offs,
                                                  pos_to_row, row_to_pos, nullptr, rows, MOE_DT_BF16, stream));
  else if (place)
    MOE_STEP("moe_select_count", moe_select_count(logits, logits_dtype, bias, T, E, k, ids, gates, ws + c.dispatch, stream));
  else if (!selects)
    MOE_STEP("moe_router_topk_fwd", moe_router_topk_fwd(logits, logits_dtype, bias, T, E, k, ids, gates, stream));
  if (few) {  // rows stay in routed order: no dispatch, no gather
    if (selects)
      MOE_STEP("moe_gateup_few", moe_gateup_few_select(x, x_dtype, logits, logits_dtype, bias, w1, w3, T, H, E, I, k,
                                                              ids, gates, act, st));
    else
      MOE_STEP("moe_gateup_few", moe_gateup_few(x, x_dtype, ids, w1, w3, T, H, E, I, k, act, st));
    if (moe_down_one_ok(T, k)) {
      MOE_STEP("moe_down_one", moe_down_one(act, ids, gates, w2, H, E, I, k, out, out_dtype, st));
      return 0;
    }
    MOE_STEP("moe_down_few", moe_down_few(act, ids, w2, T, H, E, I, k, y, st));
    MOE_STEP("moe_combine_in_order", moe_combine_in_order(y, gates, T, H, k, out, out_dtype, st));
    return 0;
  }
  if (place && !at_once) {
    MOE_STEP("moe_place_rows", moe_place_rows(x, x_dtype, ids, ws + c.dispatch, T, H, E, k, counts, offs, pos_to_row,
                                              row_to_pos, nullptr, rows, MOE_DT_BF16, false, stream));
  } else if (!place) {
    MOE_STEP("moe_histogram_scan_checked",
             moe_histogram_scan(ids, R, E, counts, offs, pos_to_row, row_to_pos, ws + c.dispatch,
                                moe_dispatch_workspace_bytes(R, E), stream));
    if (!in_place)
      MOE_STEP(k > 1 ? "moe_permute_fwd_scatter" : "moe_permute_fwd",
               k > 1 ? moe_permute_fwd_scatter(x, x_dtype, row_to_pos, T, H, k, xp, stream)
                     : moe_permute_fwd(x, x_dtype, pos_to_row, R, H, k, xp, stream));
  }
  MOE_STEP("moe_gemm_gateup_swiglu_fwd",
           in_place ? moe_gemm_gateup_from((const uint16_t*)x, pos_to_row, T, k, w1, w3, offs, E, H, I, nullptr, act, stream)
                    : moe_gemm_gateup_swiglu_fwd(xp, w1, w3, offs, E, R, H, I, nullptr, nullptr, act, stream));
  MOE_STEP("moe_gemm_down_fwd", moe_gemm_down_fwd(act, w2, offs, E, R, H, I, y, stream));
  MOE_STEP("moe_combine_fwd", moe_combine_fwd(y, gates, row_to_pos, T, H, k, out, out_dtype, stream));
  return 0;
}

extern "C" int moe_ffn_forward(const void* x, int x_dtype, const void* logits, int logits_dtype,
                               const float* bias, const uint16_t* w1, const uint16_t* w3, const uint16_t* w2,
                               int64_t T, int64_t H, int64_t E, int64_t I, int64_t k, void* out,
                               int out_dtype, void* workspace, int64_t workspace_bytes, void* stream) {
  return forward_only(moe_ffn_forward_workspace_bytes(T, H, E, I, k), x, x_dtype, logits, logits_dtype, nullptr, bias, w1, w3, w2, T, H, E, I, k,
                      out, out_dtype, workspace, workspace_bytes, stream);
}

int moe_forward_only(const MoeRouter* router, const void* x, int x_dtype, const void* logits, int logits_dtype, const float* bias,
                     const uint16_t* w1, const uint16_t* w3, const uint16_t* w2, int64_t T, int64_t H, int64_t E, int64_t I, int64_t k,
                     void* out, int out_dtype, void* workspace, int64_t workspace_bytes, void* stream) {
  return forward_only(0, x, x_dtype, logits, logits_dtype, router, bias, w1, w3, w2, T, H, E, I, k, out, out_dtype, workspace,
                      workspace_bytes, stream);
}

int moe_router_logits(const uint16_t* x, const uint16_t* wr, int64_t T, int64_t H, int64_t E, uint16_t* logits,
                      void* stream) {
  MOE_STEP("moe_router_few", moe_router_few(x, wr, T, H, E, logits, (hipStream_t)stream));
  return 0;
}

void moe_observe(const char* name, int after) {
  if (g_observer) g_observer(name, after);
}

extern "C" void moe_set_launch_observer(moe_launch_observer_fn fn) { g_observer = fn; }

// ---- training: one call per direction -------------------------------------------------------------

namespace {

struct Scratch {
  char* base;
  int64_t at, have;
  void* take(int64_t bytes) {
    void* p = base ? base + at : nullptr;
    at += up(bytes > 0 ? bytes : 1);
    return p;
  }
  bool fits() const { return at <= have; }
};

struct FwdScratch {
  uint16_t* y;
  void* dispatch;
  FwdScratch(Scratch& s, int64_t T, int64_t H, int64_t E, int64_t k, bool with_y = true) {
    y = (uint16_t*)s.take(with_y ? T * k * H * 2 : 0);
    dispatch = s.take(order_bytes(T, E, k));
  }
};

// Whether the weight gradients go to the kernel that takes all stacks at once (wgrad.hip).  Decided from shapes alone: where
// one stack's 256 x 256 tiles are at most one for every compute unit, and up to four where its launch of 128 x 128 tiles, three to
// a compute unit, comes to no more rounds than tiles of 256 x 256 do where every problem (w2's stack, and one or two for the others) begins
// a round of its own.  (The tiled kernel runs its problems in one launch, so it has fewer partial rounds than are counted here; it still pads
// the matrices to 256 and has no part of an expert's rows to deal.  Where the line lies was measured with one launch on either side, whole
// steps of 90 drawn layers, bf16 and fp32 results, tiled kernel -> small one, us: the 69 taken are 1.07 times as fast in the mean, most of all by
// skewed shares (5953 tokens, 4 of 128, 336 <-> 536, 565 -> 312; 56149 rows of 8, 2688 <-> 704, 4230 -> 2345), 15 of them slower, seven by
// more than 3 % (1392 rows of 128, 384 <-> 192, 67 -> 75; 9269 tokens, 6 of 24, 2912 <-> 432, 2107 -> 2268); the 21 past the line come
// to 1.005, from 0.91 to 1.09, but for one by Zipf's shares (15833 tokens, 2 of 128, 960 <-> 256, 679 -> 434).)
constexpr int64_t WTILE = 256;
constexpr int64_t MULTI_ROUNDS = 4;
bool wgrad_multi(int64_t E, int64_t M, int64_t N, int64_t R) {
  const int64_t cus = moe_compute_units();
  const int64_t tiles = E * ((M + WTILE - 1) / WTILE) * ((N + WTILE - 1) / WTILE);
  const int64_t rounds = (tiles + cus - 1) / cus + (M % WTILE == 0 ? (2 * tiles + cus - 1) / cus : 2 * ((tiles + cus - 1) / cus));
  return R > 0 && (tiles <= cus || (tiles <= MULTI_ROUNDS * cus && rounds * cus >= E * ((M + 127) / 128) * ((N + 127) / 128)));
}

// Router weight gradient: the tokens are cut into slices, as many as give every compute unit a job, of at least 64
// tokens, at most 16 (their partial sums are written and read once more: 16384 tokens, 64 experts, 2048 wide, products
// and sums 28 us with 16 slices, 30 with 32, 38 with 8; 4096 tokens, 128 experts, 1024 wide 17, 19 and 18).
// Up to 1024 tokens are one slice, as long a job as an expert's may be, and go straight to the result, without the launch that
// adds slices up (whole steps, us: 115 tokens, 8 of 96 experts, 1216 <-> 320, 151 -> 147; 581, 6 of 64, 304 <-> 1984, 311 -> 303; 771,
// 6 of 12, 3392 <-> 192, 255 -> 247; 1003 of 128 845 and 849).
constexpr int64_t ROUTER_WHOLE = 1024;
struct RouterSlices {
  int64_t slices, rows, Ep;
};
RouterSlices router_slices(int64_t T, int64_t H, int64_t E) {
  const int64_t tiles = (H + WTILE - 1) / WTILE;
  int64_t S = moe_compute_units() / tiles;
  if (S > 16) S = 16;
  if (S > (T + 63) / 64) S = (T + 63) / 64;
  if (T <= ROUTER_WHOLE) S = 1;
  if (S < 1) S = 1;
  RouterSlices r;
  r.rows = T > 0 ? ((T + S - 1) / S + 63) / 64 * 64 : 64;
  r.slices = T > 0 ? (T + r.rows - 1) / r.rows : 1;
  r.Ep = (E + 7) / 8 * 8;
  return r;
}

struct BwdScratch {
  uint16_t *dyp, *dg, *dxp;
  uint32_t* row_at;
  float *part, *wpart[3], *rpart;
  uint16_t* dlogits;
  BwdScratch(Scratch& s, int64_t T, int64_t H, int64_t E, int64_t I, int64_t k, bool with_dxp = true, bool with_dyp = true,
             bool with_places = false) {
    const int64_t R = T * k;
    dyp = (uint16_t*)s.take(with_dyp ? R * H * 2 : 0);
    dg = (uint16_t*)s.take(R * I * 4);
    dxp = (uint16_t*)s.take(with_dxp ? R * H * 2 : 0);
    part = (float*)s.take(moe_dgate_blocks(I) * R * 4);
    const RouterSlices rs = router_slices(T, H, E);
    dlogits = (uint16_t*)s.take(T * rs.Ep * 4);
    rpart = (float*)s.take(rs.slices * rs.Ep * H * 4);
    for (float*& w : wpart) w = (float*)s.take(wgrad_multi(E, I, H, R) ? moe_wgrad_multi_part_bytes(R, H, I) : 0);
    row_at = with_places ? (uint32_t*)s.take(R * 4) : nullptr;
  }
};

// Rows of one slot without a gate: down leaves them where they came from, and there is nothing to combine.  (That pass, and
// its counterpart behind the gate/up input gradient, each move every row in and out: 32768 rows of 16 experts, 4096 wide, 82 us
// of 3700 either way; a step of 24 drawn sizes, 288 to 46000 rows, 1.05 to 1.15 times as fast without the two.)
bool out_in_place(const moe_layer_forward_args& a) { return a.k == 1 && !a.gates && !a.residual && a.out_dtype == MOE_DT_BF16; }
// (dxp is dx but for the order, and nothing else is to be added)
bool dx_in_place(const moe_layer_backward_args& a) {
  const bool router = a.wr && !a.dgates;
  return a.k == 1 && a.dx && !a.dxp && !router && a.dx_dtype == MOE_DT_BF16;
}

bool over(const void* p, int64_t bytes, const void* q, int64_t q_bytes) {
  const uintptr_t at = (uintptr_t)p, other = (uintptr_t)q;
  return q && at < other + q_bytes && other < at + bytes;
}

// The output's gradient is theirs too but for the order.  Where the weight gradients are tiled both of its products read it where it is, and the
// pass that put it in order goes with its buffer.  Steps with the pass and without, the same bits, us: 32768 rows of 16 experts, 4096 <-> 1536, even
// and by Dirichlet's shares 3483 -> 3407 and 3458 -> 3378; 12000 of 64, 2048 <-> 1024, 743 -> 725; 30000 of 32, 1000 <-> 1000, 728 -> 711; 60000 of 128 by
// Dirichlet's shares, 768 <-> 256, 610 -> 578; 50000 of 96, 512 <-> 640, 542 -> 542.
// A result that lies over it would be there before the last of the two has read it: then it is copied first, as everywhere else.
bool dout_in_place(const moe_layer_backward_args& a) {
  if (a.k != 1 || a.gates || a.dout_dtype != MOE_DT_BF16 || !moe_rows_from_ok(a.T, a.H) || a.T < 160 * a.E || wgrad_multi(a.E, a.I, a.H, a.T))
    return false;
  const int64_t rows = a.T * a.H, bytes = rows * 2;
  const auto size = [](int64_t n, int64_t dtype) { return n * (dtype == MOE_DT_F32 ? 4 : 2); };
  bool apart = !over(a.dout, bytes, a.dx, size(rows, a.dx_dtype)) && !over(a.dout, bytes, a.dxp, bytes);
  for (int i = 0; i < 3; ++i) apart = apart && !over(a.dout, bytes, a.dw[i], size(a.E * a.I * a.H, a.dw_dtype[i]));
  return apart;
}

bool dtype_ok(int64_t d) { return d == MOE_DT_BF16 || d == MOE_DT_F32; }

}  // namespace

extern "C" int64_t moe_router_wgrad_workspace_bytes(int64_t T, int64_t H, int64_t E) {
  if (T < 0 || H <= 0 || E <= 0 || T > (int64_t)1 << 30 || H > 65536 || E > MOE_MAX_EXPERTS) return 0;
  const RouterSlices r = router_slices(T, H, E);
  return r.slices * r.Ep * H * 4;
}

extern "C" int moe_router_wgrad(const uint16_t* dlogits, const uint16_t* x, int64_t T, int64_t H, int64_t E,
                                void* dw, int dw_dtype, void* workspace, int64_t workspace_bytes, void* stream) {
  if (T < 0 || H <= 0 || E <= 0 || H % 8 != 0 || E % 8 != 0) return MOE_ERR_SHAPE;
  if (T > (int64_t)1 << 30 || H > 65536 || E > MOE_MAX_EXPERTS) return MOE_ERR_LIMIT;
  if (!dtype_ok(dw_dtype)) return MOE_ERR_DTYPE;
  MOE_CHECK_PTR(dw);
  MOE_CHECK_PTR(workspace);
  MOE_CHECK_PTR(dlogits);
  MOE_CHECK_PTR(x);
  if (workspace_bytes < moe_router_wgrad_workspace_bytes(T, H, E)) return MOE_ERR_WORKSPACE;
  const RouterSlices r = router_slices(T, H, E);
  MoeWgradStack router{};
  router.a = dlogits, router.b = x, router.out = dw, router.part = (float*)workspace;
  router.M = router.lda = E, router.N = router.ldb = H;
  router.dtype = dw_dtype;
  return moe_wgrad_multi({}, 0, &router, nullptr, E, 0, H, 0, T, r.slices, r.rows, (hipStream_t)stream);
}

extern "C" int64_t moe_layer_scratch_bytes(int64_t T, int64_t H, int64_t E, int64_t I, int64_t k, int backward) {
  if (!sizes_ok(T, H, E, I, k)) return 0;
  Scratch s{nullptr, 0, 0};
  if (backward) BwdScratch(s, T, H, E, I, k);
  else FwdScratch(s, T, H, E, k);
  return s.at;
}

int64_t moe_forward_scratch(const moe_layer_forward_args* a) {
  if (!sizes_ok(a->T, a->H, a->E, a->I, a->k)) return 0;
  Scratch s{nullptr, 0, 0};
  FwdScratch(s, a->T, a->H, a->E, a->k, !out_in_place(*a));
  return s.at;
}

int64_t moe_backward_scratch(const moe_layer_backward_args* a) {
  if (!sizes_ok(a->T, a->H, a->E, a->I, a->k)) return 0;
  Scratch s{nullptr, 0, 0};
  BwdScratch(s, a->T, a->H, a->E, a->I, a->k, a->dx && !a->dxp && !dx_in_place(*a), !dout_in_place(*a),
             !a->xp && wgrad_multi(a->E, a->I, a->H, a->T * a->k));
  return s.at;
}

// Training steps in which nobody but gate/up and the gradients of its weights would read rows in expert order: both read x where it
// is, a lane's offset a row, those of a k-tile of the gradients asked for a k-tile ahead.  Besides the pass the copies (R x H x 2 bytes, a
// step's largest buffer) go from memory's traffic and from what is held between the passes.  Steps with the copies and this one, the same bits, us:
// 16384 tokens, 8 of 64 experts, 2048 <-> 1024, 4992 -> 4909; 8192 with norm and fp32 gradients 2933 -> 2906; 4096, 8 of 128, 1024 <-> 256, fp32
// gradients, 409 -> 394; 9000, 4 of 64 by Zipf's shares, 1416 <-> 1000, 2116 -> 2091; 16000, 1 of 32, 2000 <-> 800, 980 -> 971; 8000, 8 of
// 128, 256 <-> 640, 500 -> 500.  Tiles of one or two k-tiles have none to ask ahead in: rows an expert, 64 experts, 2048 <-> 1024, 250 947 -> 932;
// 125 676 -> 687; 100 653 -> 675; 75 629 -> 651; 162 of 32 474 -> 472.  Nor are they for rows that are short beside the products: of 50 sizes drawn,
// 1.016 in the mean, those with I past 2 H 0.999: 8126, 4 of 128 by Zipf's shares, 384 <-> 1600, 1181 -> 1224; 7824, 4 of 96, 448 <-> 1152, 626 -> 630.  (Most of 128 experts by
// Zipf's shares have few rows where the mean is 160: 1024 <-> 256, 165 / 200 / 250 rows 352 -> 358, 404 -> 412, 488 -> 485, even 307 -> 302, 339 -> 324, 393 -> 376.)
// The kernel for small weight gradients finds where its rows are in a list that the pass over the output's gradient leaves (which is by token where k > 1
// and rows are at most 2048 long): 8192, 2 of 8 by Zipf's shares, 1024 <-> 512, 299 -> 282; 3333, 3 of 12, 1416 <-> 568, 294 -> 287; 8000, 4 of 16, 768 <->
// 768, 515 -> 502; 10892, 6 of 12, 448 <-> 192, 371 -> 336; 2000, 8 of 64, 320 <-> 256, 121 -> 116; 10342, 2 of 4, 832 <-> 704, fp32 gradients, 421 -> 419; of 94
// sizes drawn, those apart that the host bounds, 1.025 in the mean.  What the copies cost goes with k H, what lines from anywhere cost in the products with I:
// 2 of 4, 960 <-> 1856, 462 -> 473, 1024 <-> 1152, 496 -> 506, 2 of 64, 352 <-> 1416, 280 -> 285, 4 of 16, 512 <-> 1152, 310 -> 314, not taken.
bool moe_layer_rows_from_ok(int64_t T, int64_t H, int64_t E, int64_t I, int64_t k) {
  return T > 0 && sizes_ok(T, H, E, I, k) && moe_rows_from_ok(T, H) &&
         (wgrad_multi(E, I, H, T * k) ? k > 1 && k <= MOE_WAVE && H <= 2048 && 2 * I <= k * H : I <= 2 * H && T * k >= 160 * E);
}

// (`router` and `table`: see router.h; `in_place`: no xp, x is in bf16)
static int layer_forward(const moe_layer_forward_args* a, const MoeRouter* router, const void* table, bool in_place, void* stream) {
  if (!a) return MOE_ERR_NULL;
  const int64_t T = a->T, H = a->H, E = a->E, I = a->I, k = a->k, R = T * k;
  if (T < 0 || H <= 0 || E <= 0 || I <= 0 || k <= 0 || H % 8 != 0 || I % 8 != 0) return MOE_ERR_SHAPE;
  if (!sizes_ok(T, H, E, I, k)) return MOE_ERR_LIMIT;
  if (!dtype_ok(a->x_dtype) || !dtype_ok(a->out_dtype) || (a->logits && !dtype_ok(a->logits_dtype)))
    return MOE_ERR_DTYPE;
  MOE_CHECK_PTR(a->counts);
  MOE_CHECK_PTR(a->offs);
  MOE_CHECK_PTR(a->scratch);
  if (T > 0) {
    MOE_CHECK_PTR(a->x);
    MOE_CHECK_PTR(a->w1);
    MOE_CHECK_PTR(a->w3);
    MOE_CHECK_PTR(a->w2);
    MOE_CHECK_PTR(a->out);
    MOE_CHECK_PTR(a->ids);
    MOE_CHECK_PTR(a->pos_to_row);
    MOE_CHECK_PTR(a->row_to_pos);
    if (!in_place) MOE_CHECK_PTR(a->xp);
    else if (a->x_dtype != MOE_DT_BF16) return MOE_ERR_DTYPE;
    MOE_CHECK_PTR(a->act);
  }
  if (a->logits && !a->gates) return MOE_ERR_NULL;
  Scratch s{(char*)a->scratch, 0, a->scratch_bytes};
  const FwdScratch ws(s, T, H, E, k, !out_in_place(*a));
  if (!s.fits()) return MOE_ERR_WORKSPACE;
  if (router && T > 0) {
    if (!a->gates) return MOE_ERR_NULL;
    if (moe_place_ok(T, E, k)) table = ws.dispatch;
    MOE_STEP("moe_router_select", moe_router_select(*router, T, H, E, k, a->ids, a->gates, moe_place_ok(T, E, k) ? ws.dispatch : nullptr,
                                                    (hipStream_t)stream));
  }
  if (a->logits && !table && moe_select_place_ok(a->logits, T, E, k)) {
    MOE_STEP("moe_select_place", moe_select_place(a->x, (int)a->x_dtype, a->logits, (int)a->logits_dtype, a->bias, T, H, E, k, a->ids,
                                                  a->gates, a->counts, a->offs, a->pos_to_row, a->row_to_pos, a->bad_ids, a->xp,
                                                  MOE_DT_BF16, stream));
  } else if ((a->logits || table) && moe_place_ok(T, E, k)) {
    if (!table)
      MOE_STEP("moe_select_count", moe_select_count(a->logits, (int)a->logits_dtype, a->bias, T, E, k, a->ids, a->gates,
                                                    ws.dispatch, stream));
    MOE_STEP("moe_place_rows", moe_place_rows(a->x, (int)a->x_dtype, a->ids, table ? table : ws.dispatch, T, H, E, k, a->counts,
                                              a->offs, a->pos_to_row, a->row_to_pos, a->bad_ids, a->xp, MOE_DT_BF16, false,
                                              stream));
  } else if (!a->logits && !table && moe_count_ok(T, E, k)) {
    MOE_STEP("moe_count_ids", moe_count_ids(a->ids64, a->ids, T, E, ws.dispatch, stream));
    MOE_STEP("moe_place_rows", moe_place_rows(a->x, (int)a->x_dtype, a->ids, ws.dispatch, T, H, E, k, a->counts, a->offs,
                                              a->pos_to_row, a->row_to_pos, a->bad_ids, a->xp, MOE_DT_BF16, true, stream));
  } else {
    if (a->logits)
      MOE_STEP("moe_router_topk_fwd", moe_router_topk_fwd(a->logits, (int)a->logits_dtype, a->bias, T, E, k, a->ids,
                                                          a->gates, stream));
    else if (a->ids64 && R > 0)
      MOE_STEP("moe_narrow_ids", moe_narrow_ids(a->ids64, R, a->ids, (hipStream_t)stream));
    MOE_STEP("moe_histogram_scan_checked",
             moe_histogram_scan_checked(a->ids, R, E, a->counts, a->offs, a->pos_to_row, a->row_to_pos, a->bad_ids,
                                        ws.dispatch, moe_dispatch_workspace_bytes(R, E), stream));
    if (T == 0) return 0;
    if (!in_place)
      MOE_STEP(k > 1 ? "moe_permute_fwd_scatter" : "moe_permute_fwd",
               k > 1 ? moe_permute_fwd_scatter(a->x, (int)a->x_dtype, a->row_to_pos, T, H, k, a->xp, stream)
                     : moe_permute_fwd(a->x, (int)a->x_dtype, a->pos_to_row, R, H, k, a->xp, stream));
  }
  if (in_place)
    MOE_STEP("moe_gemm_gateup_swiglu_fwd_blocked",
             moe_gemm_gateup_from((const uint16_t*)a->x, a->pos_to_row, T, k, a->w1, a->w3, a->offs, E, H, I, a->gu, a->act, stream));
  else if (a->gu)
    MOE_STEP("moe_gemm_gateup_swiglu_fwd_blocked",
             moe_gemm_gateup_swiglu_fwd_blocked(a->xp, a->w1, a->w3, a->offs, E, R, H, I, a->gu, a->act, stream));
  else
    MOE_STEP("moe_gemm_gateup_swiglu_fwd",
             moe_gemm_gateup_swiglu_fwd(a->xp, a->w1, a->w3, a->offs, E, R, H, I, nullptr, nullptr, a->act, stream));
  if (out_in_place(*a)) {
    MOE_STEP("moe_gemm_down_fwd", moe_gemm_down_to(a->act, a->w2, a->offs, E, R, H, I, (uint16_t*)a->out, a->pos_to_row, stream));
    return 0;
  }
  MOE_STEP("moe_gemm_down_fwd", moe_gemm_down_fwd(a->act, a->w2, a->offs, E, R, H, I, ws.y, stream));
  if (a->residual)
    MOE_STEP("moe_combine_fwd_residual",
             moe_combine_fwd_residual(ws.y, a->gates, a->row_to_pos, a->residual, T, H, k, a->out,
                                      (int)a->out_dtype, stream));
  else
    MOE_STEP("moe_combine_fwd", moe_combine_fwd(ws.y, a->gates, a->row_to_pos, T, H, k, a->out, (int)a->out_dtype,
                                                stream));
  return 0;
}

extern "C" int moe_layer_forward(const moe_layer_forward_args* a, void* stream) {
  return layer_forward(a, nullptr, nullptr, false, stream);
}

int moe_selected_layer_forward(const moe_layer_forward_args* a, const MoeRouter* router, const void* table, void* stream) {
  return layer_forward(a, router, table, a && !a->xp, stream);
}

// (`in_place`: no xp, its rows are xn's; `norm`: see router.h)
static int layer_backward(const moe_layer_backward_args* a, bool in_place, const MoeNormBackward* norm, void* stream) {
  if (!a) return MOE_ERR_NULL;
  const int64_t T = a->T, H = a->H, E = a->E, I = a->I, k = a->k, R = T * k;
  if (T < 0 || H <= 0 || E <= 0 || I <= 0 || k <= 0 || H % 8 != 0 || I % 8 != 0) return MOE_ERR_SHAPE;
  if (!sizes_ok(T, H, E, I, k)) return MOE_ERR_LIMIT;
  if (!dtype_ok(a->dout_dtype) || !dtype_ok(a->dx_dtype) || !dtype_ok(a->dlogits_dtype) || !dtype_ok(a->dwr_dtype))
    return MOE_ERR_DTYPE;
  for (int i = 0; i < 3; ++i)
    if (!dtype_ok(a->dw_dtype[i])) return MOE_ERR_DTYPE;
  // (a result that is not asked for is NULL; here, so that it does not depend on which kernel the shapes pick)
  for (const void* p : {a->dw[0], a->dw[1], a->dw[2], a->dwr, a->dx, (void*)a->dxp, (void*)a->wr, (void*)a->xn})
    if (!aligned16(p)) return MOE_ERR_ALIGN;
  MOE_CHECK_PTR(a->offs);
  MOE_CHECK_PTR(a->scratch);
  const bool router = a->wr != nullptr;                               // the router product is part of the layer
  const bool to_logits = !a->dgates && (a->dlogits || router);        // ... and the gradient goes through it here
  if (T > 0) {
    MOE_CHECK_PTR(a->dout);
    MOE_CHECK_PTR(a->pos_to_row);
    MOE_CHECK_PTR(a->row_to_pos);
    MOE_CHECK_PTR(in_place ? a->xn : a->xp);
    MOE_CHECK_PTR(a->gu);
    MOE_CHECK_PTR(a->act);
    MOE_CHECK_PTR(a->w1);
    MOE_CHECK_PTR(a->w3);
    MOE_CHECK_PTR(a->w2);
    if ((to_logits || a->dgates) && (!a->gates || !a->ids)) return MOE_ERR_NULL;
    if (a->dwr && (!router || !a->xn)) return MOE_ERR_NULL;
  }
  if (in_place && !moe_layer_rows_from_ok(T, H, E, I, k)) return MOE_ERR_LIMIT;
  if (norm && (!router || !to_logits || !a->dx || a->dxp || a->dlogits || !moe_norm_rows_ok(T, H))) return MOE_ERR_SHAPE;
  Scratch s{(char*)a->scratch, 0, a->scratch_bytes};
  const bool dout_stays = dout_in_place(*a);
  const bool multi = wgrad_multi(E, I, H, R);
  const BwdScratch ws(s, T, H, E, I, k, a->dx && !a->dxp && !dx_in_place(*a), !dout_stays, in_place && multi);
  if (!s.fits()) return MOE_ERR_WORKSPACE;
  hipStream_t st = (hipStream_t)stream;
  uint16_t* dxp = a->dxp ? a->dxp : ws.dxp;
  const uint16_t* dyp = dout_stays ? (const uint16_t*)a->dout : ws.dyp;
  if (R > 0 && !dout_stays) {
    if (in_place && multi)
      MOE_STEP("moe_combine_bwd_by_token", moe_combine_bwd_places(a->dout, (int)a->dout_dtype, a->gates, a->row_to_pos, T, H, k, ws.dyp,
                                                                  ws.row_at, st));
    else if (k > 1 && H <= 2048)
      MOE_STEP("moe_combine_bwd_by_token", moe_combine_bwd_by_token(a->dout, (int)a->dout_dtype, nullptr, a->gates,
                                                                    a->row_to_pos, T, H, k, ws.dyp, nullptr, stream));
    else
      MOE_STEP("moe_combine_bwd", moe_combine_bwd(a->dout, (int)a->dout_dtype, nullptr, a->gates, a->pos_to_row, R, H,
                                                  k, ws.dyp, nullptr, stream));
  }
  // dg and du side by side where their two weight gradients can come out of one launch of the tiled kernel: both
  // wanted into results of one kind, no 256-row tile of the stacked result across the halves
  const bool pair = R > 0 && a->dw[0] && a->dw[1] && I % WTILE == 0 && !multi && a->dw_dtype[0] == a->dw_dtype[1] &&
                    a->dw_accumulate[0] == a->dw_accumulate[1];
  uint16_t* dg = ws.dg;
  uint16_t* du = pair ? ws.dg + I : ws.dg + R * I;
  float* part = (to_logits || a->dgates) ? ws.part : nullptr;
  MOE_STEP("moe_gemm_dgrad_down_swiglu_bwd_blocked",
           dout_stays ? moe_gemm_dgrad_down_from(dyp, a->pos_to_row, T, k, a->w2, a->gu, a->offs, E, H, I, dg, du, pair ? 2 * I : 0, part,
                                                 stream)
                      : moe_gemm_dgrad_down_swiglu_bwd_blocked(dyp, a->w2, a->gu, a->offs, E, R, H, I, dg, du, pair ? 2 * I : 0, part,
                                                               stream));
  if (a->dgates && R > 0)
    MOE_STEP("moe_dgates_from_blocks_by_pos", moe_dgates_from_blocks_by_pos(part, moe_dgate_blocks(I), a->gates,
                                                                            a->pos_to_row, R, a->dgates, stream));
  const RouterSlices rs = router_slices(T, H, E);
  // (for the router's weight gradient the rows of dlogits are padded to a multiple of 8 columns)
  const bool own = !a->dlogits, with_dx = router && a->dx;
  void* dlogits = own ? ws.dlogits : a->dlogits;
  const int64_t ld = own ? rs.Ep : E;
  const int dlogits_dtype = own ? MOE_DT_BF16 : (int)a->dlogits_dtype;
  if (to_logits && !with_dx && R > 0)
    MOE_STEP("moe_router_bwd_from_blocks", moe_router_bwd_from_blocks(part, moe_dgate_blocks(I), a->gates, a->ids, a->row_to_pos, T,
                                                                      E, k, ld, dlogits, dlogits_dtype, st));
  const bool dx_stays = dx_in_place(*a);
  if (a->dx || a->dxp)
    MOE_STEP(pair ? "moe_gemm_dgrad_gateup_packed" : "moe_gemm_dgrad_gateup",
             moe_gemm_dgrad_gateup_to(dg, du, pair ? 2 * I : 0, a->w1, a->w3, a->offs, E, R, H, I,
                                      dx_stays ? (uint16_t*)a->dx : dxp, dx_stays ? a->pos_to_row : nullptr, stream));
  if (a->dx && T > 0 && !dx_stays) {  // (before the weight gradients: the router's reads dlogits)
    if (norm)
      MOE_STEP("moe_rmsnorm_bwd_rows",
               moe_rmsnorm_bwd_rows(*norm, dxp, a->row_to_pos, part, moe_dgate_blocks(I), a->gates, a->ids, a->wr, T, H, k, ld,
                                    ws.dlogits, a->dx, st));
    else if (router && to_logits)
      MOE_STEP("moe_permute_bwd_router",
               moe_permute_bwd_router(dxp, a->row_to_pos, part, moe_dgate_blocks(I), a->gates, a->ids, a->wr, T, H, k, ld, dlogits,
                                      dlogits_dtype, a->dx, (int)a->dx_dtype, st));
    else
      MOE_STEP("moe_permute_bwd",
               moe_permute_bwd(dxp, a->row_to_pos, nullptr, T, H, k, a->dx, (int)a->dx_dtype, stream));
  }
  const bool router_dw = router && to_logits && a->dwr;
  if (router_dw && a->dlogits) return MOE_ERR_SHAPE;  // one or the other: the caller's dlogits are not padded
  // weight gradients, down projection first: [dyp | act], [dg | xp], [du | xp]
  MoeWgradStack stacks[3]{}, rstack{};
  int n_stacks = 0;
  for (int w : {2, 0, 1}) {
    if (!a->dw[w]) continue;
    MoeWgradStack& m = stacks[n_stacks++];
    m.a = w == 2 ? dyp : w == 0 ? dg : du;
    m.b = w == 2 ? a->act : in_place ? a->xn : a->xp;
    if (dout_stays && w == 2) m.row_from = a->pos_to_row, m.from_k = k, m.from_rows = T, m.from_a = true;
    if (in_place && w != 2) {
      m.from_k = k, m.from_rows = T;
      if (multi) m.row_at = ws.row_at;
      else m.row_from = a->pos_to_row;
    }
    m.M = w == 2 ? H : I;
    m.N = w == 2 ? I : H;
    m.lda = m.M, m.ldb = m.N;
    m.out = a->dw[w];
    m.part = ws.wpart[w];
    m.dtype = (int)a->dw_dtype[w];
    m.accumulate = a->dw_accumulate[w] ? 1 : 0;
    if (pair && w == 0) {  // the up stack's rows are the ones behind
      m.M = m.lda = 2 * I;
      m.out2 = a->dw[1];
      break;
    }
  }
  if (router_dw) {
    rstack.a = ws.dlogits, rstack.b = a->xn, rstack.out = a->dwr, rstack.part = ws.rpart;
    rstack.M = rstack.lda = rs.Ep, rstack.N = rstack.ldb = H;
    rstack.dtype = (int)a->dwr_dtype;
  }
  if (multi) {
    if (n_stacks || router_dw)
      MOE_STEP("moe_wgrad_multi", moe_wgrad_multi(stacks, n_stacks, router_dw ? &rstack : nullptr, a->offs, E, R, H, I, T,
                                                  rs.slices, rs.rows, st));
  } else {
    bool one_kind = true;
    for (int i = 1; i < n_stacks; ++i) one_kind = one_kind && stacks[i].dtype == stacks[0].dtype;
    if (one_kind && n_stacks > 1) {
      MOE_STEP("moe_gemm_wgrad_all", moe_gemm_wgrad_all(stacks, n_stacks, a->offs, E, R, stream));
    } else {
      for (int i = 0; i < n_stacks; ++i)
        MOE_STEP(stacks[i].out2 ? "moe_gemm_wgrad_pair" : "moe_gemm_wgrad",
                 moe_gemm_wgrad_all(stacks + i, 1, a->offs, E, R, stream));
    }
    if (router_dw)
      MOE_STEP("moe_router_wgrad",
               moe_wgrad_multi(stacks, 0, &rstack, a->offs, E, R, H, I, T, rs.slices, rs.rows, st));
  }
  return 0;
}

extern "C" int moe_layer_backward(const moe_layer_backward_args* a, void* stream) { return layer_backward(a, false, nullptr, stream); }

int moe_in_place_layer_backward(const moe_layer_backward_args* a, void* stream) {
  return layer_backward(a, true, nullptr, stream);
}

int moe_norm_layer_backward(const moe_layer_backward_args* a, const MoeNormBackward& norm, void* stream) {
  return layer_backward(a, a && !a->xp, &norm, stream);
}
