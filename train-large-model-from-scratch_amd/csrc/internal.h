// Launchers the library's own files share (the C ABI is in include/moe_gfx950.h).  Arguments are
// checked by the entry points that reach them.
#pragma once
#include "common.h"
#include "router.h"

// Tells the installed launch observer, if any, about one launch (layer.hip).
void moe_observe(const char* name, int after);

// Compute units of the current GPU (asked of the runtime once).
int moe_compute_units();

// Tiles of bm rows that R rows of E experts come to where a router deals them: half a tile an expert more than R / bm, and one
// each where its rows do not fill one.
inline double moe_expected_tiles(int64_t R, int64_t E, int bm) {
  const double x = (double)R / E / bm;
  return E * (x <= 0.6 ? 1 : x >= 1 ? x + 0.5 : 1 + (x - 0.6) * 1.25);
}

// Gate gradients from the dgrad-down kernel's block sums, softmax Jacobian and scatter to the logits in
// one kernel (route.hip).  dlogits [T, ld] with columns E..ld-1 zero.
int moe_router_bwd_from_blocks(const float* part, int64_t P, const float* gates, const int32_t* ids,
                               const int32_t* row_to_pos, int64_t T, int64_t E, int64_t k, int64_t ld,
                               void* dlogits, int dlogits_dtype, hipStream_t s);

// moe_permute_bwd with the router path's input gradient and what moe_router_bwd_from_blocks does in the same pass: dx[t] =
// sum_j dxp[pos(t,j)] + bf16(sum_j dsel[t,j] * wr[ids[t,j]]), dsel the k nonzero entries of a row of dlogits (dispatch.hip).
int moe_permute_bwd_router(const uint16_t* dxp, const int32_t* row_to_pos, const float* part, int64_t P, const float* gates,
                           const int32_t* ids, const uint16_t* wr, int64_t T, int64_t H, int64_t k, int64_t ld, void* dlogits,
                           int dlogits_dtype, void* dx, int dx_dtype, hipStream_t s);

// moe_permute_bwd_router and moe_rmsnorm_bwd in one pass, without what one hands on to the other (norm.hip).
int moe_rmsnorm_bwd_rows(const MoeNormBackward& n, const uint16_t* dxp, const int32_t* row_to_pos, const float* part, int64_t P,
                         const float* gates, const int32_t* ids, const uint16_t* wr, int64_t T, int64_t H, int64_t k, int64_t ld,
                         uint16_t* dlogits, void* dx, hipStream_t s);

// moe_combine_bwd_by_token without y, which also leaves where a position's token is, in bytes of rows of H elements of bf16 (dispatch.hip).
int moe_combine_bwd_places(const void* dy, int dy_dtype, const float* gates, const int32_t* row_to_pos, int64_t T, int64_t H, int64_t k,
                           uint16_t* dyp, uint32_t* row_at, hipStream_t s);

// Bytes of scratch that a call with these arguments (all but the scratch filled in) uses: rows that stay in place need no
// buffer for them (layer.hip), and it is no more than moe_layer_scratch_bytes says but for the list of where they are, without xp.
int64_t moe_forward_scratch(const moe_layer_forward_args* a);
int64_t moe_backward_scratch(const moe_layer_backward_args* a);

// fp32 to bf16, two tensors of multiples of 8 elements in one launch (dispatch.hip).
int moe_cast_two(const float* a, uint16_t* to_a, int64_t na, const float* b, uint16_t* to_b, int64_t nb, void* stream);

// int64 expert ids to int32, values outside int32 to -1 (dispatch.hip).
int moe_narrow_ids(const int64_t* ids, int64_t R, int32_t* out, hipStream_t s);

// ---- weight gradients of small launches (wgrad.hip) ----
// out [E,M,N] (+)= a^T b per expert, a [R,M] and b [R,N] with row strides lda and ldb; part: room for partial sums.
struct MoeWgradStack {
  const uint16_t *a, *b;
  void* out;
  float* part;
  int64_t lda, ldb, M, N;
  int dtype, accumulate;
  void* out2;  // moe_gemm_wgrad_all: an expert's rows M / 2 .. M - 1 go here (NULL: all to out)
  // moe_gemm_wgrad_all: row r of b, or with from_a of a, is row row_from[r] / from_k of its from_rows (NULL: row r)
  const int32_t* row_from;
  int64_t from_k, from_rows;
  // moe_wgrad_multi: row r of b, of from_rows rows, is row_at[r] bytes from its beginning (NULL: row r).
  const uint32_t* row_at;
  bool from_a;
};
// Weight gradients leave with streaming stores from so many bytes of results in a launch on, an eighth of the memory-side cache: a
// model of a few such layers finds smaller ones there when it adds them up, clips them or steps.  Pass, pass with its gradients added
// to another's, and pass with their norms taken, us, ordinary stores -> streaming: 1.5 MB 49 -> 49, 99 -> 100, 66 -> 70; 25 MB 128 -> 128, 256 ->
// 257, 138 -> 143, and 298 -> 296, 608 -> 605, 311 -> 319; 48 MB 157 -> 154, 326 -> 325, 181 -> 192; 96 MB 204 -> 191, 465 -> 452, 234 -> 249;
// 144 MB 183 -> 166, 461 -> 432, 268 -> 255; 192 MB 361 -> 331, 821 -> 767, 423 -> 403; 240 MB 405 -> 369, 943 -> 869, 495 -> 474.
constexpr int64_t MOE_STREAMED_RESULTS = 32 << 20;
// moe_gemm_wgrad, and moe_gemm_wgrad_pair where there is an out2, of up to three stacks with results of one kind in one launch.
int moe_gemm_wgrad_all(const MoeWgradStack* stacks, int n, const int32_t* offs, int64_t E, int64_t R, void* stream);
// Bytes of each stack's part for R rows.
int64_t moe_wgrad_multi_part_bytes(int64_t R, int64_t H, int64_t I);
// The stacks (the first n_stacks, all of the size I x H or H x I; without any, offs may be NULL) and, unless NULL, the router: a [T, M >= E] and b
// [T,N] contracted in router_slices slices of router_rows rows (part [slices][M][N]), out [E,N].
int moe_wgrad_multi(const MoeWgradStack (&stacks)[3], int n_stacks, const MoeWgradStack* router, const int32_t* offs,
                    int64_t E, int64_t R, int64_t H, int64_t I, int64_t T, int64_t router_slices,
                    int64_t router_rows, hipStream_t s);

// ---- selection, places and rows in two launches (place.hip) ----
// Sizes it takes, and the bytes of its table of counts: (E + 3) / 4 words for every so many tokens, a byte an expert.
constexpr int MOE_PLACE_CHUNK = 16;
bool moe_place_ok(int64_t T, int64_t E, int64_t k);
int64_t moe_place_bytes(int64_t T, int64_t E);
// moe_router_topk_fwd that leaves the table, and from it the results of moe_histogram_scan and moe_permute_fwd (fp32 rows
// where x is fp32 and xp_dtype says so; xp NULL: no rows); *bad_ids, unless NULL, becomes 0.
int moe_select_count(const void* logits, int logits_dtype, const float* bias, int64_t T, int64_t E, int64_t k,
                     int32_t* ids, float* gates, void* table, void* stream);
int moe_place_rows(const void* x, int x_dtype, const int32_t* ids, const void* table, int64_t T, int64_t H, int64_t E,
                   int64_t k, int32_t* counts, int32_t* offs, int32_t* pos_to_row, int32_t* row_to_pos, int32_t* bad_ids,
                   void* xp, int xp_dtype, bool counted, void* stream);
// Both in one launch, for few logits.
bool moe_select_place_ok(const void* logits, int64_t T, int64_t E, int64_t k);
int moe_select_place(const void* x, int x_dtype, const void* logits, int logits_dtype, const float* bias, int64_t T, int64_t H,
                     int64_t E, int64_t k, int32_t* ids, float* gates, int32_t* counts, int32_t* offs, int32_t* pos_to_row,
                     int32_t* row_to_pos, int32_t* bad_ids, void* xp, int xp_dtype, void* stream);
// The table where the experts are given, one a row (`counted` above), and how many of them are outside [0, E) behind it:
// sizes it takes, bytes of both, and the launch.  ids64, unless NULL, are left in `ids` in 32 bits, else `ids` are given.
bool moe_count_ok(int64_t T, int64_t E, int64_t k);
int64_t moe_count_bytes(int64_t T, int64_t E);
int moe_count_ids(const int64_t* ids64, int32_t* ids, int64_t T, int64_t E, void* table, void* stream);

// The router's product, the selection and its table of counts (NULL: not wanted) in one launch (router.hip).
int moe_router_select(const MoeRouter& r, int64_t T, int64_t H, int64_t E, int64_t k, int32_t* ids, float* gates, void* table,
                      hipStream_t s);

// moe_rmsnorm_router_fwd that leaves the table too, unless it is NULL (norm.hip).
int moe_rmsnorm_router_count(const void* x, int x_dtype, const float* weight, float eps, const uint16_t* router_weight,
                             int64_t T, int64_t H, int64_t E, int64_t k, uint16_t* xn, float* rstd, uint16_t* logits,
                             int32_t* ids, float* gates, void* table, void* stream);

// ---- grouped products (gemm.hip) ----
// moe_gemm_down_fwd and moe_gemm_dgrad_gateup (ld_in: 0, or the row stride of dg and du) whose result's row of position p is row
// row_map[p] (a permutation of the R rows; NULL: row p).
int moe_gemm_down_to(const uint16_t* act, const uint16_t* w2, const int32_t* offs, int64_t E, int64_t R, int64_t H, int64_t I,
                     uint16_t* y, const int32_t* row_map, void* stream);
int moe_gemm_dgrad_gateup_to(const uint16_t* dg, const uint16_t* du, int64_t ld_in, const uint16_t* w1, const uint16_t* w3,
                             const int32_t* offs, int64_t E, int64_t R, int64_t H, int64_t I, uint16_t* dxp,
                             const int32_t* row_map, void* stream);
// moe_gemm_gateup_swiglu_fwd_blocked (gu_blocked NULL: moe_gemm_gateup_swiglu_fwd without g and u) whose row p of xp is x[pos_to_row[p] / k], for x [T,H] of sizes that it takes.
bool moe_rows_from_ok(int64_t T, int64_t H);
int moe_gemm_gateup_from(const uint16_t* x, const int32_t* pos_to_row, int64_t T, int64_t k, const uint16_t* w1, const uint16_t* w3,
                         const int32_t* offs, int64_t E, int64_t H, int64_t I, void* gu_blocked, uint16_t* act, void* stream);
// moe_gemm_dgrad_down_swiglu_bwd_blocked whose row p of dyp is dy[pos_to_row[p] / k], for dy [T,H] of sizes that moe_rows_from_ok takes.
int moe_gemm_dgrad_down_from(const uint16_t* dy, const int32_t* pos_to_row, int64_t T, int64_t k, const uint16_t* w2,
                             const void* gu_blocked, const int32_t* offs, int64_t E, int64_t H, int64_t I, uint16_t* dg, uint16_t* du,
                             int64_t ld_out, float* dgate_part, void* stream);
// ---- few tokens (few.hip) ----
constexpr int FEW_MAX_TOKENS = 64;
constexpr int FEW_MAX_EXPERTS = 128;

// Router product rounded to bf16: shapes it takes, and the launch.
bool moe_router_few_ok(int64_t T, int64_t H, int64_t E, int64_t k);
int moe_router_few(const uint16_t* x, const uint16_t* wr, int64_t T, int64_t H, int64_t E, uint16_t* logits,
                   hipStream_t s);
// The experts on at most 64 tokens, rows in routed order: act [T*k, I] from x and the expert ids, y [T*k, H]
// from act, and for one token the combined output from act.
bool moe_few_ok(int64_t T, int64_t H, int64_t E, int64_t I, int64_t k, int x_dtype);
int moe_gateup_few(const void* x, int x_dtype, const int32_t* ids, const uint16_t* w1, const uint16_t* w3, int64_t T,
                   int64_t H, int64_t E, int64_t I, int64_t k, uint16_t* act, hipStream_t s);
// The same from the logits, the selection with it: ids and gates [T*k] are results.
bool moe_gateup_few_selects(int64_t T, int64_t E, int64_t I, int64_t k);
int moe_gateup_few_select(const void* x, int x_dtype, const void* logits, int logits_dtype, const float* bias, const uint16_t* w1,
                          const uint16_t* w3, int64_t T, int64_t H, int64_t E, int64_t I, int64_t k, int32_t* ids, float* gates,
                          uint16_t* act, hipStream_t s);
// The same for one token, its selection with it: ids and gates [k] are results.
bool moe_gateup_one_ok(int64_t T, int64_t E, int64_t k);
int moe_gateup_one(const void* x, int x_dtype, const void* logits, int logits_dtype, const float* bias, const uint16_t* w1,
                   const uint16_t* w3, int64_t H, int64_t E, int64_t I, int64_t k, int32_t* ids, float* gates,
                   uint16_t* act, hipStream_t s);
int moe_down_few(const uint16_t* act, const int32_t* ids, const uint16_t* w2, int64_t T, int64_t H, int64_t E, int64_t I,
                 int64_t k, uint16_t* y, hipStream_t s);
bool moe_down_one_ok(int64_t T, int64_t k);
int moe_down_one(const uint16_t* act, const int32_t* ids, const float* gates, const uint16_t* w2, int64_t H, int64_t E,
                 int64_t I, int64_t k, void* out, int out_dtype, hipStream_t s);
// moe_combine_fwd with the rows of y in routed order (dispatch.hip).
int moe_combine_in_order(const uint16_t* y, const float* gates, int64_t T, int64_t H, int64_t k, void* out,
                         int out_dtype, hipStream_t s);
