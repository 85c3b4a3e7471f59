// What the router's product is made of, and the layer calls that it is part of (declared for host code too, which internal.h is not).
#pragma once
#include <stdint.h>

#include "moe_gfx950.h"

struct MoeRouter {
  const void *x, *wr;  // [T,H] and [E,H], each bf16 or fp32
  int x_dtype, wr_dtype;
  const float* bias;   // [E] or NULL: added to the logits for the selection
  uint16_t *xn, *wrb;  // where bf16 copies of an fp32 x and wr are left (NULL: they are not wanted)
  uint16_t* logits;    // [T,E]
};

// Sizes for which product and selection are one launch (router.hip).
bool moe_router_select_ok(int64_t T, int64_t H, int64_t E, int64_t k, int wr_dtype);
// moe_ffn_forward, and moe_layer_forward (x: the bf16 rows), with the router's product part of it: sizes that moe_router_few_ok (x and
// wr in bf16) or moe_router_select_ok takes, the latter alone in training.  moe_selected_layer_forward: with a `table` instead the
// selection is done, ids and gates are there, and so are its counts; with neither it is moe_layer_forward.
// moe_forward_only without a router is moe_ffn_forward, in a workspace without room for copies that are not made.
int64_t moe_forward_only_scratch(int64_t T, int64_t H, int64_t E, int64_t I, int64_t k, int x_dtype);
int moe_forward_only(const MoeRouter* router, const void* x, int x_dtype, const void* logits, int logits_dtype, const float* bias,
                     const uint16_t* w1, const uint16_t* w3, const uint16_t* w2, int64_t T, int64_t H, int64_t E, int64_t I, int64_t k,
                     void* out, int out_dtype, void* workspace, int64_t workspace_bytes, void* stream);
// Without xp the experts read x where it is (then in bf16), for sizes that moe_layer_rows_from_ok takes; the backward pass is then
// moe_in_place_layer_backward, which has x as xn.
bool moe_layer_rows_from_ok(int64_t T, int64_t H, int64_t E, int64_t I, int64_t k);
int moe_in_place_layer_backward(const moe_layer_backward_args* a, void* stream);
// moe_layer_backward, or moe_in_place_layer_backward where there is no xp, with the backward pass of the norm in front of the layer: dx is the
// gradient of the norm's input, of its type.  For a router whose gradients are worked out in the call, and sizes that moe_norm_rows_ok takes.
struct MoeNormBackward {
  const void* x;        // the norm's input [T,H]
  int x_dtype;
  const float *weight, *rstd;
  const void* dres;     // gradient of a residual branch, of x's type (NULL: there is none)
  float* dweight;       // [H]
  void* workspace;      // of moe_rmsnorm_bwd_workspace_bytes
  int64_t workspace_bytes;
};
bool moe_norm_rows_ok(int64_t T, int64_t H);
int moe_norm_layer_backward(const moe_layer_backward_args* a, const MoeNormBackward& norm, void* stream);
int moe_selected_layer_forward(const moe_layer_forward_args* a, const MoeRouter* router, const void* table, void* stream);
