"""Differentiable entry points built on the HIP kernels.

`moe_ffn`      x [T,H] + router logits [T,E] -> out [T,H]: the body of the reference's
               `MoE.forward` after the router linear (model/modules/mlp.py:101-167).
`experts_rows` rows [R,H] + local expert ids [R] -> out [R,H] in arrival order: the part
               between the two all-to-alls (mlp.py:122-161), i.e. one rank's local share.

`router_linear` x [T,H], Wr [E,H] -> logits [T,E]: the router product (mlp.py:100) with the same
               autocast rule as `nn.Linear`; its weight gradient, a 64 x 2048 x 16384 product
               in benchmark config 3 that the BLAS library has no good kernel for, runs as a
               split-k sum on the grouped weight-gradient kernel.

`prenorm_moe`  x [T,H] residual stream -> x + MoE(RMSNorm(x)) and the router logits: the caller's
               two lines around the layer (model/gpt.py:32-33) in one differentiable call.  The
               normalisation writes the bf16 rows the layer consumes in one pass over x, the
               residual add rides in the combine kernel, and in the backward pass the three
               gradient streams into x (expert path, router path, residual) meet inside the
               normalisation's backward kernel instead of in separate additions.

`moe_ffn` and `experts_rows` compute in bf16 on the matrix cores with fp32 accumulation,
whatever the input dtype; outputs and input gradients take the dtype of `x`, weight gradients
the dtype of the weights.  `moe_ffn_f32` is the same function with every step in fp32 (fp32
matrix instructions, fp32 rows): what the reference computes when it is called without autocast
on fp32 tensors.  There is no host synchronisation anywhere in either direction.

Weight gradients into `.grad` (`accumulate_into_grad=True`): the reference's trainer sums
the gradients of several micro-steps in the parameters' `.grad` (training/trainer.py:241-248),
which costs autograd one more read-add-write pass over every expert weight gradient per
micro-step.  With the option on, the weight-gradient kernel adds its result to the existing
`.grad` in its own epilogue (or creates `.grad` on the first micro-step) and autograd
receives no gradient for the three stacks.  The sums are the same numbers (one fp32 add per
element either way); what changes is that autograd hooks on these parameters no longer see
the gradient (tensor hooks are called with None, nothing reaches the accumulation node), so
a data-parallel wrapper that reduces gradients from such hooks must leave the option off.
"""
from __future__ import annotations

import torch

from . import lib as _lib, ops


def _first_order_only():
    """Called at the top of every backward here.  The backward passes run kernels autograd cannot
    see through, so a gradient of a gradient would silently lack their terms: refuse to build a
    graph over them (grad mode is on inside a backward pass only under `create_graph=True`)."""
    if torch.is_grad_enabled():
        raise RuntimeError("the MoE kernels' backward pass is not differentiable: call backward()/grad() "
                           "without create_graph=True")


class _RouterLinear(torch.autograd.Function):
    @staticmethod
    @torch.amp.custom_fwd(device_type="cuda", cast_inputs=torch.bfloat16)
    def forward(ctx, x, w):
        ctx.save_for_backward(x, w)
        return _lib.native().router_logits(x, w)

    @staticmethod
    @torch.amp.custom_bwd(device_type="cuda")
    def backward(ctx, dlogits):
        _first_order_only()
        x, w = ctx.saved_tensors
        dx = dw = None
        if ctx.needs_input_grad[0]:
            dx = dlogits @ w
        if ctx.needs_input_grad[1]:
            dw = _lib.native().router_wgrad(dlogits, x, w.dtype)
        return dx, dw


def router_linear(x: torch.Tensor, weight: torch.Tensor) -> torch.Tensor:
    """Router logits `x @ weight^T` (mlp.py:100) for x [..., H], weight [E, H].  Forward and
    input gradient are the library products `nn.Linear` would run, under the same autocast
    rule (bf16 operands and result inside a bf16 autocast region), but for a bf16 forward of at
    most 64 tokens and 128 experts: that is a kernel here, whose own summation order can move a
    bf16 logit by one unit in the last place.  The weight gradient is computed here (see the
    module docstring)."""
    lead = x.shape[:-1]
    out = _RouterLinear.apply(x.reshape(-1, x.shape[-1]), weight)
    return out.reshape(*lead, weight.shape[0])


def _call(x, k, w1, w3, w2, *, norm_weight=None, router_weight=None, logits=None, ids=None, bias=None,
          bf16_weights=None, eps=0.0, add_residual=False, fused_router=True, accumulate=False, routing=False):
    """The layer through its autograd node: -> (out, router logits or None, routing or None)."""
    out, lg, words = _lib.native().layer(x, norm_weight, router_weight, logits, ids, w1, w3, w2, bias,
                                         *(bf16_weights or (None, None, None)), k, eps, add_residual, fused_router,
                                         accumulate, routing)
    return out, lg, (ops.Routing(words, x.shape[0] * k, w1.shape[0]) if routing else None)


def _routing_dict(r):
    return {"ids": r.ids, "gates": r.gates, "counts": r.counts, "offs": r.offs, "pos_to_row": r.pos_to_row,
            "row_to_pos": r.row_to_pos}


def _rows_dict(r):
    return {"counts": r.counts, "offs": r.offs, "pos_to_row": r.pos_to_row, "row_to_pos": r.row_to_pos,
            "bad_ids": r.bad_ids}


def _check_ids(name, routing, n_ids, E):
    n = int(routing.bad_ids.item())
    if n:
        raise ValueError(f"{name}: {n} of {n_ids} expert ids lie outside [0, {E})")


def moe_ffn(x: torch.Tensor, logits: torch.Tensor, w1: torch.Tensor, w3: torch.Tensor,
            w2: torch.Tensor, k: int, bias: torch.Tensor | None = None, return_routing: bool = False,
            bf16_weights=None, accumulate_into_grad: bool = False):
    """out[t] = sum_j gate[t,j] * FFN_{e(t,j)}(x[t]).  x [T,H]; logits [T,E]; w1,w3 [E,I,H];
    w2 [E,H,I].  `bias` (fp32 [E]) is added to the logits in fp32 and is part of them from
    there on: both the selection and the softmax over the selected values see logit + bias
    (a per-expert constant in the router, as benchmark config 2 specifies); when it requires a
    gradient it receives the column sum of the logits' gradient (fp32, summed before that gradient
    is rounded to the logits' dtype).
    With `return_routing` also returns a dict of the integer routing tensors and gates.
    `bf16_weights`: bf16 copies of (w1, w3, w2) to compute with (None entries are cast here).
    `accumulate_into_grad`: w1, w3, w2 must be leaf tensors; see the module docstring."""
    out, _, routing = _call(x, k, w1, w3, w2, logits=logits, bias=bias, bf16_weights=bf16_weights,
                            accumulate=accumulate_into_grad, routing=return_routing)
    return (out, _routing_dict(routing)) if return_routing else out


def moe_ffn_f32(x: torch.Tensor, logits: torch.Tensor, w1: torch.Tensor, w3: torch.Tensor,
                w2: torch.Tensor, k: int, bias: torch.Tensor | None = None, return_routing: bool = False):
    """`moe_ffn` with every tensor and every product in fp32 (all arguments fp32; H and the FFN
    width multiples of 4).  Routing, counts and the permutation are the same kernels and the same
    bits as in `moe_ffn` given the same logits."""
    for name, t in (("x", x), ("logits", logits), ("w1", w1), ("w3", w3), ("w2", w2)):
        if t.dtype != torch.float32:
            raise TypeError(f"moe_ffn_f32: {name} must be fp32, got {t.dtype}")
    out, _, words = _lib.native().layer_f32(x, None, logits, None, w1, w3, w2, bias, k, return_routing)
    return (out, _routing_dict(ops.Routing(words, x.shape[0] * k, w1.shape[0]))) if return_routing else out


def routed_moe_f32(x: torch.Tensor, router_weight: torch.Tensor, w1: torch.Tensor, w3: torch.Tensor, w2: torch.Tensor, k: int):
    """(MoE(x), router logits) for x [..., H], all fp32: `nn.Linear`'s product and `moe_ffn_f32`, the router path's gradients
    worked out along with the experts'.  The logits are between the two as if they were called one after the other: where a hook
    is on them, their gradient is retained or asked for, it is handed to the product's own backward instead."""
    out, logits, _ = _lib.native().layer_f32(x, router_weight, None, None, w1, w3, w2, None, k, False)
    return out.reshape(x.shape), logits


def prenorm_moe(x: torch.Tensor, norm_weight: torch.Tensor, router_weight: torch.Tensor,
                w1: torch.Tensor, w3: torch.Tensor, w2: torch.Tensor, k: int, eps: float = 1e-6,
                add_residual: bool = True, bf16_weights=None, accumulate_into_grad: bool = False,
                return_routing: bool = False, fused_router: bool = True):
    """(x + MoE(RMSNorm(x)), router logits) for x [T,H]: model/gpt.py:32-33 with
    model/modules/norm.py:14-19 and model/modules/mlp.py:95-169 in one differentiable call.
    Router logits are bf16 (what the reference produces under its bf16 autocast); the output
    has the dtype of x.  H <= 8192.  `fused_router=False` takes the logits from the product that
    `routed_moe` and `MoE.forward` run on the same rows (the same bits they select on) instead of the
    fused norm+router kernel, whose own summation order can move a bf16 logit by one unit in the
    last place."""
    out, logits, routing = _call(x, k, w1, w3, w2, norm_weight=norm_weight, router_weight=router_weight,
                                 bf16_weights=bf16_weights, eps=float(eps), add_residual=add_residual,
                                 fused_router=fused_router, accumulate=accumulate_into_grad, routing=return_routing)
    return (out, logits, _routing_dict(routing)) if return_routing else (out, logits)


def routed_moe(x: torch.Tensor, router_weight: torch.Tensor, w1: torch.Tensor, w3: torch.Tensor,
               w2: torch.Tensor, k: int, bias: torch.Tensor | None = None, bf16_weights=None,
               accumulate_into_grad: bool = False, return_routing: bool = False):
    """(MoE(x), router logits) for x [T,H]: `router_linear` and `moe_ffn` as one autograd node
    (mlp.py:100-167), so that the two gradient contributions to x (expert path, router path)
    are summed inside the k-row-sum kernel.  The router product is a bf16 product whatever the
    dtypes (the reference's behaviour under its bf16 autocast), the one of `router_linear`; the
    output has the dtype of x.  With nothing to differentiate, at most 64 tokens run on kernels
    whose sums are formed in another order, so their output can differ from the differentiable
    call's, and from that of the same tokens in a larger batch, in its last bits.  With `return_routing` a dict of the integer routing tensors and gates is
    returned as a third value."""
    out, logits, routing = _call(x, k, w1, w3, w2, router_weight=router_weight, bias=bias, bf16_weights=bf16_weights,
                                 accumulate=accumulate_into_grad, routing=return_routing)
    return (out, logits, _routing_dict(routing)) if return_routing else (out, logits)


def experts_rows_f32(rows: torch.Tensor, ids: torch.Tensor, w1, w3, w2, return_routing: bool = False,
                     check_ids: bool = False):
    """`experts_rows` with every tensor and every product in fp32 (rows and weights fp32)."""
    for name, t in (("rows", rows), ("w1", w1), ("w3", w3), ("w2", w2)):
        if t.dtype != torch.float32:
            raise TypeError(f"experts_rows_f32: {name} must be fp32, got {t.dtype}")
    want = check_ids or return_routing
    out, _, words = _lib.native().layer_f32(rows, None, None, ids, w1, w3, w2, None, 1, want)
    routing = ops.Routing(words, rows.shape[0], w1.shape[0]) if want else None
    if check_ids:
        _check_ids("experts_rows_f32", routing, ids.numel(), w1.shape[0])
    return (out, _rows_dict(routing)) if return_routing else out


def experts_rows(rows: torch.Tensor, ids: torch.Tensor, w1, w3, w2, return_routing: bool = False,
                 accumulate_into_grad: bool = False, check_ids: bool = False):
    """One rank's local expert share: rows [R,H] already dispatched to this rank, ids [R]
    local expert index of each row -> FFN output rows in the same (arrival) order.

    ids must lie in [0, E).  The dispatch kernels count the ids that do not (and treat such a
    row as belonging to the nearest valid expert, so nothing reads out of bounds); the count is
    a device tensor, `bad_ids` in the routing dict, so the hot path never waits for it.  With
    `check_ids` the call synchronises and raises ValueError if the count is not zero."""
    out, _, routing = _call(rows, 1, w1, w3, w2, ids=ids, accumulate=accumulate_into_grad,
                            routing=check_ids or return_routing)
    if check_ids:
        _check_ids("experts_rows", routing, ids.numel(), w1.shape[0])
    return (out, _rows_dict(routing)) if return_routing else out
