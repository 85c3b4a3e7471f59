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

from . import ops
from .ops import dense as _dense


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
        return torch.nn.functional.linear(x, w)

    @staticmethod
    @torch.amp.custom_bwd(device_type="cuda")
    def backward(ctx, dlogits):
        _first_order_only()
        x, w = ctx.saved_tensors
        dx = dw = None
        if ctx.needs_input_grad[0]:
            dx = dlogits @ w
        if ctx.needs_input_grad[1]:
            dw = _router_wgrad(dlogits, x, w.dtype)
        return dx, dw


def _router_wgrad(dlogits, x, w_dtype):
    """dWr = dlogits^T x for dlogits [T,E], x [T,H]."""
    T, H = x.shape
    E = dlogits.shape[1]
    fast = (x.is_cuda and x.dtype == torch.bfloat16 and dlogits.dtype == torch.bfloat16
            and E % 8 == 0 and H % 8 == 0 and T > 0)
    if not fast:
        return (dlogits.t() @ x).to(w_dtype)
    if w_dtype not in (torch.bfloat16, torch.float32):
        return ops.router_wgrad(_dense(dlogits), _dense(x), torch.float32).to(w_dtype)
    return ops.router_wgrad(_dense(dlogits), _dense(x), w_dtype)


def router_linear(x: torch.Tensor, weight: torch.Tensor) -> torch.Tensor:
    """Router logits `x @ weight^T` (mlp.py:100) for x [..., H], weight [E, H].  Forward and
    input gradient are the library products `nn.Linear` would run, under the same autocast
    rule (bf16 operands and result inside a bf16 autocast region); the weight gradient is
    computed here (see the module docstring)."""
    lead = x.shape[:-1]
    out = _RouterLinear.apply(x.reshape(-1, x.shape[-1]), weight)
    return out.reshape(*lead, weight.shape[0])


def _weight_gradients(needed, params, weights, wdtype):
    """Where the gradients of the three stacks go, given which are `needed`, the parameters whose `.grad`
    the kernel may write (or None each) and the stacks themselves: -> (tensors or None, whether each is
    added to, what autograd receives, [(parameter, its new .grad)])."""
    out, acc, ret, fresh = [], [], [], []
    for need, param, w in zip(needed, params or (None, None, None), weights):
        into, add, give = None, False, None
        if need:
            held = None if param is None else param.grad
            if param is not None and held is None:
                into = torch.empty(w.shape, dtype=param.dtype, device=w.device)
                fresh.append((param, into))
            elif (param is not None and held.dtype in (torch.float32, torch.bfloat16) and held.is_contiguous()
                  and held.shape == w.shape and held.device == w.device):
                into, add = held, True
            else:  # autograd takes the gradient (and sums it with a .grad the kernel cannot add to)
                into = give = torch.empty(w.shape, dtype=wdtype, device=w.device)
        out.append(into)
        acc.append(add)
        ret.append(give)
    return out, acc, ret, fresh


def _expert_gradients(ctx, dout, needed, routing, xp, gu, act, w1b, w3b, w2b, k, **results):
    """The layer body's backward call with the weight gradients put where they belong; -> what autograd
    receives for the three stacks."""
    dw, acc, ret, fresh = _weight_gradients(needed, ctx.grad_params, (w1b, w3b, w2b), ctx.w_dtype)
    ids, gates, _, offs, pos_to_row, row_to_pos, _ = routing
    ops.layer_backward(dout, dout.shape[0], k, gates, ids, offs, pos_to_row, row_to_pos, xp, gu, act, w1b, w3b, w2b,
                       dw, acc, **results)
    for param, grad in fresh:
        param.grad = grad
    return ret


def _routing_dict(r):
    return {"ids": r.ids, "gates": r.gates, "counts": r.counts, "offs": r.offs, "pos_to_row": r.pos_to_row,
            "row_to_pos": r.row_to_pos}


class _MoEFFN(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, logits, w1, w3, w2, k, bias, shadows, grad_params, routing_out):
        T, H = x.shape
        E, I = logits.shape[1], w1.shape[1]
        x = _dense(x)
        logits = _dense(logits)
        w1b, w3b, w2b = _weights_bf16(w1, w3, w2, shadows)
        routing = ops.new_routing(T, H, E, I, k, x.device)
        train = any(ctx.needs_input_grad)
        out, xp, gu, act = ops.layer_forward(x, w1b, w3b, w2b, k, routing, x.dtype, logits=logits, bias=bias,
                                             train=train)
        if train:  # (y is not kept: the gate gradients come out of the dgrad-down kernel)
            ctx.save_for_backward(xp, gu, act, routing.buf, w1b, w3b, w2b)
        ctx.k, ctx.E = k, E
        ctx.grad_params = grad_params
        ctx.x_dtype, ctx.logits_dtype, ctx.w_dtype = x.dtype, logits.dtype, w1.dtype
        ctx.set_materialize_grads(False)
        ctx.out_shape = out.shape
        if routing_out is not None:
            routing_out.append(routing)
        return out

    @staticmethod
    def backward(ctx, dout):
        _first_order_only()
        xp, gu, act, buf, w1b, w3b, w2b = ctx.saved_tensors
        k, E = ctx.k, ctx.E
        dev = xp.device
        if dout is None:
            dout = torch.zeros(ctx.out_shape, dtype=ctx.x_dtype, device=dev)
        T, H = dout.shape
        dout = _dense(dout)
        if dout.dtype not in (torch.bfloat16, torch.float32):
            dout = dout.float()
        need = ctx.needs_input_grad
        routing = ops.new_routing(T, H, E, w1b.shape[1], k, dev, buf)
        dx = torch.empty((T, H), dtype=ctx.x_dtype, device=dev) if need[0] else None
        dlogits = dgates = dbias = None
        if need[6]:
            dgates = torch.empty(T * k, dtype=torch.float32, device=dev)
        elif need[1]:
            dlogits = torch.empty((T, E), dtype=ctx.logits_dtype, device=dev)
        dw1, dw3, dw2 = _expert_gradients(ctx, dout, need[2:5], routing.pointers(), xp, gu, act, w1b, w3b, w2b, k,
                                          dlogits=dlogits, dgates=dgates, dx=dx)
        if need[6]:  # column sum of the logits' gradient, before any rounding
            dl32 = ops.router_topk_bwd(routing.gates, dgates, routing.ids, T, E, k, torch.float32)
            dbias = dl32.sum(0)
            dlogits = dl32.to(ctx.logits_dtype) if need[1] else None
        return dx, dlogits, dw1, dw3, dw2, None, dbias, None, None, None


def _forward_only(*tensors) -> bool:
    """Whether a call needs nothing kept for a backward pass: then nothing is (`ops.ffn_forward`)."""
    return not (torch.is_grad_enabled() and any(t is not None and t.requires_grad for t in tensors))


def _weights_bf16(w1, w3, w2, shadows):
    shadows = shadows or (None, None, None)
    return [sh if sh is not None else ops.cast_bf16(_dense(w)) for w, sh in zip((w1, w3, w2), shadows)]


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
    if not return_routing and x.shape[0] > 0 and _forward_only(x, logits, w1, w3, w2, bias):
        w1b, w3b, w2b = _weights_bf16(w1, w3, w2, bf16_weights)
        return ops.ffn_forward(_dense(x), _dense(logits), w1b, w3b, w2b, k, bias)
    grad_params = None
    if accumulate_into_grad:
        grad_params = tuple(w if (w.requires_grad and w.is_leaf) else None for w in (w1, w3, w2))
    routing = [] if return_routing else None
    out = _MoEFFN.apply(x, logits, w1, w3, w2, k, bias, bf16_weights, grad_params, routing)
    return (out, _routing_dict(routing[0])) if return_routing else out


class _MoEFFNf32(torch.autograd.Function):
    """The fp32 path: model/modules/mlp.py:101-167 with fp32 operands and no autocast."""

    @staticmethod
    def forward(ctx, x, logits, w1, w3, w2, k, bias):
        T, H = x.shape
        E = logits.shape[1]
        x, logits = _dense(x), _dense(logits)
        w1, w3, w2 = _dense(w1), _dense(w3), _dense(w2)
        ids, gates = ops.router_topk(logits, k, bias)
        counts, offs, pos_to_row, row_to_pos = ops.histogram_scan(ids, E)
        xp = ops.f32_gather_rows(x, pos_to_row, k)
        g = ops.f32_gemm_rows(xp, w1, offs, True)
        u = ops.f32_gemm_rows(xp, w3, offs, True)
        act = ops.f32_swiglu(g, u)
        y = ops.f32_gemm_rows(act, w2, offs, True)
        out = ops.f32_combine_fwd(y, gates, row_to_pos, T, k)
        if any(ctx.needs_input_grad):
            ctx.save_for_backward(xp, g, u, act, y, gates, ids, offs, pos_to_row, row_to_pos, w1, w3, w2)
        ctx.k, ctx.E = k, E
        ctx.mark_non_differentiable(ids, gates, counts, offs, pos_to_row, row_to_pos)
        ctx.set_materialize_grads(False)
        ctx.out_shape = out.shape
        return out, ids, gates, counts, offs, pos_to_row, row_to_pos

    @staticmethod
    def backward(ctx, dout, *unused):
        _first_order_only()
        xp, g, u, act, y, gates, ids, offs, pos_to_row, row_to_pos, w1, w3, w2 = ctx.saved_tensors
        k, E = ctx.k, ctx.E
        if dout is None:
            dout = torch.zeros(ctx.out_shape, dtype=torch.float32, device=xp.device)
        T = dout.shape[0]
        need = ctx.needs_input_grad
        dyp, dgates = ops.f32_combine_bwd(_dense(dout.float()), y if (need[1] or need[6]) else None, gates,
                                          pos_to_row, k)
        dact = ops.f32_gemm_rows(dyp, w2, offs, False)
        dg, du = ops.f32_swiglu_bwd(dact, g, u)
        dx = None
        if need[0]:
            dxp = ops.f32_gemm_rows(dg, w1, offs, False)
            ops.f32_gemm_rows(du, w3, offs, False, out=dxp)
            dx = ops.f32_permute_bwd(dxp, row_to_pos, T, k)
        dw1 = ops.f32_gemm_wgrad(dg, xp, offs, E) if need[2] else None
        dw3 = ops.f32_gemm_wgrad(du, xp, offs, E) if need[3] else None
        dw2 = ops.f32_gemm_wgrad(dyp, act, offs, E) if need[4] else None
        dlogits = dbias = None
        if need[1] or need[6]:
            dlogits = ops.router_topk_bwd(gates, dgates, ids, T, E, k, torch.float32)
            dbias = dlogits.sum(0) if need[6] else None
            if not need[1]:
                dlogits = None
        return dx, dlogits, dw1, dw3, dw2, None, dbias


def moe_ffn_f32(x: torch.Tensor, logits: torch.Tensor, w1: torch.Tensor, w3: torch.Tensor,
                w2: torch.Tensor, k: int, bias: torch.Tensor | None = None, return_routing: bool = False):
    """`moe_ffn` with every tensor and every product in fp32 (all arguments fp32; H and the FFN
    width multiples of 4).  Routing, counts and the permutation are the same kernels and the same
    bits as in `moe_ffn` given the same logits."""
    for name, t in (("x", x), ("logits", logits), ("w1", w1), ("w3", w3), ("w2", w2)):
        if t.dtype != torch.float32:
            raise TypeError(f"moe_ffn_f32: {name} must be fp32, got {t.dtype}")
    out, ids, gates, counts, offs, pos_to_row, row_to_pos = _MoEFFNf32.apply(x, logits, w1, w3, w2, k, bias)
    if return_routing:
        return out, {"ids": ids, "gates": gates, "counts": counts, "offs": offs,
                     "pos_to_row": pos_to_row, "row_to_pos": row_to_pos}
    return out


class _PreNormMoE(torch.autograd.Function):
    """Router product, routing, experts and combine as one node, optionally with the caller's
    RMSNorm in front (norm_w) and residual add behind.  Without the norm, xn is x itself
    (rounded to bf16 once if it is fp32)."""

    @staticmethod
    def forward(ctx, x, norm_w, wr, w1, w3, w2, eps, k, bias, shadows, grad_params, add_residual,
                fused_router, routing_out):
        T, H = x.shape
        E, I = wr.shape[0], w1.shape[1]
        x = _dense(x)
        w1b, w3b, w2b = _weights_bf16(w1, w3, w2, shadows)
        wrb = _dense(wr.detach().to(torch.bfloat16))
        routing = ops.new_routing(T, H, E, I, k, x.device)
        nw = rstd = None
        if norm_w is not None:
            nw = norm_w.detach().float().contiguous()
        if (fused_router and norm_w is not None and bias is None and T > 0
                and ops.rmsnorm_router_supported(H, E, k)):
            # norm, router product and selection in one kernel: the normalised rows are not read
            # a second time for the router, the logits are selected on before they leave the chip
            xn, rstd, logits, _, _ = ops.rmsnorm_router_fwd(x, nw, eps, wrb, k, routing)
            selected = True
        else:
            if norm_w is not None:
                xn, rstd = ops.rmsnorm_fwd(x, nw, eps)
            else:
                xn = ops.cast_bf16(x)
            with torch.autocast("cuda", enabled=False):
                logits = xn @ wrb.t()
            selected = False
        train = any(ctx.needs_input_grad)
        out, xp, gu, act = ops.layer_forward(xn, w1b, w3b, w2b, k, routing, x.dtype,
                                             logits=None if selected else logits, bias=bias,
                                             residual=x if add_residual else None, train=train)
        ctx.has_norm = norm_w is not None
        if train:
            ctx.save_for_backward(x if ctx.has_norm else None, nw, rstd, xn, wrb, xp, gu, act, routing.buf,
                                  w1b, w3b, w2b)
        ctx.k, ctx.E, ctx.add_residual = k, E, add_residual
        ctx.grad_params = grad_params
        ctx.x_dtype, ctx.x_shape = x.dtype, x.shape
        ctx.nw_dtype = norm_w.dtype if ctx.has_norm else None
        ctx.wr_dtype, ctx.w_dtype = wr.dtype, w1.dtype
        ctx.set_materialize_grads(False)
        if routing_out is not None:
            routing_out.append(routing)
        return out, logits

    @staticmethod
    def backward(ctx, dout, dlogits_ext):
        _first_order_only()
        x, nw, rstd, xn, wrb, xp, gu, act, buf, w1b, w3b, w2b = ctx.saved_tensors
        k, E = ctx.k, ctx.E
        T, H = ctx.x_shape
        dev = xn.device
        if dout is None:
            dout = torch.zeros(ctx.x_shape, dtype=ctx.x_dtype, device=dev)
        dout = _dense(dout)
        if dout.dtype != ctx.x_dtype:
            dout = dout.to(ctx.x_dtype)
        need = ctx.needs_input_grad
        routing = ops.new_routing(T, H, E, w1b.shape[1], k, dev, buf)
        want_dx = need[0] or (ctx.has_norm and need[1])
        dx = torch.empty((T, H), dtype=ctx.x_dtype, device=dev) if want_dx else None
        dwr = torch.empty((E, H), dtype=ctx.wr_dtype, device=dev) if need[2] else None
        dbias = dnw = d2 = None
        if not need[8] and dlogits_ext is None:
            # the gradients of the rows' two paths (experts, router) meet inside the k-row sum
            dw1, dw3, dw2 = _expert_gradients(ctx, dout, need[3:6], routing.pointers(), xp, gu, act, w1b, w3b, w2b, k,
                                              wr=wrb, xn=xn, dwr=dwr, dx=dx)
        else:
            # the logits' gradient is wanted by itself (for the bias), or has a share from outside
            dgates = torch.empty(T * k, dtype=torch.float32, device=dev)
            dxp = torch.empty((T * k, H), dtype=torch.bfloat16, device=dev) if want_dx else None
            dw1, dw3, dw2 = _expert_gradients(ctx, dout, need[3:6], routing.pointers(), xp, gu, act, w1b, w3b, w2b, k,
                                              dgates=dgates, dxp=dxp)
            if need[8]:
                # the bias is a per-expert constant added to the logits (in fp32): its gradient is the
                # column sum of the logits' gradient, taken before that is rounded to bf16
                dl32 = ops.router_topk_bwd(routing.gates, dgates, routing.ids, T, E, k, torch.float32)
                if dlogits_ext is not None:
                    dl32 = dl32 + dlogits_ext.float()
                dbias = dl32.sum(0)
                dlogits = dl32.to(torch.bfloat16)
            else:
                dlogits = ops.router_topk_bwd(routing.gates, dgates, routing.ids, T, E, k, torch.bfloat16)
                dlogits = dlogits + dlogits_ext.to(dlogits.dtype)
            if need[2]:
                dwr = _router_wgrad(dlogits, xn, ctx.wr_dtype)
            if want_dx:
                with torch.autocast("cuda", enabled=False):
                    d2 = dlogits @ wrb
                # (with the norm, the router's share joins inside the norm's backward kernel)
                dx = ops.permute_bwd(dxp, routing.row_to_pos, T, k, ctx.x_dtype, addend=None if ctx.has_norm else d2)
        if want_dx:
            if ctx.has_norm:
                dx, dnw = ops.rmsnorm_bwd(x, nw, rstd, dx, d2, dout if ctx.add_residual else None)
                dnw = dnw.to(ctx.nw_dtype) if need[1] else None
            elif ctx.add_residual:
                dx = dx + dout
            if not need[0]:
                dx = None
        return dx, dnw, dwr, dw1, dw3, dw2, None, None, dbias, None, None, None, None, None


def prenorm_moe(x: torch.Tensor, norm_weight: torch.Tensor, router_weight: torch.Tensor,
                w1: torch.Tensor, w3: torch.Tensor, w2: torch.Tensor, k: int, eps: float = 1e-6,
                add_residual: bool = True, bf16_weights=None, accumulate_into_grad: bool = False,
                return_routing: bool = False, fused_router: bool = True):
    """(x + MoE(RMSNorm(x)), router logits) for x [T,H]: model/gpt.py:32-33 with
    model/modules/norm.py:14-19 and model/modules/mlp.py:95-169 in one differentiable call.
    Router logits are bf16 (what the reference produces under its bf16 autocast); the output
    has the dtype of x.  H <= 8192.  `fused_router=False` takes the logits from the library's
    product (bit-identical to what `routed_moe` and `MoE.forward` select on) instead of the fused
    norm+router kernel, whose own summation order can move a bf16 logit by one unit in the last
    place."""
    grad_params = None
    if accumulate_into_grad:
        grad_params = tuple(w if (w.requires_grad and w.is_leaf) else None for w in (w1, w3, w2))
    routing = [] if return_routing else None
    res = _PreNormMoE.apply(x, norm_weight, router_weight, w1, w3, w2, float(eps), k, None, bf16_weights,
                            grad_params, add_residual, fused_router, routing)
    return (*res, _routing_dict(routing[0])) if return_routing else res


def routed_moe(x: torch.Tensor, router_weight: torch.Tensor, w1: torch.Tensor, w3: torch.Tensor,
               w2: torch.Tensor, k: int, bias: torch.Tensor | None = None, bf16_weights=None,
               accumulate_into_grad: bool = False, return_routing: bool = False):
    """(MoE(x), router logits) for x [T,H]: `router_linear` and `moe_ffn` as one autograd node
    (mlp.py:100-167), so that the two gradient contributions to x (expert path, router path)
    are summed inside the k-row-sum kernel.  The router product is a bf16 library product
    whatever the dtypes (the reference's behaviour under its bf16 autocast); the output has
    the dtype of x.  With `return_routing` a dict of the integer routing tensors and gates is
    returned as a third value."""
    if not return_routing and x.shape[0] > 0 and _forward_only(x, router_weight, w1, w3, w2, bias):
        # nothing to keep for a backward pass: the router product, then the rest in one call
        w1b, w3b, w2b = _weights_bf16(w1, w3, w2, bf16_weights)
        xn = ops.cast_bf16(_dense(x))
        with torch.autocast("cuda", enabled=False):
            logits = xn @ router_weight.detach().to(torch.bfloat16).t()
        return ops.ffn_forward(xn, logits, w1b, w3b, w2b, k, bias, out_dtype=x.dtype), logits
    grad_params = None
    if accumulate_into_grad:
        grad_params = tuple(w if (w.requires_grad and w.is_leaf) else None for w in (w1, w3, w2))
    routing = [] if return_routing else None
    res = _PreNormMoE.apply(x, None, router_weight, w1, w3, w2, 0.0, k, bias, bf16_weights, grad_params,
                            False, True, routing)
    return (*res, _routing_dict(routing[0])) if return_routing else res


class _ExpertsRows(torch.autograd.Function):
    @staticmethod
    def forward(ctx, rows, ids, w1, w3, w2, grad_params, routing_out):
        R, H = rows.shape
        E, I = w1.shape[0], w1.shape[1]
        rows = _dense(rows)
        if ids.dtype != torch.int64:
            ids = ids.to(torch.int32)
        w1b, w3b, w2b = _weights_bf16(w1, w3, w2, None)
        routing = ops.new_routing(R, H, E, I, 1, rows.device)
        train = any(ctx.needs_input_grad)
        out, xp, gu, act = ops.layer_forward(rows, w1b, w3b, w2b, 1, routing, rows.dtype, ids=_dense(ids), train=train)
        if train:
            ctx.save_for_backward(xp, gu, act, routing.buf, w1b, w3b, w2b)
        ctx.x_dtype, ctx.w_dtype = rows.dtype, w1.dtype
        ctx.grad_params = grad_params
        ctx.set_materialize_grads(False)
        ctx.out_shape = out.shape
        if routing_out is not None:
            routing_out.append(routing)
        return out

    @staticmethod
    def backward(ctx, dout):
        _first_order_only()
        xp, gu, act, buf, w1b, w3b, w2b = ctx.saved_tensors
        if dout is None:
            dout = torch.zeros(ctx.out_shape, dtype=ctx.x_dtype, device=xp.device)
        R, H = dout.shape
        dout = _dense(dout)
        if dout.dtype not in (torch.bfloat16, torch.float32):
            dout = dout.float()
        need = ctx.needs_input_grad
        ids, _, counts, offs, p2r, r2p, bad = ops.new_routing(R, H, w1b.shape[0], w1b.shape[1], 1, xp.device,
                                                              buf).pointers()
        drows = torch.empty((R, H), dtype=ctx.x_dtype, device=xp.device) if need[0] else None
        dw1, dw3, dw2 = _expert_gradients(ctx, dout, need[2:5], (0, 0, counts, offs, p2r, r2p, bad), xp, gu, act,
                                          w1b, w3b, w2b, 1, dx=drows)
        return drows, None, dw1, dw3, dw2, None, None


class _ExpertsRowsF32(torch.autograd.Function):
    @staticmethod
    def forward(ctx, rows, ids, w1, w3, w2):
        R, H = rows.shape
        E = w1.shape[0]
        rows, w1, w3, w2 = _dense(rows), _dense(w1), _dense(w3), _dense(w2)
        ids32 = _dense(ids.to(torch.int32))
        counts, offs, pos_to_row, row_to_pos, bad = ops.histogram_scan(ids32, E, return_bad=True)
        xp = ops.f32_gather_rows(rows, pos_to_row, 1)
        g = ops.f32_gemm_rows(xp, w1, offs, True)
        u = ops.f32_gemm_rows(xp, w3, offs, True)
        act = ops.f32_swiglu(g, u)
        y = ops.f32_gemm_rows(act, w2, offs, True)
        out = ops.f32_combine_fwd(y, None, row_to_pos, R, 1)
        if any(ctx.needs_input_grad):
            ctx.save_for_backward(xp, g, u, act, offs, pos_to_row, row_to_pos, w1, w3, w2)
        ctx.mark_non_differentiable(counts, offs, pos_to_row, row_to_pos, bad)
        ctx.set_materialize_grads(False)
        ctx.out_shape = out.shape
        return out, counts, offs, pos_to_row, row_to_pos, bad

    @staticmethod
    def backward(ctx, dout, *unused):
        _first_order_only()
        xp, g, u, act, offs, pos_to_row, row_to_pos, w1, w3, w2 = ctx.saved_tensors
        if dout is None:
            dout = torch.zeros(ctx.out_shape, dtype=torch.float32, device=xp.device)
        R, E = dout.shape[0], w1.shape[0]
        need = ctx.needs_input_grad
        dyp, _ = ops.f32_combine_bwd(_dense(dout.float()), None, None, pos_to_row, 1)
        dg, du = ops.f32_swiglu_bwd(ops.f32_gemm_rows(dyp, w2, offs, False), g, u)
        drows = None
        if need[0]:
            dxp = ops.f32_gemm_rows(dg, w1, offs, False)
            ops.f32_gemm_rows(du, w3, offs, False, out=dxp)
            drows = ops.f32_permute_bwd(dxp, row_to_pos, R, 1)
        dw1 = ops.f32_gemm_wgrad(dg, xp, offs, E) if need[2] else None
        dw3 = ops.f32_gemm_wgrad(du, xp, offs, E) if need[3] else None
        dw2 = ops.f32_gemm_wgrad(dyp, act, offs, E) if need[4] else None
        return drows, None, dw1, dw3, dw2


def experts_rows_f32(rows: torch.Tensor, ids: torch.Tensor, w1, w3, w2, return_routing: bool = False,
                     check_ids: bool = False):
    """`experts_rows` with every tensor and every product in fp32 (rows and weights fp32)."""
    for name, t in (("rows", rows), ("w1", w1), ("w3", w3), ("w2", w2)):
        if t.dtype != torch.float32:
            raise TypeError(f"experts_rows_f32: {name} must be fp32, got {t.dtype}")
    out, counts, offs, pos_to_row, row_to_pos, bad = _ExpertsRowsF32.apply(rows, ids, w1, w3, w2)
    if check_ids:
        n = int(bad.item())
        if n:
            raise ValueError(f"experts_rows_f32: {n} of {ids.numel()} expert ids lie outside [0, {w1.shape[0]})")
    if return_routing:
        return out, {"counts": counts, "offs": offs, "pos_to_row": pos_to_row, "row_to_pos": row_to_pos,
                     "bad_ids": bad}
    return out


def experts_rows(rows: torch.Tensor, ids: torch.Tensor, w1, w3, w2, return_routing: bool = False,
                 accumulate_into_grad: bool = False, check_ids: bool = False):
    """One rank's local expert share: rows [R,H] already dispatched to this rank, ids [R]
    local expert index of each row -> FFN output rows in the same (arrival) order.

    ids must lie in [0, E).  The dispatch kernels count the ids that do not (and treat such a
    row as belonging to the nearest valid expert, so nothing reads out of bounds); the count is
    a device tensor, `bad_ids` in the routing dict, so the hot path never waits for it.  With
    `check_ids` the call synchronises and raises ValueError if the count is not zero."""
    grad_params = None
    if accumulate_into_grad:
        grad_params = tuple(w if (w.requires_grad and w.is_leaf) else None for w in (w1, w3, w2))
    routing = [] if (check_ids or return_routing) else None
    out = _ExpertsRows.apply(rows, ids, w1, w3, w2, grad_params, routing)
    if check_ids:
        n = int(routing[0].bad_ids.item())
        if n:
            raise ValueError(f"experts_rows: {n} of {ids.numel()} expert ids lie outside [0, {w1.shape[0]})")
    if return_routing:
        r = routing[0]
        return out, {"counts": r.counts, "offs": r.offs, "pos_to_row": r.pos_to_row, "row_to_pos": r.row_to_pos,
                     "bad_ids": r.bad_ids}
    return out
