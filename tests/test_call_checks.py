"""What a call is refused for on the host, before anything is launched: on tensors that only claim to be on a
GPU (no storage, no kernel runs), so that the checks are seen without one."""
import importlib

import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode

from conftest import load_pkg

BF16, F32 = torch.bfloat16, torch.float32
T, H, E, I, K = 4, 64, 8, 32, 2


def _gpu(*shape, dtype=BF16):
    return torch.empty(*shape, device="cuda", dtype=dtype)


def _weights(dtype=BF16):
    return [_gpu(E, I, H, dtype=dtype), _gpu(E, I, H, dtype=dtype), _gpu(E, H, I, dtype=dtype)]


@pytest.mark.parametrize("entry", ["moe_ffn", "routed_moe", "prenorm_moe"])
@pytest.mark.parametrize("which", [0, 1, 2])
@pytest.mark.parametrize("wrong,error,match", [
    (lambda c: c.transpose(1, 2).contiguous().transpose(1, 2), RuntimeError, "contiguous"),
    (lambda c: c.float(), TypeError, "bf16"),
    (lambda c: c[:-1], RuntimeError, "shape"),
    (lambda c: c.new_empty(E, c.shape[2], c.shape[1]), RuntimeError, "shape"),
    (lambda c: torch.empty(c.shape, dtype=BF16, device="cpu"), RuntimeError, "GPU"),
])
def test_copies_of_the_weights_are_what_a_cast_would_give(entry, which, wrong, error, match):
    pkg = load_pkg()
    with FakeTensorMode():
        x, wr = _gpu(T, H, dtype=F32), _gpu(E, H)
        masters, copies = _weights(F32), _weights()
        copies[which] = wrong(copies[which])
        front = {"moe_ffn": (x, _gpu(T, E)), "routed_moe": (x, wr), "prenorm_moe": (x, _gpu(H, dtype=F32), wr)}[entry]
        with pytest.raises(error, match=match):
            getattr(pkg, entry)(*front, *masters, K, bf16_weights=copies)


@pytest.mark.parametrize("tokens", [T, 65])
@pytest.mark.parametrize("shape", [(E, H - 8), (E, H + 8), (E, H, 1)])
def test_router_weight_has_the_width_of_x(tokens, shape):
    pkg = load_pkg()
    with FakeTensorMode():
        x, wr = _gpu(tokens, H), _gpu(*shape)
        for call in (lambda: pkg.routed_moe(x, wr, *_weights(), K),
                     lambda: pkg.prenorm_moe(x, _gpu(H, dtype=F32), wr, *_weights(), K)):
            with pytest.raises(RuntimeError, match="router weight"):
                call()
        with pytest.raises(RuntimeError, match="mat1 and mat2|reduction dim|expects a tensor"):
            pkg.router_linear(x, wr)


def test_router_weight_is_where_x_is():
    pkg = load_pkg()
    with FakeTensorMode():
        x, wr = _gpu(T, H), torch.empty(E, H, dtype=BF16, device="cpu")
        with pytest.raises(RuntimeError, match="GPU"):
            pkg.routed_moe(x, wr, *_weights(), K)
        with pytest.raises(RuntimeError, match="device"):
            pkg.router_linear(x, wr)


@pytest.mark.parametrize("weight,match", [
    (lambda: torch.empty(H, device="cpu"), "GPU"),
    (lambda: _gpu(H - 8, dtype=F32), "norm's weight"),
    (lambda: _gpu(2 * H, dtype=F32), "norm's weight"),
])
def test_norm_weight_is_on_the_gpu_and_as_wide_as_x(weight, match):
    pkg = load_pkg()
    with FakeTensorMode():
        with pytest.raises(RuntimeError, match=match):
            pkg.prenorm_moe(_gpu(T, H), weight(), _gpu(E, H), *_weights(), K)


@pytest.mark.parametrize("dual", [0, 1, 2, 3, 4])
@pytest.mark.parametrize("entry", ["moe_ffn", "moe_ffn_f32", "routed_moe", "prenorm_moe", "experts_rows",
                                   "experts_rows_f32"])
@pytest.mark.parametrize("grad", [False, True])
@pytest.mark.parametrize("return_routing", [False, True])
def test_forward_mode_is_refused(entry, dual, grad, return_routing):
    """... whether or not anything requires a gradient (plain host tensors: the refusal comes first)."""
    pkg = load_pkg()
    w = [torch.zeros(E, I, H, requires_grad=grad), torch.zeros(E, I, H), torch.zeros(E, H, I)]
    x, wr, norm, logits, ids = torch.zeros(T, H), torch.zeros(E, H), torch.ones(H), torch.zeros(T, E), torch.zeros(T)
    args = {"moe_ffn": [x, logits, *w, K], "moe_ffn_f32": [x, logits, *w, K], "routed_moe": [x, wr, *w, K],
            "prenorm_moe": [x, norm, wr, *w, K], "experts_rows": [x, ids.long(), *w],
            "experts_rows_f32": [x, ids.long(), *w]}[entry]
    floats = [i for i, a in enumerate(args) if torch.is_tensor(a) and a.is_floating_point()]
    at = floats[dual % len(floats)]
    fn = getattr(importlib.import_module(pkg.__name__ + ".functional"), entry)
    with torch.autograd.forward_ad.dual_level():
        args[at] = torch.autograd.forward_ad.make_dual(args[at], torch.ones_like(args[at]))
        with pytest.raises(NotImplementedError):
            fn(*args, return_routing=return_routing)
        with torch.no_grad(), pytest.raises(NotImplementedError):
            fn(*args, return_routing=return_routing)


@pytest.mark.parametrize("dtype,entry", [(BF16, "moe_ffn"), (F32, "moe_ffn_f32")])
@pytest.mark.parametrize("logits,bias,error,match", [
    (lambda d: _gpu(T - 1, E, dtype=d), lambda: None, RuntimeError, "logits"),
    (lambda d: _gpu(1, T, E, dtype=d), lambda: None, RuntimeError, "logits|shapes"),
    (lambda d: _gpu(T, E - 1, dtype=d), lambda: None, RuntimeError, "logits|shapes"),
    (lambda d: _gpu(T, E, dtype=d), lambda: _gpu(E - 1, dtype=F32), RuntimeError, "bias"),
    (lambda d: _gpu(T, E, dtype=d), lambda: _gpu(E), TypeError, "bias"),
])
def test_logits_and_bias_belong_to_x(dtype, entry, logits, bias, error, match):
    pkg = load_pkg()
    with FakeTensorMode():
        with pytest.raises(error, match=match):
            getattr(pkg, entry)(_gpu(T, H, dtype=dtype), logits(dtype), *_weights(dtype), K, bias=bias())


def test_fp32_rows_are_a_matrix():
    pkg = load_pkg()
    with FakeTensorMode():
        w = [_gpu(E, I, H, dtype=F32), _gpu(E, I, H, dtype=F32), _gpu(E, H, I, dtype=F32)]
        with pytest.raises(RuntimeError, match="x .tokens, hidden."):
            pkg.moe_ffn_f32(_gpu(T, H, 2, dtype=F32), _gpu(T, E, dtype=F32), *w, K)
