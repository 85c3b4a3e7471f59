"""The fp32 layer with the router product inside: the same outputs, bit for bit, and the same gradients as `nn.Linear` and the
experts apart, for every set of gradients that can be asked for."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


def inputs(T, E, H, I, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    r = lambda *s, std=1.0: torch.randn(*s, generator=g, device="cuda") * std
    return [t.requires_grad_(True) for t in (r(T, H), r(E, H, std=0.05), r(E, I, H, std=0.05), r(E, I, H, std=0.05),
                                             r(E, H, I, std=0.05))], r(T, H), r(T, E, std=0.1)


def both(pkg, T, E, k, H, I):
    from importlib import import_module
    routed = import_module(pkg.__name__ + ".functional").routed_moe_f32

    def apart(x, wr, w1, w3, w2):
        logits = F.linear(x, wr)
        return pkg.moe_ffn_f32(x, logits, w1, w3, w2, k), logits

    return (lambda *t: routed(*t, k)), apart


def close(name, a, b):
    # sums of up to T or H products in fp32, on both sides: sqrt(n) 2^-24, and the gate gradients' differences, of which the
    # largest terms cancel
    assert (a is None) == (b is None), name
    if a is not None:
        assert (a - b).norm() <= 1e-5 * b.norm() + 1e-30, (name, float((a - b).norm() / b.norm()))


@pytest.mark.parametrize("T,E,k,H,I", [
    (1, 4, 2, 64, 32), (7, 5, 3, 260, 36), (300, 8, 2, 1024, 64), (513, 64, 8, 252, 64), (4099, 4, 1, 512, 32),
    (5000, 4, 2, 260, 32),   # slices of an expert's rows
    (900, 96, 6, 2052, 16),
])
@pytest.mark.parametrize("outs", ["out", "logits", "both"])
def test_gradients(pkg, lib, T, E, k, H, I, outs):
    print("fp32 router", T, E, k, H, I, outs, flush=True)
    leaves, dy, dl = inputs(T, E, H, I, T + E)
    res = []
    for call in both(pkg, T, E, k, H, I):
        for t in leaves:
            t.grad = None
        out, logits = call(*leaves)
        if outs == "both":
            torch.autograd.backward([out, logits], [dy, dl])
        else:
            (out if outs == "out" else logits).backward(dy if outs == "out" else dl)
        res.append([out.detach(), logits.detach()] + [t.grad for t in leaves])
    assert torch.equal(res[0][0], res[1][0]) and torch.equal(res[0][1], res[1][1])
    for name, a, b in zip(("dx", "dwr", "dw1", "dw3", "dw2"), res[0][2:], res[1][2:]):
        close(name, a, b)


@pytest.mark.parametrize("wanted", [(0,), (1,), (0, 1), (2, 4), (1, 3)])
def test_some_gradients(pkg, lib, wanted):
    T, E, k, H, I = 200, 8, 2, 128, 64
    print("fp32 router, gradients of", wanted, flush=True)
    leaves, dy, _ = inputs(T, E, H, I, 5)
    for i, t in enumerate(leaves):
        t.requires_grad_(i in wanted)
    res = [torch.autograd.grad(call(*leaves)[0], [leaves[i] for i in wanted], dy) for call in both(pkg, T, E, k, H, I)]
    for i, a, b in zip(wanted, *res):
        close(str(i), a, b)


def test_no_tokens_and_logits_twice(pkg, lib):
    print("fp32 router: no tokens, logits differentiated twice", flush=True)
    leaves, dy, dl = inputs(0, 4, 64, 32, 1)
    routed, apart = both(pkg, 0, 4, 2, 64, 32)
    out, _ = routed(*leaves)
    out.backward(dy)
    assert all(not bool(t.grad.any()) for t in leaves)
    leaves, dy, dl = inputs(50, 4, 64, 32, 1)
    second = []
    for call in (routed, apart):
        dx, = torch.autograd.grad(call(*leaves)[1], leaves[0], dl, create_graph=True)
        second.append(torch.autograd.grad((dx * dx).sum(), leaves[1])[0])
    close("second", *second)
    with pytest.raises(RuntimeError):
        torch.autograd.grad(routed(*leaves)[0], leaves[0], dy, create_graph=True)


def test_module_takes_it_unless_the_router_is_more_than_a_product(pkg, lib):
    print("fp32 module, router with a hook", flush=True)
    m = pkg.MoE(pkg.ModelConfig(hidden_size=128, num_experts=8, num_experts_per_tok=2, moe_intermediate_size=64, init_std=0.05), 2)
    x = torch.randn(2, 50, 128, device="cuda")
    out, logits = m(x)
    seen = []
    h = m.router.register_forward_hook(lambda mod, inp, o: seen.append(1))
    out2, logits2 = m(x)
    h.remove()
    assert seen and torch.equal(out, out2) and torch.equal(logits, logits2)
