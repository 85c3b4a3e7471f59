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


@pytest.mark.parametrize("T,E,k,H", [(3001, 64, 2, 260), (2500, 128, 3, 1024), (63, 64, 2, 128), (65, 128, 2, 64), (9000, 512, 2, 32)])
@pytest.mark.parametrize("share", ["all", "falling"])
def test_router_weight_gradient_of_skewed_routing(pkg, lib, T, E, k, H, share):
    """All tokens with the same k experts, which lie apart, or most with a few: parts of an expert's rows and experts without any."""
    print("fp32 router, skewed", T, E, k, H, share, flush=True)
    (x, wr, w1, w3, w2), dy, _ = inputs(T, E, H, 16, T + E)
    g = torch.Generator(device="cuda").manual_seed(1)
    order = torch.randperm(E, generator=g, device="cuda").float()
    bias = -4.0 * order if share == "all" else -1.5 * torch.log1p(order)
    with torch.no_grad():  # (the last column of x is one)
        x[:, -1] = 1.0
        wr[:, -1] = bias
    leaves = [x, wr, w1, w3, w2]
    res = []
    for call in both(pkg, T, E, k, H, 16):
        out, logits = call(*leaves)
        res.append(torch.autograd.grad(out, leaves[1], dy)[0])
    rows = torch.bincount(logits.topk(k, -1).indices.flatten(), minlength=E)
    assert share != "all" or int((rows == T).sum()) >= 1
    close("dwr", *res)
    assert not bool(res[0][rows == 0].any())


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


@pytest.mark.parametrize("loss_on_logits", [False, True])
@pytest.mark.parametrize("who", ["hook", "hook that changes it", "retain_grad", "asked for", "node", "product's node"])
def test_the_logits_are_on_the_way_to_the_output(pkg, lib, who, loss_on_logits):
    """Whoever looks at the logits' gradient sees the experts' share of it, and what a hook makes of it is what goes on."""
    print("fp32 router, logits observed:", who, loss_on_logits, flush=True)
    T, E, k, H, I = 150, 8, 2, 128, 64
    leaves, dy, dl = inputs(T, E, H, I, 7)
    leaves[0] = leaves[0].detach().view(3, 50, H).requires_grad_(True)
    dy, dl = dy.view(3, 50, H), dl.view(3, 50, E)
    routed = both(pkg, T, E, k, H, I)[0]

    def apart(x, wr, w1, w3, w2):
        logits = F.linear(x, wr)
        return pkg.moe_ffn_f32(x.reshape(T, H), logits.reshape(T, E), w1, w3, w2, k).reshape(x.shape), logits

    res = []
    for call in (routed, apart):
        out, logits = call(*leaves)
        assert out.shape == (3, 50, H) and logits.shape == (3, 50, E) and not logits._is_view()
        outs, given = ([out, logits], [dy, dl]) if loss_on_logits else ([out], [dy])
        seen = []
        if who == "hook":
            logits.register_hook(lambda g: seen.append(g.clone()))
        elif who == "hook that changes it":
            logits.register_hook(lambda g: seen.append(g.clone()) or 3 * g)
        elif who == "retain_grad":
            logits.retain_grad()
        elif who == "node":
            logits.grad_fn.register_prehook(lambda g: seen.append(g[0].clone()))
        elif who == "product's node":
            node = logits.grad_fn
            while len(node.next_functions) == 1:
                node = node.next_functions[0][0]
            node.register_prehook(lambda g: seen.append(g[0].clone().view(3, 50, E)))
        want = leaves + ([logits] if who == "asked for" else [])
        grads = list(torch.autograd.grad(outs, want, given))
        if who == "retain_grad":
            seen.append(logits.grad)
        if seen:
            grads.append(seen[0])
        assert len(grads) == 6 and len(seen) == (who != "asked for")
        res.append(grads)
    for name, a, b in zip(("dx", "dwr", "dw1", "dw3", "dw2", "dlogits"), *res):
        close(name, a, b)
    assert bool(res[0][5].any())


def test_logits_may_be_written_to(pkg, lib):
    print("fp32 router, logits changed in place", flush=True)
    T, E, k, H, I = 40, 8, 2, 64, 32
    leaves, dy, dl = inputs(T, E, H, I, 3)
    res = []
    for call in both(pkg, T, E, k, H, I):
        out, logits = call(*leaves)
        logits.mul_(2)
        res.append(torch.autograd.grad([out, logits], leaves, [dy, dl]))
    for name, a, b in zip(("dx", "dwr", "dw1", "dw3", "dw2"), *res):
        close(name, a, b)


class Linear(torch.nn.Linear):
    pass


def global_hook(m):
    h = torch.nn.modules.module.register_module_forward_hook(lambda mod, inp, o: None)
    return h.remove


def own_forward(m):
    r = m.router
    r.forward = lambda x: F.linear(x, r.weight)
    return lambda: delattr(r, "forward")


def other_router(make):
    def change(m):
        old, new = m.router, make(m.router)
        with torch.no_grad():
            new.weight.copy_(old.weight)
        m.router = new
        return lambda: setattr(m, "router", old)
    return change


def with_bias(r):
    new = torch.nn.Linear(r.in_features, r.out_features, device="cuda")
    torch.nn.init.zeros_(new.bias)
    return new


MORE_THAN_A_PRODUCT = {
    "forward hook": lambda m: m.router.register_forward_hook(lambda mod, inp, o: None).remove,
    "pre-hook": lambda m: m.router.register_forward_pre_hook(lambda mod, inp: None).remove,
    "backward hook": lambda m: m.router.register_full_backward_hook(lambda mod, gi, go: None).remove,
    "global hook": global_hook,
    "bias": other_router(with_bias),
    "subclass": other_router(lambda r: Linear(r.in_features, r.out_features, bias=False, device="cuda")),
    "own forward": own_forward,
}


@pytest.mark.parametrize("what", ["plain"] + list(MORE_THAN_A_PRODUCT))
def test_module_takes_it_unless_the_router_is_more_than_a_product(pkg, lib, what):
    print("fp32 module, router:", what, flush=True)
    m = pkg.MoE(pkg.ModelConfig(hidden_size=128, num_experts=8, num_experts_per_tok=2, moe_intermediate_size=64, init_std=0.05), 2)
    g = torch.Generator(device="cuda").manual_seed(2)
    x, dy = (torch.randn(2, 50, 128, generator=g, device="cuda") for _ in range(2))

    def launches():
        names = []

        class Obs:
            def before(self, name):
                names.append(name)

            def after(self, name):
                pass

        lib.observer = Obs()
        try:
            out, logits = m(x)
            out.backward(dy)
        finally:
            lib.observer = None
        return [out.detach(), logits.detach()], names.count("moe_f32_permute_bwd_router")

    plain, times = launches()
    assert times == 1
    undo = MORE_THAN_A_PRODUCT.get(what, lambda m: lambda: None)(m)
    try:
        outs, times = launches()
    finally:
        undo()
    assert times == (what == "plain")
    for name, a, b in zip(("out", "logits"), plain, outs):
        close(name, a, b)
