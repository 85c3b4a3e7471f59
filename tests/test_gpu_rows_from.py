"""A layer with its router keeps no rows in expert order where its weight gradients are tiled: gate/up and the gradients of its weights read
the tokens' rows.  With the logits given it keeps them: the same bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def up(n):
    return -(-n // 256) * 256


class Kept(torch.autograd.graph.saved_tensors_hooks):
    """Bytes that a layer keeps for its backward pass in one buffer: rows in expert order, if it keeps any, g and u, act."""

    def __init__(self):
        self.bytes = 0
        super().__init__(self.pack, lambda t: t)

    def __enter__(self):
        super().__enter__()
        return self

    def pack(self, t):
        if t.dtype == torch.uint8:
            self.bytes += t.numel()
        return t


@pytest.mark.parametrize("T,H,E,I,k,skew", [
    (2600, 1024, 128, 256, 8, 0.6),   # two stacks in one result; experts of one k-tile to a dozen
    (1800, 2040, 64, 520, 6, 0.5),    # three problems, columns that end in the middle
    (5200, 2048, 64, 1024, 2, 2.0),   # dealt longest first; experts with a row or two and without any
    (10400, 1992, 64, 1000, 1, 1.0),
    (9216, 1536, 48, 768, 1, -1.0),   # 192 rows each: whole k-tiles
    # ... and in the kernel for small launches: a step or two, ends inside a step, experts cut into segments, more experts than lanes
    (5, 72, 4, 24, 2, 0.0),
    (130, 264, 16, 136, 4, 0.5),
    (3333, 1416, 12, 568, 3, 0.3),
    (8192, 1024, 8, 512, 2, 1.5),
    (900, 512, 96, 192, 4, 0.4),
])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])  # of the weights and their gradients
def test_training_reads_the_tokens(pkg, T, H, E, I, k, skew, dtype):
    print("rows from the tokens, training", T, H, E, I, k, skew, dtype, flush=True)
    g = torch.Generator(device="cuda").manual_seed(T + H)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda").to(torch.bfloat16)
    x, dy, ws = r(T, H), r(T, H), [w.to(dtype) for w in (r(E, I, H), r(E, I, H), r(E, H, I))]
    wr = r(E, H) * 0.02
    bias = -skew * torch.arange(E, device="cuda", dtype=torch.float32).log1p()
    if skew < 0:  # every expert in turn
        wr = wr * 0
        x[:, :E] = 0
        x[torch.arange(T, device="cuda"), torch.arange(T, device="cuda") % E] = 1
        wr[torch.arange(E, device="cuda"), torch.arange(E, device="cuda")] = 1
        bias = None
    calls = []

    class Obs:
        def before(self, name):
            calls.append(name)

        def after(self, name):
            pass

    def passed(layer):
        leaves = [w.detach().requires_grad_(True) for w in ws]
        lib.observer = Obs()
        try:
            with Kept() as kept:
                out, logits = layer(*leaves)
            out.backward(dy)
        finally:
            lib.observer = None
        return out.detach(), logits.detach(), [w.grad for w in leaves], kept.bytes

    lib = pkg.ops._lib.load()
    xr = x.detach().requires_grad_(True)
    out, logits, grads, kept = passed(lambda a, b, c: pkg.routed_moe(xr, wr, a, b, c, k, bias=bias))
    assert ("moe_gemm_wgrad_all" if E >= 48 and H > 1000 else "moe_wgrad_multi") in calls
    want, _, want_grads, want_kept = passed(lambda a, b, c: (pkg.moe_ffn(x, logits, a, b, c, k, bias=bias), logits))
    assert want_kept - kept == up(T * k * H * 2)  # the rows in expert order
    assert torch.equal(out, want)
    for i, (a, b) in enumerate(zip(grads, want_grads)):
        assert torch.equal(a.view(torch.uint8), b.view(torch.uint8)), i


@pytest.mark.parametrize("T,H,E,I,k", [(2600, 1024, 128, 256, 8), (700, 512, 16, 192, 4)])  # tiled; in the kernel for small launches
@pytest.mark.parametrize("types", [(torch.float32,) * 3, (torch.float32, torch.bfloat16, torch.bfloat16)])  # w1, w3, w2: in one launch or not
@pytest.mark.parametrize("beside", ["nothing", "bias", "logits"])  # what else takes part in the router's gradient
def test_added_up_with_the_tokens_rows(pkg, T, H, E, I, k, types, beside):
    """Gradients of the weights added to .grad over two passes, of one type or of several, with the router's gradient worked out inside the call or
    beside it."""
    print("rows from the tokens, added up", T, H, E, I, k, types, beside, flush=True)
    g = torch.Generator(device="cuda").manual_seed(T)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda").to(torch.bfloat16)
    x, dy, dl = r(T, H), r(T, H), r(T, E)
    ws = [w.to(t) for w, t in zip((r(E, I, H), r(E, I, H), r(E, H, I)), types)]
    wr, bias = r(E, H) * 0.02, torch.randn(E, generator=g, device="cuda") * 0.1
    lib = pkg.ops._lib.load()
    names = []

    class Obs:
        before = staticmethod(names.append)
        after = staticmethod(lambda name: None)

    def passes(layer):
        leaves = [w.detach().requires_grad_(True) for w in ws]
        b = bias.detach().requires_grad_(beside == "bias")
        names.clear()
        with Kept() as kept:
            for _ in range(2):
                out, logits = layer(leaves, b)
                loss = [(out, dy)] + ([(logits, dl)] if beside == "logits" and logits.requires_grad else [])
                lib.observer = Obs()
                try:
                    torch.autograd.backward([t for t, _ in loss], [d for _, d in loss])
                finally:
                    lib.observer = None
        return out.detach(), logits.detach(), [w.grad for w in leaves] + ([b.grad] if beside == "bias" else []), kept.bytes

    xr, wrr = x.detach().requires_grad_(True), wr.detach().requires_grad_(True)
    out, logits, grads, kept = passes(lambda w, b: pkg.routed_moe(xr, wrr, *w, k, bias=b, accumulate_into_grad=True))
    wgrads = {n for n in names if "wgrad" in n} - {"moe_router_wgrad"}
    if E == 16:
        assert wgrads == {"moe_wgrad_multi"}
    elif types[0] == types[1]:
        assert "moe_gemm_wgrad_all" in wgrads
    else:
        assert "moe_gemm_wgrad" in wgrads and "moe_gemm_wgrad_all" not in wgrads
    assert ("moe_permute_bwd_router" in names) == (beside == "nothing")
    want, _, want_grads, want_kept = passes(
        lambda w, b: (pkg.moe_ffn(x, logits, *w, k, bias=b, accumulate_into_grad=True), logits))
    assert want_kept - kept == 2 * up(T * k * H * 2)
    assert torch.equal(out, want)
    for i, (a, b) in enumerate(zip(grads, want_grads)):
        assert torch.equal(a.view(torch.uint8), b.view(torch.uint8)), i


@pytest.mark.parametrize("counts,H,I", [
    ([160] * 64, 2048, 1024),                          # two and a half k-tiles each
    ([0, 1, 63, 64, 65, 127, 128, 129, 900] * 8, 2040, 520),  # three problems; all numbers of k-tiles around one and two
    ([40, 30] * 31 + [9000, 0], 2048, 1024),           # longest first
    ([250, 0, 130, 400] * 12, 1536, 768),
])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_rows_gradient_is_read_where_it_is(pkg, counts, H, I, dtype):
    """In fp32 the output's gradient is rounded and put in order by a pass of its own."""
    E, R = len(counts), sum(counts)
    assert R >= 160 * E
    g = torch.Generator(device="cuda").manual_seed(R)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda").to(torch.bfloat16)
    x, dy, ws = r(R, H), r(R, H), [w.to(dtype) for w in (r(E, I, H), r(E, I, H), r(E, H, I))]
    ids = torch.arange(E, device="cuda").repeat_interleave(torch.tensor(counts, device="cuda"))
    ids = ids[torch.randperm(R, generator=g, device="cuda")]
    lib = pkg.ops._lib.load()
    force = lib.cdll.moe_gemm_force_row_tile

    def passed(kind, height):
        print("rows, gradient in place", E, R, H, I, dtype, kind, height, flush=True)
        leaf, leaves = x.to(kind, copy=True).requires_grad_(True), [w.detach().requires_grad_(True) for w in ws]
        names = []

        class Obs:
            before = staticmethod(names.append)
            after = staticmethod(lambda name: None)

        try:
            force(height)
            out = pkg.experts_rows(leaf, ids, *leaves)
            lib.observer = Obs()
            out.backward(dy.to(kind))
        finally:
            lib.observer = None
            force(0)
        assert ("moe_combine_bwd" in names) == (kind == torch.float32), names
        return [leaf.grad.bfloat16()] + [w.grad for w in leaves]

    want = passed(torch.float32, 0)
    for height in (0, 1, 64, 128, 256):
        for i, (a, b) in enumerate(zip(passed(torch.bfloat16, height), want)):
            assert torch.equal(a.view(torch.uint8), b.view(torch.uint8)), (height, i)


@pytest.mark.parametrize("over", ["dx", "dxp", "dw1", "dw2"])
def test_a_result_over_the_outputs_gradient(pkg, over):
    """Through the C interface a result may take the place of dout; dout is then read before anything is written there."""
    ops = pkg.ops
    E, R, H, I = 128, 20480, 1024, 256
    print("rows, a result over the gradient", over, flush=True)
    g = torch.Generator(device="cuda").manual_seed(R)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda").to(torch.bfloat16)
    x, dy, ws = r(R, H), r(R, H), (r(E, I, H), r(E, I, H), r(E, H, I))
    _, rt, xp, gu, act = ops.layer_forward(x, r(R, E), *ws, 1, train=True)

    def passed(name):
        room = torch.empty(max(R * H, E * I * H), dtype=torch.bfloat16, device="cuda")
        dout = room[:R * H].view(R, H).copy_(dy)
        t = {n: torch.empty_like(w) for n, w in zip(("dw1", "dw3", "dw2"), ws)}
        t["dx"] = torch.empty_like(x)
        if name == "dxp" or over == "dxp":
            t["dxp"] = torch.empty_like(x)
        if name:
            t[name] = room[:t[name].numel()].view(t[name].shape)
        ops.layer_backward(dout, 1, None, rt.ids, rt.offs, rt.pos_to_row, rt.row_to_pos, xp, gu, act, *ws,
                           (t["dw1"], t["dw3"], t["dw2"]), dx=t["dx"], dxp=t.get("dxp"))
        return t

    want, got = passed(None), passed(over)
    for name in want:
        assert torch.equal(got[name].view(torch.uint8), want[name].view(torch.uint8)), name
