"""The router product and the selection in one launch: logits of the bits that the library's product has, the selection that
`moe_ffn` makes on them, and the same rest of the layer; at the edges of the sizes that it takes."""
import math
import random

import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu

BF16, F32 = torch.bfloat16, torch.float32


@pytest.mark.parametrize("T,E,k,H,taken", [
    (65, 2, 1, 64, True), (65, 64, 8, 2048, True), (66, 128, 8, 1024, True), (70, 33, 3, 72, True),  # the fewest tokens; ends of slices
    (256, 8, 2, 1016, True), (257, 8, 2, 1016, True), (257, 12, 3, 128, True), (300, 16, 16, 320, True),  # one chain and four, to 16 experts
    (2048, 12, 4, 256, True), (3200, 16, 2, 512, True), (3333, 12, 3, 1416, True), (12288, 8, 2, 1024, True), (8192, 3, 3, 2048, True),
    (4081, 32, 4, 1032, True), (4096, 32, 32, 1032, True), (2048, 64, 6, 1600, True), (4096, 64, 8, 2048, True),
    (1360, 96, 6, 1360, True), (1361, 96, 6, 1360, True), (1031, 77, 5, 1208, True), (1009, 128, 8, 1000, True), (4091, 100, 7, 1000, True),
    (64, 8, 2, 1024, False), (4097, 64, 8, 1024, False), (8193, 8, 2, 2048, False), (1531, 24, 4, 1024, False), (700, 128, 8, 1032, False),
])
@pytest.mark.parametrize("x_type,w_type", [(BF16, BF16), (F32, F32)])
def test_bits_of_the_two_calls(pkg, lib, T, E, k, H, taken, x_type, w_type):
    print("router select", T, E, k, H, x_type, flush=True)
    g = torch.Generator(device="cuda").manual_seed(T + E + H)
    r = lambda *s, std=1.0: torch.randn(*s, generator=g, device="cuda") * std
    I = 8
    x, wr = r(T, H).to(x_type), r(E, H, std=0.05).to(w_type)
    w1, w3, w2 = (r(*s, std=0.05).to(BF16) for s in ((E, I, H), (E, I, H), (E, H, I)))
    bias = r(E) if k % 2 else None
    want = F.linear(x.to(BF16), wr.to(BF16))
    names = []

    class Obs:
        before = staticmethod(names.append)
        after = staticmethod(lambda name: None)

    lib.observer = Obs()
    try:
        out, lg = pkg.routed_moe(x, wr, w1, w3, w2, k, bias=bias)   # nothing to differentiate: one call for the pass
    finally:
        lib.observer = None
    assert ("moe_router_select" in names) == taken, names
    if T <= 64:
        return  # (the kernels for few tokens sum up in an order of their own)
    assert torch.equal(lg, want)
    ref, routing = pkg.moe_ffn(x, want, w1, w3, w2, k, bias=bias, return_routing=True)
    assert torch.equal(out, ref)
    ws = [t.clone().requires_grad_(True) for t in (wr, w1, w3, w2)]
    out, lg, kept = pkg.routed_moe(x, *ws, k, bias=bias, return_routing=True)
    assert torch.equal(lg, want) and torch.equal(out, ref)
    for name in ("ids", "gates", "counts", "offs", "pos_to_row", "row_to_pos"):
        assert torch.equal(kept[name], routing[name]), name
    # what the backward pass reads: the router's weight and x in bf16
    dy = r(T, H).to(x_type)
    out.backward(dy)
    xr, wd = x.to(BF16).float(), ws[0].grad.float()
    lr = want.clone().requires_grad_(True)
    pkg.moe_ffn(x, lr, w1, w3, w2, k, bias=bias).backward(dy)
    ref_w = lr.grad.float().T @ xr
    # (roundings of dlogits and of the result to bf16, sums of T products in fp32)
    assert (wd - ref_w).norm() <= 2.0 ** -7 * ref_w.norm() + 1e-6


@pytest.mark.parametrize("T,E,k,H,w_type,taken", [
    (1024, 96, 6, 1360, F32, False), (1024, 96, 6, 1360, BF16, True), (1025, 96, 6, 1360, F32, True), (70, 65, 3, 1032, F32, False),
    (70, 64, 3, 1032, F32, True), (70, 65, 3, 1024, F32, True),
])
def test_long_rows_of_fp32_weights(pkg, lib, T, E, k, H, w_type, taken):
    """Few tokens and long router rows in fp32: the product stays with the library.  The same bits either way."""
    print("router select, long rows", T, E, k, H, w_type, flush=True)
    g = torch.Generator(device="cuda").manual_seed(T + E + H)
    x, wr = torch.randn(T, H, generator=g, device="cuda"), (torch.randn(E, H, generator=g, device="cuda") * 0.05).to(w_type)
    ws = [(torch.randn(*s, generator=g, device="cuda") * 0.05).to(BF16) for s in ((E, 8, H), (E, 8, H), (E, H, 8))]
    names = []

    class Obs:
        before = staticmethod(names.append)
        after = staticmethod(lambda name: None)

    lib.observer = Obs()
    try:
        out, lg = pkg.routed_moe(x, wr, *ws, k)
    finally:
        lib.observer = None
    assert ("moe_router_select" in names) == taken, names
    want = F.linear(x.to(BF16), wr.to(BF16))
    assert torch.equal(lg, want)
    assert torch.equal(out, pkg.moe_ffn(x, want, *ws, k))


def edges():
    """Sizes on both sides of the lines where the order of a logit's sum changes, or the launch that makes it."""
    few = [(T, E, H) for T in (65, 256, 257, 2048, 2049, 3200, 3201) for E in (2, 12, 13, 16)
           for H in (64, 120, 128, 312, 320, 504, 512, 1016, 1024, 2048)]
    few += [(T, E, H) for T in (8192, 8193, 12288, 12289) for E in (2, 16) for H in (1016, 1024, 1032)]
    many = [(T, E, H) for E in (17, 31, 32, 48, 49, 64, 65, 80, 112, 113, 128) for H in (64, 1024, 1032, 1536, 2048)
            for T in {t + d for n in (512, 1024) for t in (16 * (n // -(-E // 16)),) for d in (0, 1)} | {65, 4096, 4097}]
    return few + many


def test_bits_at_the_lines_and_over_the_ranges(pkg, lib):
    """Whichever launch makes a logit, it has the bits that nn.Linear gives it: at every line of the rule, and for 300 sizes drawn."""
    rng = random.Random(7)
    log = lambda lo, hi: int(math.exp(rng.uniform(math.log(lo), math.log(hi))))
    sizes = edges() + [(log(65, 12288), rng.choice([log(2, 16), log(32, 128)]), log(8, 256) * 8) for _ in range(300)]
    names, taken = [], 0

    class Obs:
        before = staticmethod(names.append)
        after = staticmethod(lambda name: None)

    g = torch.Generator(device="cuda").manual_seed(7)
    x_all = torch.randn(12289 * 2048, generator=g, device="cuda").to(BF16)
    wr_all = (torch.randn(128 * 2048, generator=g, device="cuda") * 0.05).to(BF16)
    w_all = torch.zeros(128 * 2048 * 8, dtype=BF16, device="cuda")
    for i, (T, E, H) in enumerate(sizes):
        if i % 100 == 0:
            print("router select, sizes from", i, "of", len(sizes), flush=True)
        x, wr = x_all[:T * H].view(T, H), wr_all[:E * H].view(E, H)
        w1, w2 = w_all[:E * H * 8].view(E, 8, H), w_all[:E * H * 8].view(E, H, 8)
        names.clear()
        lib.observer = Obs()
        try:
            _, lg = pkg.routed_moe(x, wr, w1, w1, w2, min(E, 2))
        finally:
            lib.observer = None
        taken += "moe_router_select" in names
        assert torch.equal(lg, F.linear(x, wr)), (T, E, H)
    assert 3 * taken >= len(sizes)


def test_values_that_are_not_finite(pkg):
    print("router select, not finite", flush=True)
    g = torch.Generator(device="cuda").manual_seed(3)
    r = lambda *s: (torch.randn(*s, generator=g, device="cuda") * 0.1).to(BF16)
    for T, E, k, H in ((130, 8, 2, 256), (130, 64, 8, 1536), (130, 128, 8, 512)):
        x, wr = r(T, H), r(E, H)
        x[3, 5], x[64, 7], wr[1, 2] = float("nan"), float("inf"), float("-inf")
        w1, w3, w2 = r(E, 8, H), r(E, 8, H), r(E, H, 8)
        _, lg = pkg.routed_moe(x, wr, w1, w3, w2, k)
        want = F.linear(x, wr)
        assert torch.equal(lg.isnan(), want.isnan())
        ok = ~want.isnan()
        assert torch.equal(lg[ok], want[ok])
