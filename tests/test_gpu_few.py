"""The kernels for few tokens (a forward without gradients of at most 64): against the oracle at the edges
of their blocks of 16 rows, 16 columns and 32-deep steps, and at the ends of their range."""
import pytest
import torch

from _tol import check
from oracle import moe_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,E,k,H,I,x_dt", [
    (1, 64, 8, 256, 136, torch.bfloat16),    # one token: the kernel that also combines
    (1, 4, 3, 2056, 1032, torch.float32),    # ... contractions that end inside a step, experts' shares split
    (1, 8, 2, 4104, 72, torch.bfloat16),     # ... that many columns that a workgroup takes 16
    (1, 8, 3, 4096, 2120, torch.float32),    # ... and several requests for each share
    (1, 16, 8, 2040, 2120, torch.bfloat16),  # ... 8
    (1, 40, 33, 64, 64, torch.bfloat16),     # ... more experts a token than that kernel takes
    (1, 128, 8, 264, 520, torch.bfloat16),   # ... selected from two logits a lane
    (1, 65, 32, 72, 136, torch.float32),     # ... the most experts a token that the combining kernel takes
    (1, 130, 8, 264, 24, torch.bfloat16),    # ... selected by the router kernel
    (2, 128, 1, 520, 8, torch.float32),
    (16, 4, 4, 136, 248, torch.bfloat16),    # every expert has 16 rows
    (17, 4, 4, 136, 248, torch.bfloat16),    # ... 17
    (33, 3, 3, 1032, 72, torch.float32),     # ... 33
    (64, 2, 2, 4104, 40, torch.bfloat16),    # ... 64; shares of the contraction too long for registers
    (48, 130, 8, 264, 520, torch.bfloat16),  # more experts than the router kernel takes
])
def test_forward_of_few_tokens_matches_the_oracle(pkg, lib, T, E, k, H, I, x_dt):
    print("few tokens", T, E, k, H, I, x_dt, flush=True)
    g = torch.Generator().manual_seed(T * 1000 + E)
    r = lambda *s, std=1.0: (torch.randn(*s, generator=g) * std).to(torch.bfloat16)
    x, wr, w1, w3, w2 = r(T, H), r(E, H, std=0.3), r(E, I, H, std=0.05), r(E, I, H, std=0.05), r(E, H, I, std=0.05)
    xd = x.cuda().to(x_dt)
    ws = [w.cuda() for w in (w1, w3, w2)]
    bias = torch.randn(E, generator=g) if T % 2 else None
    with torch.no_grad():
        out, logits = pkg.routed_moe(xd, wr.cuda(), *ws, k, bias=None if bias is None else bias.cuda())
        given = pkg.moe_ffn(xd, logits, *ws, k, bias=None if bias is None else bias.cuda())
    assert out.dtype == x_dt and torch.equal(out, given)
    lg = logits.cpu()
    check("logits", lg, x.float() @ wr.float().t(), (x.float() @ wr.float().t()).bfloat16().float())
    sel = lg.float() + bias if bias is not None else lg
    f = O.moe_forward(x, wr, w1, w3, w2, k, logits=sel)
    fe = O.moe_forward(x, wr, w1, w3, w2, k, logits=sel, emulate_bf16=True)
    check("out", out, f["out"], fe["out"])


@pytest.mark.parametrize("E,H,I,x_dt,few", [  # 64 tokens, every expert asked for by each
    (9, 1032, 792, torch.bfloat16, True), (9, 1032, 808, torch.bfloat16, False),  # 2.47 and 2.52 GB past 8 rows each
    (9, 1032, 400, torch.float32, True), (9, 1032, 408, torch.float32, False),    # ... of fp32 rows
    (8, 1368, 1352, torch.bfloat16, True), (8, 1368, 1360, torch.bfloat16, False),  # 4.97 and 5.0009, at most 8 experts
])
def test_many_rows_an_expert_take_the_tiled_kernels(pkg, lib, E, H, I, x_dt, few):
    print("few or tiled", E, H, I, x_dt, flush=True)
    g = torch.Generator().manual_seed(H + I)
    r = lambda *s, std=0.05: (torch.randn(*s, generator=g) * std).to(torch.bfloat16)
    x, wr, w1, w3, w2, lg = r(64, H, std=1.0), r(E, H), r(E, I, H), r(E, I, H), r(E, H, I), r(64, E, std=1.0)
    names = []

    class Obs:
        before = names.append
        after = staticmethod(lambda name: None)

    lib.observer = Obs()
    try:
        with torch.no_grad():
            out = pkg.moe_ffn(x.cuda().to(x_dt), lg.cuda(), w1.cuda(), w3.cuda(), w2.cuda(), E)
    finally:
        lib.observer = None
    assert ("moe_gateup_few" in names, "moe_gemm_gateup_swiglu_fwd" in names) == (few, not few), names
    f = O.moe_forward(x, wr, w1, w3, w2, E, logits=lg)
    check("out", out, f["out"], O.moe_forward(x, wr, w1, w3, w2, E, logits=lg, emulate_bf16=True)["out"])


@pytest.mark.parametrize("H", [2048, 4104])  # columns in workgroups of 8 and of 16
@pytest.mark.parametrize("k,I", [(1, 264), (2, 72), (3, 1032), (8, 72)])
def test_one_infinite_activation_makes_infinite_outputs(pkg, lib, H, k, I):
    """One token, an activation that overflows: every output is infinite, none a NaN, wherever in its expert's
    contraction that activation lies (in workgroups' shares other than its own it must not be there at all)."""
    print("infinite activation", H, k, I, flush=True)
    E = 2 * k
    w1, w3, w2 = torch.zeros(E, I, H), torch.zeros(E, I, H), torch.full((E, H, I), 0.5)
    x = torch.zeros(1, H)
    x[0, 0] = 1.0
    logits = torch.arange(E, 0, -1).float()[None].cuda()  # experts 0 .. k-1
    bf = torch.bfloat16
    for i in sorted({0, 31, I // 2, I - 1}):
        w1[:, :, 0] = w3[:, :, 0] = 1e-3
        w1[k - 1, i, 0] = w3[k - 1, i, 0] = 1e30
        with torch.no_grad():
            out = pkg.moe_ffn(x.cuda().to(bf), logits, *(w.cuda().to(bf) for w in (w1, w3, w2)), k)
        assert torch.isposinf(out).all(), (i, out.isnan().sum().item(), out.isfinite().sum().item())


@pytest.mark.parametrize("T,E,k,H,I,x_dt,given", [
    (2, 1, 1, 8, 8, torch.bfloat16, torch.bfloat16),       # one expert, all of both tokens
    (5, 65, 7, 40, 24, torch.float32, torch.float32),      # one expert more than lanes in a wave; logits in fp32
    (64, 4, 3, 136, 120, torch.bfloat16, torch.float32),   # more tokens than workgroups; more rows than 32 an expert
    (33, 16, 16, 72, 40, torch.float32, torch.bfloat16),   # every token asks for every expert
    (13, 128, 2, 264, 56, torch.bfloat16, torch.bfloat16),  # turns of four tokens and one, the most experts (2048 turns)
    (17, 128, 2, 264, 56, torch.bfloat16, torch.bfloat16),  # ... past them: the launch of its own
])
def test_selection_inside_gate_up(pkg, lib, T, E, k, H, I, x_dt, given):
    """Which rows an expert has, from the logits themselves: ties, a bias, infinities and a NaN, as the selection's own launch
    (which the oracle stands for) decides them."""
    print("selection inside gate/up", T, E, k, H, I, x_dt, given, flush=True)
    g = torch.Generator().manual_seed(T + E)
    r = lambda *s, std=1.0: (torch.randn(*s, generator=g) * std).to(torch.bfloat16)
    x, w1, w3, w2 = r(T, H), r(E, I, H, std=0.05), r(E, I, H, std=0.05), r(E, H, I, std=0.05)
    lg = torch.randn(T, E, generator=g).round(decimals=1).to(given)
    if E > k:
        lg[1, 0] = -float("inf")
    bias = torch.randn(E, generator=g).round(decimals=1) if T % 2 else None
    sel = lg.float() + bias if bias is not None else lg.float()
    f = O.moe_forward(x, torch.zeros(E, H), w1, w3, w2, k, logits=sel)
    fe = O.moe_forward(x, torch.zeros(E, H), w1, w3, w2, k, logits=sel, emulate_bf16=True)
    ws = [w.cuda() for w in (w1, w3, w2)]
    call = lambda logits: pkg.moe_ffn(x.cuda().to(x_dt), logits.cuda(), *ws, k, bias=None if bias is None else bias.cuda())
    out = call(lg)
    check("out", out, f["out"], fe["out"])
    lg[0, E - 1] = float("nan")  # (its expert comes first and its token's gates are NaN; the others stay as they are)
    bad = call(lg)
    assert bad[0].isnan().all() and torch.equal(bad[1:], out[1:])
