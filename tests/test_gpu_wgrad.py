"""The weight-gradient kernel of small launches (all stacks and the router in one launch, long experts cut into
segments of at least 512 rows): against the oracle where tiles, steps and segments end."""
import pytest
import torch

from _tol import check
from oracle import moe_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,E,k,H,I,shares", [
    (9, 3, 2, 64, 8, None),                          # less than a step, tiles nearly empty
    (700, 5, 1, 264, 136, (0.0, 0.05, 0.1, 0.85, 0.0)),   # one expert cut in two, two without rows
    (2300, 4, 1, 136, 264, (0.9, 0.06, 0.03, 0.01)),      # ... in five
    (1030, 70, 2, 128, 128, None),                   # more experts than lanes in a wave
    (513, 1, 1, 256, 128, None),                     # one expert of one row more than a segment
])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_small_launch_weight_gradients(pkg, lib, T, E, k, H, I, shares, dtype):
    print("weight gradients", T, E, k, H, I, shares, dtype, flush=True)
    g = torch.Generator().manual_seed(T + E)
    r = lambda *s, std=1.0: (torch.randn(*s, generator=g) * std).to(torch.bfloat16)
    x, wr, w1, w3, w2 = r(T, H), r(E, H, std=0.02), r(E, I, H, std=0.08), r(E, I, H, std=0.08), r(E, H, I, std=0.08)
    dy = r(T, H, std=0.1)
    bias = None
    if shares is not None:  # one large feature per expert pins the routing
        wr = torch.zeros_like(wr)
        pick = torch.multinomial(torch.tensor(shares), T, replacement=True, generator=g)
        x[:, :8] = 0
        x[torch.arange(T), pick] = 4.0
        wr[torch.arange(E), torch.arange(E)] = 4.0
    ws = [w.cuda().to(dtype).requires_grad_(True) for w in (wr, w1, w3, w2)]
    xd = x.cuda().requires_grad_(True)
    out, logits = pkg.routed_moe(xd, *ws, k, bias=bias)
    out.backward(dy.cuda())
    lg = logits.detach().cpu()
    f = O.moe_forward(x, wr, w1, w3, w2, k, logits=lg)
    b = O.moe_backward(f, dy.float(), wr, w1, w3, w2)
    fe = O.moe_forward(x, wr, w1, w3, w2, k, logits=lg, emulate_bf16=True)
    be = O.moe_backward(fe, dy.float(), wr, w1, w3, w2, emulate_bf16=True)
    if shares is not None:
        assert f["counts"].max() > 512
    for name, t in (("dw1", ws[1]), ("dw3", ws[2]), ("dw2", ws[3]), ("dx", xd)):
        check(name, t.grad, b[name], be[name])
    if k > 1:  # (with one expert a token its gate is 1 and the router's gradient rounding noise)
        check("dwr", ws[0].grad, b["dwr"], be["dwr"])
    again = [w.detach().clone().requires_grad_(True) for w in ws]
    x2 = xd.detach().clone().requires_grad_(True)
    for _ in range(2):  # added to .grad by the kernel: twice the first gradient, to the rounding of the sum
        pkg.routed_moe(x2, *again, k, accumulate_into_grad=True)[0].backward(dy.cuda())
    for w, a in zip(ws[1:], again[1:]):
        assert torch.allclose(a.grad.float(), 2 * w.grad.float(), rtol=2e-2 if dtype == torch.bfloat16 else 1e-5,
                              atol=1e-6 * float(w.grad.abs().max()))


@pytest.mark.parametrize("H,I", [(128, 128), (136, 264)])
def test_steps_and_stages(pkg, lib, H, I):
    """Experts that end at and around every step (32 rows) of the ring of three stages, and one without rows: one
    launch without and one with a second column tile."""
    print("steps and stages", H, I, flush=True)
    counts = [1, 31, 32, 33, 0, 63, 64, 65, 95, 96, 97, 128, 129]
    g = torch.Generator().manual_seed(H)
    E = len(counts)
    ids = torch.repeat_interleave(torch.arange(E), torch.tensor(counts))
    ids = ids[torch.randperm(len(ids), generator=g)]
    r = lambda *s, std=1.0: (torch.randn(*s, generator=g) * std).to(torch.bfloat16)
    x, w1, w3, w2 = r(len(ids), H), r(E, I, H, std=0.08), r(E, I, H, std=0.08), r(E, H, I, std=0.08)
    dy = r(len(ids), H, std=0.1)
    ws = [w.cuda().requires_grad_(True) for w in (w1, w3, w2)]
    pkg.experts_rows(x.cuda(), ids.cuda(), *ws).backward(dy.cuda())
    b, be = (O.experts_rows_backward(O.experts_rows_forward(x, ids.numpy(), w1, w3, w2, emulate_bf16=e), dy.float(), w1, w3,
                                     w2, emulate_bf16=e) for e in (False, True))
    for name, w in zip(("dw1", "dw3", "dw2"), ws):
        check(name, w.grad, b[name], be[name])
        assert not w.grad[counts.index(0)].any()


@pytest.mark.parametrize("T,E,k,H,I", [
    (1100, 70, 2, 520, 264),   # 420 tiles of 256 x 256, six rounds against 4.1 of small tiles: taken
    (600, 65, 2, 512, 512),    # 260, five rounds (two of the launches one) against 4.1: taken
    (300, 66, 1, 512, 1024),   # 528, eight rounds against 8.25: not taken
])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_weight_gradients_past_a_round_of_tiles(pkg, lib, T, E, k, H, I, dtype):
    test_small_launch_weight_gradients(pkg, lib, T, E, k, H, I, None, dtype)
