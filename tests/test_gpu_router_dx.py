"""The router's backward inside the pass that sums up the input gradient, against the kernel of its own that runs where no input
gradient is wanted: the same rows of dlogits, so the same bits of the router weight's gradient."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,E,k,H,I", [
    (1, 2, 2, 8, 8),
    (5, 3, 3, 64, 136),         # rows of dlogits padded, 4 blocks
    (67, 130, 9, 72, 264),      # more experts than lanes, 8 blocks
    (33, 512, 64, 520, 520),    # a slot for every lane, 12 blocks
    (300, 64, 8, 1032, 1064),   # 20 blocks
    (1100, 8, 1, 256, 128),     # (one expert a token: no gradient but rounding)
])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_router_gradient_with_and_without_dx(pkg, lib, T, E, k, H, I, dtype):
    print("router and dx", T, E, k, H, I, dtype, flush=True)
    g = torch.Generator(device="cuda").manual_seed(T)
    r = lambda *s, std=0.05: (torch.randn(*s, generator=g, device="cuda") * std).to(dtype)
    x, dy, ws = r(T, H, std=1.0), r(T, H, std=1.0), [r(E, H), r(E, I, H), r(E, I, H), r(E, H, I)]
    got = []
    for with_x in (False, True):
        w = [t.clone().requires_grad_(True) for t in ws]
        pkg.routed_moe(x.clone().requires_grad_(with_x), *w, k)[0].backward(dy)
        got.append([t.grad for t in w])
    for a, b in zip(*got):
        assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))
