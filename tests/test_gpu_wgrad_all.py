"""The three weight gradients in one launch of the tiled kernel against the launches that one of them takes by itself: the same tiles,
the same bits, whichever workgroups they are dealt to."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("counts,H,I", [
    ([7, 0, 130, 64] * 32, 1024, 256),            # two and four rounds of tiles, dealt round-robin
    ([1, 300, 0, 65] * 20 + [129] * 3, 1000, 256),  # 83 experts: a first problem that ends within a round
    ([5] * 62 + [900, 0], 2048, 1024),            # dealt longest first, both problems together
    ([33] * 64, 2048, 1024),                      # whole groups an expert, even loads
    ([65, 2, 140, 0] * 32, 2040, 192),            # gate's and up's by themselves: three problems
    ([5] * 31 + [900], 2040, 1000),               # three, longest first
], ids=["rounds", "partial", "skewed", "even", "three", "three skewed"])
def test_one_launch_has_the_bits_of_two(pkg, counts, H, I, dtype):
    print("weight gradients", len(counts), sum(counts), H, I, dtype, flush=True)
    E, R = len(counts), sum(counts)
    g = torch.Generator(device="cuda").manual_seed(R)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda").to(torch.bfloat16)
    x, dy, ws = r(R, H), r(R, H), [w.to(dtype) for w in (r(E, I, H), r(E, I, H), r(E, H, I))]
    ids = torch.arange(E, device="cuda").repeat_interleave(torch.tensor(counts, device="cuda"))
    ids = ids[torch.randperm(R, generator=g, device="cuda")]
    calls = []

    class Obs:
        def before(self, name):
            calls.append(name)

        def after(self, name):
            pass

    lib = pkg.ops._lib.load()

    def grads(wanted):
        leaves = [w.detach().requires_grad_(i in wanted) for i, w in enumerate(ws)]
        out = pkg.experts_rows(x, ids, *leaves)
        lib.observer = Obs()
        try:
            out.backward(dy)
        finally:
            lib.observer = None
        return [w.grad for w in leaves]

    w1, w3, w2 = grads((0, 1, 2))
    assert "moe_gemm_wgrad_all" in calls
    for i, got in enumerate((w1, w3, w2)):
        assert torch.equal(got.view(torch.uint8), grads((i,))[i].view(torch.uint8)), i
    assert calls.count("moe_gemm_wgrad_all") == 1 and calls.count("moe_gemm_wgrad") == 3
