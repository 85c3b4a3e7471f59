"""Where the tiled products find their tiles' experts, rows and columns: up to, at and past whole waves of experts, runs of
experts without rows, one to seven column tiles."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("E", [1, 63, 64, 65, 127, 128, 129, 193, 1024])
@pytest.mark.parametrize("N", [256, 648, 1792])
def test_every_tile_of_every_expert(pkg, lib, E, N):
    print("tiles", E, N, flush=True)
    ops, K = pkg.ops, 64
    g = torch.Generator(device="cuda").manual_seed(E + N)
    counts = [(0, 300, 0, 0, 1, 256, 129)[e % 7] for e in range(1, E + 1)]
    counts[-1] += 77
    offs = torch.tensor([0] + counts).cumsum(0).to(torch.int32).cuda()
    R = sum(counts)
    x, w = (torch.randn(*s, generator=g, device="cuda").to(torch.bfloat16) for s in ((R, K), (E, N, K)))
    force = ops._lib.load().cdll.moe_gemm_force_row_tile
    o = offs.tolist()
    ref = torch.cat([x[o[e]:o[e + 1]].float() @ w[e].float().T for e in range(E)])
    for height in (256, 128):
        try:
            force(height)
            got = ops.gemm_down(x, w, offs).float()
        finally:
            force(0)
        # a rounding to bf16, and sums of K products of unit variance in fp32 on both sides
        assert bool(((got - ref).abs() <= ref.abs() * 2.0 ** -8 + 2.0 ** -22 * K * K ** 0.5).all()), height


@pytest.mark.parametrize("M,N", [(256, 264), (1288, 256), (520, 1792)])
def test_every_tile_of_every_weight_gradient(pkg, lib, M, N):
    print("weight gradients", M, N, flush=True)
    ops, E = pkg.ops, 67
    g = torch.Generator(device="cuda").manual_seed(M + N)
    counts = [(0, 70, 1, 0, 33)[e % 5] for e in range(E)]
    offs = torch.tensor([0] + counts).cumsum(0).to(torch.int32).cuda()
    a, b = (torch.randn(sum(counts), n, generator=g, device="cuda").to(torch.bfloat16) for n in (M, N))
    got = ops.gemm_wgrad(a, b, offs, E, torch.float32)
    o = offs.tolist()
    for e in range(E):
        ref = a[o[e]:o[e + 1]].float().T @ b[o[e]:o[e + 1]].float()
        assert bool(((got[e] - ref).abs() <= 2.0 ** -22 * 70 * 70 ** 0.5).all()), e
