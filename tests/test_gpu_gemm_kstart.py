"""Gate/up and down with weight rows of a multiple of 4 KB, whose experts start their contraction at different k-tiles and
go round: every k counts once, whichever expert, the first and the last k-tile included."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K", [2048, 4096])
@pytest.mark.parametrize("rows", [128, 256])
def test_every_k_counts_once(pkg, lib, K, rows):
    print("k start", K, rows, flush=True)
    ops = pkg.ops
    E, N = 33, 40  # (every start the rule has, and the first again)
    counts = [1 + 9 * (e % 3) for e in range(E)]
    R = sum(counts)
    offs = torch.tensor([0] + counts).cumsum(0).to(torch.int32).cuda()
    eid = torch.repeat_interleave(torch.arange(E), torch.tensor(counts)).cuda()
    g = torch.Generator(device="cuda").manual_seed(K)
    # whole numbers small enough that every sum of K products is exact in fp32 in any order
    a = torch.randint(-2, 3, (R, K), generator=g, device="cuda").to(torch.bfloat16)
    w = torch.randint(-2, 3, (2, E, N, K), generator=g, device="cuda").to(torch.bfloat16)
    ops._lib.load().cdll.moe_gemm_force_row_tile(rows)
    try:
        gg, uu, _ = ops.gemm_gateup(a, w[0].contiguous(), w[1].contiguous(), offs, save_gu=True)
        y = ops.gemm_down(a, w[0].contiguous(), offs)
    finally:
        ops._lib.load().cdll.moe_gemm_force_row_tile(0)
    for got, m in ((gg, 0), (uu, 1), (y, 0)):
        want = torch.stack([w[m, e].float() @ a[r].float() for r, e in enumerate(eid.tolist())])
        assert torch.equal(got, want.to(torch.bfloat16))
