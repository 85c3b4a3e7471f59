"""The row-ragged products where whole tiles, half tiles and a mixture of them are taken: the same bits whichever it is,
and the products in fp32."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("counts,H,I", [
    ([4000, 4200, 300], 1024, 1024),     # a little more than a round of whole tiles: what is left in halves
    ([612] * 12, 1024, 1024),            # ... the round before too (most experts end in a short tile)
    ([612] * 11 + [0, 1], 1000, 1016),   # ... with tiles that end past the columns
    ([5120, 5120, 5120], 1024, 1024),    # what is left too much for halves
    ([100] * 40, 512, 1024),             # every tile short
    ([0, 129, 0, 5000], 2048, 256),      # less than a round, experts without rows
    ([1] * 70 + [0] * 60, 512, 512),     # more experts than lanes in a wave
])
def test_tile_heights(pkg, lib, counts, H, I):
    print("tile heights", len(counts), sum(counts), H, I, flush=True)
    ops = pkg.ops
    g = torch.Generator(device="cuda").manual_seed(H + I)
    E, R = len(counts), sum(counts)
    offs = torch.tensor([0] + counts).cumsum(0).to(torch.int32).cuda()
    r = lambda *s: torch.randn(*s, generator=g, device="cuda").to(torch.bfloat16)
    xp, act, dg, du, dy = r(R, H), r(R, I), r(R, I), r(R, I), r(R, H)
    w1, w3, w2 = r(E, I, H), r(E, I, H), r(E, H, I)

    def products(fwd, bwd):
        force = ops._lib.load().cdll.moe_gemm_force_row_tile
        try:
            force(fwd)
            gu, a = ops.gemm_gateup_blocked(xp, w1, w3, offs)
            y = ops.gemm_down(act, w2, offs)
            force(bwd)  # (the blocked g and u do not depend on the tiles that wrote them)
            d = ops.gemm_dgrad_down_blocked(dy, w2, gu, offs, dgate_blocks=True)
            return [a, y, *d, ops.gemm_dgrad_gateup(dg, du, w1, w3, offs)]
        finally:
            force(0)

    want = products(256, 256)
    for heights in ((0, 0), (128, 0), (0, 256), (128, 128)):
        for n, (a, b) in enumerate(zip(products(*heights), want)):
            assert torch.equal(a.view(torch.uint8), b.view(torch.uint8)), (heights, n)
    starts = offs.tolist()
    ref = torch.cat([act[starts[e]:starts[e + 1]].float() @ w2[e].float().T for e in range(E)])
    # a rounding to bf16, and sums of I products of unit variance in fp32 on both sides
    err = (want[1].float() - ref).abs()
    assert bool((err <= ref.abs() * 2.0 ** -8 + 2.0 ** -22 * I * I ** 0.5).all())
