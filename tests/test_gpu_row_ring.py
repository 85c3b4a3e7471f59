"""The row-ragged products in tiles of 64 rows against the larger ones: every output element is the sum over k in the
same order, so that the bits are the same, rows and columns of partial tiles, experts without rows and the blocks of the
gates' gradient included."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("counts,H,I", [
    ([64, 64, 64, 64], 256, 128),                  # whole tiles
    ([1], 8, 8),                                   # the smallest widths, less than a k-tile
    ([0, 31, 32, 33, 0, 63, 65, 129], 200, 136),   # edges of a wave's rows and of a tile; k and columns off the tiles
    ([5, 0, 70] * 21 + [9], 2048, 320),            # 64 experts; a contraction that starts at another k-tile
    ([3] * 64 + [100], 72, 264),                   # 65
    ([2, 0, 7, 1] * 32, 128, 64),                  # 128, columns of half a tile
    ([300, 2, 900], 1000, 512),                    # more row tiles than an XCD's share
    ([513, 511, 0, 900, 1, 640, 384, 513], 1000, 520),   # down and dgrad-gate/up in tiles of 128 rows by themselves
    # more small tiles than run at once: taken for down, dgrad-down and dgrad-gate/up; for down (dgrad-down has fewer) alone
    ([50] * 46 + [70, 64], 1536, 640),
    ([24] * 16, 4096, 2048),
    # a little more than a round of tiles of 256 rows (gate/up and dgrad-gate/up, then dgrad-down): the rest in quarters (in
    # dgrad-down in halves)
    ([8193], 2048, 1016),
    ([8200, 0, 70, 190], 1992, 1032),
    ([4100, 4300], 520, 2048),
], ids=["whole", "least", "edges", "64", "65", "128", "long", "tall", "by rounds", "whole rounds", "quarter of one row", "quarters", "quarters down"])
def test_row_ring_bits(pkg, lib, counts, H, I):
    print("row ring", len(counts), sum(counts), H, I, flush=True)
    ops = pkg.ops
    force = ops._lib.load().cdll.moe_gemm_force_row_tile
    g = torch.Generator(device="cuda").manual_seed(H + I)
    E, R = len(counts), sum(counts)
    offs = torch.tensor([0] + counts).cumsum(0).to(torch.int32).cuda()
    r = lambda *s: torch.randn(*s, generator=g, device="cuda").to(torch.bfloat16)
    xp, act, dg, du, dy = r(R, H), r(R, I), r(R, I), r(R, I), r(R, H)
    w1, w3, w2 = r(E, I, H), r(E, I, H), r(E, H, I)

    def products(fwd, bwd):
        try:
            force(fwd)
            gu, a = ops.gemm_gateup_blocked(xp, w1, w3, offs)
            y = ops.gemm_down(act, w2, offs)
            force(bwd)
            return [a, y, *ops.gemm_dgrad_down_blocked(dy, w2, gu, offs, dgate_blocks=True),
                    *ops.gemm_dgrad_down_blocked(dy, w2, gu, offs, dgate_blocks=True, packed=True),
                    ops.gemm_dgrad_gateup(dg, du, w1, w3, offs)]
        finally:
            force(0)

    want = products(256, 256)
    for heights in ((64, 64), (64, 256), (256, 64), (0, 0)):
        for n, (a, b) in enumerate(zip(products(*heights), want)):
            assert torch.equal(a.contiguous().view(torch.uint8), b.contiguous().view(torch.uint8)), (heights, n)
