"""The row-ragged products in tiles of 128 rows of the ring, by themselves (forced) and where the library takes them, against tiles
of 256 rows: the same bits, also where one writes g and u and another reads them."""
import pytest
import torch

pytestmark = pytest.mark.gpu
TALL = 1


@pytest.mark.parametrize("counts,H,I", [
    ([513, 511, 0, 897, 1, 640, 384, 1150], 616, 520),    # gate/up: edges of a tile and of a wave's rows, k and columns off the tiles
    ([513, 511, 0, 897, 33, 607, 384, 1151], 520, 1000),  # dgrad-down too; columns past the last, for which sums are due
    ([1700, 1701, 1663, 1729], 264, 1032),                # two rounds of a short contraction
    ([70] * 90 + [0, 127, 128, 129, 1, 65], 256, 328),    # many experts, one tile each
    ([4096], 8, 2048),                                    # less than a k-tile
    ([1, 31, 33, 0, 63, 65, 127, 129, 159, 161, 191, 193, 255], 200, 136),  # what is left of a tile, a wave's rows and a strip
])
def test_tall_ring_tiles(pkg, lib, counts, H, I):
    print("tall ring tiles", len(counts), sum(counts), H, I, flush=True)
    ops = pkg.ops
    force = ops._lib.load().cdll.moe_gemm_force_row_tile
    g = torch.Generator(device="cuda").manual_seed(H + I)
    E, R = len(counts), sum(counts)
    offs = torch.tensor([0] + counts).cumsum(0).to(torch.int32).cuda()
    r = lambda *s: torch.randn(*s, generator=g, device="cuda").to(torch.bfloat16)
    xp, dy, w1, w3, w2 = r(R, H), r(R, H), r(E, I, H), r(E, I, H), r(E, H, I)
    act, dg, du = r(R, I), r(R, I), r(R, I)

    def products(fwd, bwd):
        try:
            force(fwd)
            gu, a = ops.gemm_gateup_blocked(xp, w1, w3, offs)
            force(bwd)
            return [a, ops.gemm_down(act, w2, offs), ops.gemm_dgrad_gateup(dg, du, w1, w3, offs),
                    *ops.gemm_dgrad_down_blocked(dy, w2, gu, offs, dgate_blocks=True),
                    *ops.gemm_dgrad_down_blocked(dy, w2, gu, offs, dgate_blocks=True, packed=True)]
        finally:
            force(0)

    want = products(256, 256)
    for tiles in ((TALL, TALL), (TALL, 256), (256, TALL), (0, 0), (0, 256), (256, 0)):
        for n, (a, b) in enumerate(zip(products(*tiles), want)):
            assert torch.equal(a.contiguous().view(torch.uint8), b.contiguous().view(torch.uint8)), (tiles, n)
