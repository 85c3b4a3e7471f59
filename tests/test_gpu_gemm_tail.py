"""The row-ragged products where the contraction length is no multiple of a k-tile (64): its last k-tile holds the
start of the operands' next rows, which must not count.  One, two and several k-tiles, an odd and an even number of
them, both segments of the gate/up input gradient; against the products in fp32."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,I", [(8, 72), (72, 136), (136, 200), (200, 264), (328, 392), (456, 8), (520, 584),
                                 (1416, 568)])
@pytest.mark.parametrize("rows", [128, 256])
def test_contraction_tails(pkg, lib, H, I, rows):
    print("contraction tails", H, I, rows, flush=True)
    ops = pkg.ops
    g = torch.Generator().manual_seed(H + I)
    counts = [130, 0, 300, 1]
    E, R = len(counts), sum(counts)
    offs = torch.tensor([0] + counts).cumsum(0).to(torch.int32).cuda()
    r = lambda *s: torch.randn(*s, generator=g).to(torch.bfloat16).cuda()
    xp, act, dg, du = r(R, H), r(R, I), r(R, I), r(R, I)
    w1, w3, w2 = r(E, I, H), r(E, I, H), r(E, H, I)
    starts = offs.tolist()

    def per_expert(f):
        return torch.cat([f(e, slice(starts[e], starts[e + 1])) for e in range(E) if counts[e]]).double()

    d = lambda t: t.double()
    ops._lib.load().cdll.moe_gemm_force_row_tile(rows)
    try:
        y, dxp = ops.gemm_down(act, w2, offs), ops.gemm_dgrad_gateup(dg, du, w1, w3, offs)
        gg, uu, _ = ops.gemm_gateup(xp, w1, w3, offs, save_gu=True)
    finally:
        ops._lib.load().cdll.moe_gemm_force_row_tile(0)
    want = {
        "y": (y, per_expert(lambda e, s: d(act[s]) @ d(w2[e]).T)),
        "dxp": (dxp, per_expert(lambda e, s: d(dg[s]) @ d(w1[e]) + d(du[s]) @ d(w3[e]))),
        "g": (gg, per_expert(lambda e, s: d(xp[s]) @ d(w1[e]).T)),
        "u": (uu, per_expert(lambda e, s: d(xp[s]) @ d(w3[e]).T)),
    }
    for name, (got, ref) in want.items():
        # one rounding to bf16 (half of 2^-8 of the value) and fp32 sums of K products of unit
        # variance: K roundings of 2^-24 of partial sums around sqrt(K)
        err = (got.double() - ref).abs()
        K = {"y": I, "dxp": 2 * I}.get(name, H)
        bound = ref.abs() * 2.0 ** -8 + 2.0 ** -23 * K * K ** 0.5
        assert bool((err <= bound).all()), (name, float((err - bound).max()))
