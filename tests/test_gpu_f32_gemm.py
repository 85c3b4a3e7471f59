"""The fused fp32 products (gate/up with SwiGLU, down backward with SwiGLU's, the two-operand input gradient,
the three weight gradients of one launch) against fp64: where tiles and their quarters end."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("counts,H,I", [
    ([1, 0, 33], 4, 4),                                # the smallest widths, quarters nearly empty
    ([65, 0, 130, 31, 97], 100, 36),                   # ragged everything, fewer tiles than compute units
    ([300, 7, 0, 513, 64, 1, 0, 200] * 9, 132, 260),   # more experts than lanes in a wave, a cut last round
    ([700, 650, 500], 1028, 132),
])
@pytest.mark.parametrize("tile", [0, 64, 128])
def test_fused_f32_products(pkg, lib, counts, H, I, tile):
    print("fused fp32 products", len(counts), sum(counts), H, I, tile, flush=True)
    g = torch.Generator().manual_seed(sum(counts) + H)
    E, R = len(counts), sum(counts)
    offs = torch.tensor(np.concatenate([[0], np.cumsum(counts)]), dtype=torch.int32)
    r = lambda *s: torch.randn(*s, generator=g) * 0.3
    xp, dyp, w1, w3, w2 = r(R, H), r(R, H), r(E, I, H), r(E, I, H), r(E, H, I)
    per = lambda f: torch.cat([f(e, slice(int(offs[e]), int(offs[e + 1]))) for e in range(E)])
    G = per(lambda e, s: xp[s].double() @ w1[e].double().t())
    U = per(lambda e, s: xp[s].double() @ w3[e].double().t())
    A = torch.nn.functional.silu(G) * U
    D = per(lambda e, s: dyp[s].double() @ w2[e].double())
    sg = torch.sigmoid(G)
    dG, dU = D * U * (sg * (1 + G * (1 - sg))), D * G * sg
    dX = per(lambda e, s: dG[s] @ w1[e].double() + dU[s] @ w3[e].double())
    t = lambda a, b: torch.stack([a[offs[e]:offs[e + 1]].t() @ b[offs[e]:offs[e + 1]] for e in range(E)])
    ops = pkg.ops
    cu = [v.cuda() for v in (xp, dyp, w1, w3, w2, offs)]
    x_, dy_, w1_, w3_, w2_, o_ = cu
    before = pkg.lib.load().cdll.moe_f32_gemm_force_tile(tile)
    try:
        g_, u_, a_ = ops.f32_gateup_swiglu(x_, w1_, w3_, o_)
        dg_, du_ = ops.f32_down_swiglu_bwd(dy_, w2_, g_, u_, o_)
        dx_ = ops.f32_gateup_bwd(dg_, du_, w1_, w3_, o_)
        dw = ops.f32_wgrads(dg_, du_, dy_, x_, a_, o_)
    finally:
        pkg.lib.load().cdll.moe_f32_gemm_force_tile(before)
    xd, dyd = xp.double(), dyp.double()
    refs = dict(g=(g_, G), u=(u_, U), act=(a_, A), dg=(dg_, dG), du=(du_, dU), dx=(dx_, dX), dw1=(dw[0], t(dG, xd)),
                dw3=(dw[1], t(dU, xd)), dw2=(dw[2], t(dyd, A)))
    for name, (got, ref) in refs.items():
        rel = ((got.cpu().double() - ref).norm() / ref.norm()).item()
        print("  ", name, rel, flush=True)
        assert rel <= 1e-5, name
