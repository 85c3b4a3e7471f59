"""Tiles that a workgroup of the tiled products does one after the other, each handing over to the next one's first k-tiles: odd
and even numbers of k-tiles, one and two of them, ends past the contraction, tiles without rows for half of the waves, empty
experts between others."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def experts(offs):
    o = offs.tolist()
    return [(e, slice(o[e], o[e + 1])) for e in range(len(o) - 1)]


@pytest.mark.parametrize("K", [64, 128, 136, 192, 328])
def test_rows(pkg, lib, K):
    print("rows", K, flush=True)
    ops, g = pkg.ops, torch.Generator(device="cuda").manual_seed(K)
    counts = ([300, 129, 1, 0, 256, 65] * 47)[:280]  # 370 row tiles, two or four column tiles: at least three a workgroup
    E, R, N = len(counts), sum(counts), 512
    offs = torch.tensor([0] + counts).cumsum(0).to(torch.int32).cuda()
    r = lambda *s: torch.randn(*s, generator=g, device="cuda").to(torch.bfloat16)
    x, x2, gate, up, down, dw1, dw3 = r(R, K), r(R, K), r(E, N, K), r(E, N, K), r(E, N, K), r(E, K, N), r(E, K, N)

    def products(height):
        force = ops._lib.load().cdll.moe_gemm_force_row_tile
        try:
            force(height)
            gu, a = ops.gemm_gateup_blocked(x, gate, up, offs)
            d = ops.gemm_dgrad_down_blocked(x2, dw1, gu, offs, dgate_blocks=True)
            return [a, ops.gemm_gateup(x, gate, up, offs, False)[2], ops.gemm_down(x, down, offs), *d,
                    ops.gemm_dgrad_gateup(x, x2, dw1, dw3, offs)]
        finally:
            force(0)

    want = products(64)  # (a kernel of its own, a tile to a workgroup)
    for height in (256, 128):
        for n, (a, b) in enumerate(zip(products(height), want)):
            assert torch.equal(a.view(torch.uint8), b.view(torch.uint8)), (height, n)
    # a rounding to bf16, and sums of K products of unit variance in fp32 on both sides
    ref = torch.cat([x[s].float() @ down[e].float().T for e, s in experts(offs)])
    assert bool(((want[2].float() - ref).abs() <= ref.abs() * 2.0 ** -8 + 2.0 ** -22 * K * K ** 0.5).all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("counts", [
    [64, 65, 0, 1, 128, 129, 0, 0, 200, 63, 256, 300] * 2,  # 0 to 5 k-tiles in every order of odd and even
    [64] * 24,                                              # one each
    [130] * 23 + [1000],
])
@pytest.mark.parametrize("N", [1280, 1000])  # results that leave with streaming stores, and whose rows are not whole pieces of 64 bytes
def test_weight_gradients(pkg, lib, counts, dtype, N):
    print("weight gradients", counts, dtype, N, flush=True)
    ops, g = pkg.ops, torch.Generator(device="cuda").manual_seed(len(counts))
    E, R, M = len(counts), sum(counts), 1016
    offs = torch.tensor([0] + counts).cumsum(0).to(torch.int32).cuda()
    a, b = (torch.randn(R, n, generator=g, device="cuda").to(torch.bfloat16) for n in (M, N))
    got = ops.gemm_wgrad(a, b, offs, E, dtype)
    K = max(counts)
    for e, s in experts(offs):
        ref = a[s].float().T @ b[s].float()
        bound = ref.abs() * (2.0 ** -8 if dtype == torch.bfloat16 else 0) + 2.0 ** -22 * K * K ** 0.5
        assert bool(((got[e].float() - ref).abs() <= bound).all()), (e, counts[e])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("E,H,I", [
    (61, 1024, 88), (65, 1024, 88), (65, 1016, 88),   # small launches: bf16 results of 32.8, 34.9 and 34.6 MB, around the line and rows of no whole pieces
    (24, 2048, 256), (3, 264, 264),                   # ... of 75 and 1.3 MB
    (33, 1024, 1024), (512, 520, 8),                  # tiled ones: 208 and 12.8 MB
])
def test_results_on_both_sides_of_the_streaming_line(pkg, lib, E, H, I, dtype):
    print("weight gradients, streaming", E, H, I, dtype, flush=True)
    g = torch.Generator(device="cuda").manual_seed(E)
    counts = torch.randint(0, 60, (E,), generator=torch.Generator().manual_seed(E))
    ids = torch.arange(E).repeat_interleave(counts).cuda()
    R = len(ids)
    r = lambda *s, std=1.0: (torch.randn(*s, generator=g, device="cuda") * std).to(torch.bfloat16)
    x, dy = r(R, H), r(R, H)
    ws = [w.to(dtype).requires_grad_(True) for w in (r(E, I, H, std=0.05), r(E, I, H, std=0.05), r(E, H, I, std=0.05))]
    pkg.experts_rows(x, ids, *ws).backward(dy)
    both = [w.detach().clone().requires_grad_(True) for w in ws]
    for w in both:  # (added to zeros: ordinary stores)
        w.grad = torch.zeros_like(w)
    pkg.experts_rows(x, ids, *both, accumulate_into_grad=True).backward(dy)
    for n, (a, b) in enumerate(zip(ws, both)):
        assert torch.equal(a.grad, b.grad), n
    one = 7 % E  # one expert's against fp32 products of its rows
    s = ids == one
    xe, de, w1, w3, w2 = x[s].float(), dy[s].float(), *[w.detach()[one].float() for w in ws]
    gate, up = xe @ w1.T, xe @ w3.T
    act = (torch.nn.functional.silu(gate) * up).to(torch.bfloat16).float()
    ref = de.T @ act
    assert (ws[2].grad[one].float() - ref).norm() <= 1e-2 * ref.norm()  # (act and the result each rounded to bf16)
