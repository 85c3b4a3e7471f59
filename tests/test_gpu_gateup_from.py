"""A forward without gradients reads the tokens' rows where they are.  The separate steps copy them into expert order first: the same
bits, whichever tiles the product takes."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,H,E,I,k", [
    (65, 8, 4, 8, 1),            # a k-tile with one piece of eight
    (65, 72, 5, 24, 5),          # every expert for every token
    (129, 264, 128, 136, 8),     # a few rows an expert
    (1000, 1416, 12, 568, 3),    # k-tiles and columns that end in the middle
    (2048, 512, 8, 192, 2),
    (1531, 2048, 6, 256, 4),     # whole tiles, and what is left in quarters; starts at different k-tiles
    (4321, 640, 130, 328, 6),    # past the sizes that have a table of counts
])
def test_rows_from_the_tokens(pkg, T, H, E, I, k):
    ops, cdll = pkg.ops, pkg.ops._lib.load().cdll
    force, workspace = cdll.moe_gemm_force_row_tile, cdll.moe_ffn_forward_workspace_bytes
    g = torch.Generator(device="cuda").manual_seed(T + H)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda").to(torch.bfloat16)
    x, logits, w1, w3, w2 = r(T, H), r(T, E), r(E, I, H), r(E, I, H), r(E, H, I)
    logits[:, E // 2] -= 20.0  # (an expert without rows, or with a few)
    ids, gates = ops.router_topk(logits, k)
    _, offs, pos_to_row, row_to_pos = ops.histogram_scan(ids, E)[:4]
    act = ops.gemm_gateup(ops.permute_fwd(x, pos_to_row, k), w1, w3, offs, False)[-1]
    want = ops.combine_fwd(ops.gemm_down(act, w2, offs), gates, row_to_pos, T, k, torch.bfloat16)
    for height in (0, 1, 64, 128, 256):
        print("rows from the tokens", T, H, E, I, k, height, flush=True)
        torch.cuda.reset_peak_memory_stats()
        before = torch.cuda.memory_stats()["requested_bytes.all.current"]
        try:
            force(height)
            with torch.no_grad():
                out = pkg.moe_ffn(x, logits, w1, w3, w2, k)
        finally:
            force(0)
        held = torch.cuda.memory_stats()["requested_bytes.all.peak"] - before
        assert torch.equal(out, want), height
        # (no room for copies, of which the documented workspace has some; parts of it begin at multiples of 256 bytes)
        assert held <= workspace(T, H, E, I, k) - T * k * H * 2 + out.numel() * 2 + 256, held
