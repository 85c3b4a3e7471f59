"""Rows whose experts are given: in bf16 the products leave them where they came from.  In fp32 the results are the same bf16 rows,
put in place by a pass of their own, so that both have the same values, whichever tiles the products take."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("counts,H,I", [
    ([1], 8, 8),
    ([0, 31, 33, 0, 65, 129], 200, 136),         # edges of a wave's rows and of a tile
    ([64, 128, 256, 0, 255, 257], 1000, 320),
    ([513, 511, 0, 900, 1, 640, 384, 513], 1000, 520),
    ([8193], 2048, 1016),                        # whole tiles and what is left of them
    ([8200, 0, 70, 190], 1992, 1032),
])
def test_rows_go_where_they_came_from(pkg, counts, H, I):
    force = pkg.ops._lib.load().cdll.moe_gemm_force_row_tile
    E, R = len(counts), sum(counts)
    g = torch.Generator(device="cuda").manual_seed(R)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda").to(torch.bfloat16)
    x, dy, ws = r(R, H), r(R, H), [r(E, I, H), r(E, I, H), r(E, H, I)]
    ids = torch.arange(E, device="cuda").repeat_interleave(torch.tensor(counts, device="cuda"))
    ids = ids[torch.randperm(R, generator=g, device="cuda")]

    def passed(dtype, height):
        print("rows in place", counts, H, I, dtype, height, flush=True)
        leaf = x.to(dtype, copy=True).requires_grad_(True)
        try:
            force(height)
            out = pkg.experts_rows(leaf, ids, *ws)
            out.backward(dy.to(dtype))
        finally:
            force(0)
        return out.detach().bfloat16(), leaf.grad.bfloat16()

    want = passed(torch.float32, 0)
    for height in (0, 1, 64, 128, 256):
        for a, b in zip(passed(torch.bfloat16, height), want):
            assert torch.equal(a, b), height


def test_no_room_is_held_for_rows_that_stay_in_place(pkg, lib):
    """Besides the results a direction holds one buffer of the size of the rows: those by expert, and the output's gradient by expert."""
    print("rows in place, memory", flush=True)
    R, E, H, I = 8192, 4, 2048, 8
    r = lambda *s: torch.randn(*s, device="cuda").to(torch.bfloat16)
    x, dy, ws, ids = r(R, H).requires_grad_(True), r(R, H), [r(E, I, H), r(E, I, H), r(E, H, I)], torch.randint(0, E, (R,), device="cuda")
    rows = R * H * 2

    def held(call):
        torch.cuda.synchronize()
        torch.cuda.reset_peak_memory_stats()
        before = torch.cuda.memory_allocated()
        result = call()
        return result, torch.cuda.max_memory_allocated() - before

    out, forward = held(lambda: pkg.experts_rows(x, ids, *ws))
    _, backward = held(lambda: out.backward(dy))
    assert forward < 2.5 * rows and backward < 2.5 * rows, (forward / rows, backward / rows)
