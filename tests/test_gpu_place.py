"""Selection and rows in expert order in two launches (csrc/place.hip): the routing it leaves against numpy on the same
logits, at the edges of what it takes, and the rows against a gather."""
import numpy as np
import pytest
import torch

from oracle import moe_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,E,k,H", [
    (65, 4, 1, 8),           # a token past the kernels for few tokens, one piece of a row
    (2047, 8, 2, 136),       # chunks of 8 tokens, the last one short
    (2048, 128, 8, 64),      # ... all full, as many experts as are taken
    (2049, 65, 64, 16),      # chunks of 16; more than a wave of experts, as many a token as are taken
    (4096, 128, 3, 64),      # the largest table, one workgroup a chunk
    (4097, 128, 3, 64),      # one token more: the general path
    (5000, 1, 1, 2056),      # one expert; more than four pieces a lane
    (8001, 31, 5, 24),       # a last word with one count missing
    (300, 8, 2, 12),         # rows that only the fp32 layer takes, which the general path moves
])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_places(pkg, lib, T, E, k, H, dtype):
    print("places", T, E, k, H, dtype, flush=True)
    if H % 8 and dtype == torch.bfloat16:
        pytest.skip("the bf16 layer takes widths that are multiples of 8")
    g = torch.Generator().manual_seed(T)
    logits = torch.randn(T, E, generator=g).round(decimals=1).to(dtype)  # (ties)
    if E > k:
        logits[:: 7, 0] = -float("inf")
        logits[3, E - 1] = float("nan")
    x = torch.randn(T, H, generator=g).to(dtype)
    ws = [(torch.randn(*s, generator=g) * 0.1).to(dtype).cuda() for s in ((E, 8, H), (E, 8, H), (E, H, 8))]
    call = pkg.moe_ffn if dtype == torch.bfloat16 else pkg.moe_ffn_f32
    out, rt = call(x.cuda(), logits.cuda(), *ws, k, return_routing=True)
    ids, _ = O.topk_select(logits.float(), k)
    flat = ids.reshape(-1)
    order = np.argsort(flat, kind="stable")
    assert np.array_equal(rt["ids"].cpu().numpy(), flat.astype(np.int32))
    assert np.array_equal(rt["counts"].cpu().numpy(), np.bincount(flat, minlength=E).astype(np.int32))
    assert np.array_equal(rt["offs"].cpu().numpy(), np.concatenate([[0], np.bincount(flat, minlength=E).cumsum()]).astype(np.int32))
    assert np.array_equal(rt["pos_to_row"].cpu().numpy(), order.astype(np.int32))
    inverse = np.empty_like(order)
    inverse[order] = np.arange(T * k)
    assert np.array_equal(rt["row_to_pos"].cpu().numpy(), inverse.astype(np.int32))
    # the rows: the same call on the general path, which is given the experts (k = 1 there: a row each), summed with the
    # same gates; bf16 rounds the expert's row and the sum (2^-8 each)
    rows = x.cuda().repeat_interleave(k, 0)
    entry = pkg.experts_rows if dtype == torch.bfloat16 else pkg.experts_rows_f32
    y = entry(rows, rt["ids"].long(), *ws).float().view(T, k, H)
    want = (rt["gates"].view(T, k, 1) * y).sum(1)
    rel = 2.0 ** -7 if dtype == torch.bfloat16 else 1e-5
    nan = torch.isnan(want)
    assert torch.equal(nan, torch.isnan(out))
    assert ((out.float() - want)[~nan].abs() <= rel * (want[~nan].abs() + 1e-3)).all()
