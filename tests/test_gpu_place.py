"""Selection and rows in expert order in two launches (csrc/place.hip): the routing it leaves against numpy on the same
logits, at the edges of what it takes, and the rows against a gather."""
import numpy as np
import pytest
import torch

from oracle import moe_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,E,k,H", [
    (65, 4, 1, 8),           # a token past the kernels for few tokens, one piece of a row
    (2047, 8, 2, 136),       # the last chunk of 16 tokens one short
    (2048, 128, 8, 64),      # ... all full, as many experts as are taken
    (2049, 65, 64, 16),      # more than a wave of experts, as many a token as are taken
    (4096, 128, 3, 64),      # a table of which one workgroup a chunk reads
    (4097, 128, 3, 64),
    (12288, 128, 2, 16),     # the largest table
    (12289, 128, 2, 16),     # one token more: the general path
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


# (two launches; more experts than they take: the general path; no tokens)
@pytest.mark.parametrize("T,E", [(100, 8), (2100, 8), (100, 136), (0, 8)])
def test_the_count_of_bad_ids_is_written_with_logits(pkg, lib, T, E):
    """The C entry, which takes the pointer also where the experts come from the logits: 0, whichever launches run."""
    print("bad ids", T, E, flush=True)
    ops, H, I, k = pkg.ops, 64, 32, 2
    r = lambda *s: torch.randn(*s, device="cuda").to(torch.bfloat16)
    i32 = lambda n: torch.empty(n, dtype=torch.int32, device="cuda")
    n = max(T, 1)  # (no tokens: pointers all the same)
    x, logits, w1, w3, w2, out = r(n, H), r(n, E), r(E, I, H), r(E, I, H), r(E, H, I), r(n, H)
    ids, gates, counts, offs, p2r, r2p = i32(n * k), i32(n * k), i32(E), i32(E + 1), i32(n * k), i32(n * k)
    bad = torch.full((1,), 7, dtype=torch.int32, device="cuda")
    xp, act = r(n * k, H), r(n * k, I)
    scratch = torch.empty(max(lib.cdll.moe_layer_scratch_bytes(T, H, E, I, k, 0), 256), dtype=torch.uint8, device="cuda")
    p = lambda t: t.data_ptr()
    bf16 = pkg.lib.DT_BF16
    lib.call_layer("moe_layer_forward", ops._FORWARD_ARGS.pack(
        T, H, E, I, k, p(x), bf16, p(logits), bf16, 0, 0, p(w1), p(w3), p(w2), 0, p(out), bf16, p(ids), p(gates),
        p(counts), p(offs), p(p2r), p(r2p), p(bad), p(xp), 0, p(act), p(scratch), scratch.numel()), ops._stream())
    assert bad.item() == 0 and counts.sum().item() == T * k


@pytest.mark.parametrize("T,E,k,H,x_dt", [
    (1, 16, 1, 32, torch.float32),         # one token, one wave of experts' product
    (15, 16, 16, 64, torch.bfloat16),      # a chunk one token short, every expert asked for
    (16, 48, 3, 544, torch.float32),       # a full one; column blocks that not every wave has
    (17, 128, 64, 1056, torch.float32),    # one more; as many experts as are taken
    (300, 80, 2, 2080, torch.bfloat16),    # rows that leave LDS for one block
    (2049, 112, 8, 128, torch.float32),
    (12288, 128, 2, 32, torch.float32),    # the largest table
    (12289, 128, 2, 32, torch.float32),    # one token more: the general path
])
def test_places_behind_the_norm(pkg, lib, T, E, k, H, x_dt):
    """Norm, router and selection in one kernel, which leaves the counts: the routing against numpy on its logits, the output
    against the layer on the normalised rows with those logits."""
    print("places behind the norm", T, E, k, H, x_dt, flush=True)
    g = torch.Generator().manual_seed(T + E)
    r = lambda *s, std=1.0: (torch.randn(*s, generator=g) * std).cuda()
    x, nw, wr = r(T, H).to(x_dt), 1.0 + r(H, std=0.1), r(E, H, std=0.05).to(torch.bfloat16)
    ws = [r(*s, std=0.1).to(torch.bfloat16) for s in ((E, 8, H), (E, 8, H), (E, H, 8))]
    out, logits, rt = pkg.prenorm_moe(x, nw, wr, *ws, k, eps=1e-6, add_residual=False, return_routing=True)
    flat = O.topk_select(logits.float().cpu(), k)[0].reshape(-1)
    order = np.argsort(flat, kind="stable")
    counts = np.bincount(flat, minlength=E)
    inverse = np.empty_like(order)
    inverse[order] = np.arange(T * k)
    for name, want in (("ids", flat), ("counts", counts), ("offs", np.concatenate([[0], counts.cumsum()])),
                       ("pos_to_row", order), ("row_to_pos", inverse)):
        assert np.array_equal(rt[name].cpu().numpy(), want.astype(np.int32)), name
    xn, _ = pkg.ops.rmsnorm_fwd(x, nw, 1e-6)
    y, rows = pkg.moe_ffn(xn, logits, *ws, k, return_routing=True)
    assert torch.equal(rt["gates"], rows["gates"])
    assert torch.equal(out.to(torch.bfloat16), y)  # (the same kernels from the rows on; fp32 x: an fp32 result, rounded here)


@pytest.mark.parametrize("T,E,H", [
    (1, 1, 8),
    (15, 4, 16),          # a chunk one row short
    (257, 31, 2056),      # a row past a workgroup's 16 chunks; a last word with one count missing
    (4097, 128, 64),      # the most experts
    (12288, 128, 16),     # the largest table
    (12289, 128, 16),     # one row more: the general path
    (16384, 8, 8),        # the most rows
    (16385, 8, 8),
])
@pytest.mark.parametrize("dtype", [torch.int64, torch.int32])
def test_places_of_given_experts(pkg, lib, T, E, H, dtype):
    """Rows whose experts are given, some of them outside [0, E): placed with the nearest expert, and counted."""
    print("places of given experts", T, E, H, dtype, flush=True)
    rng = np.random.default_rng(T + E)
    ids = rng.integers(0, E, T)
    outside = rng.choice(T, T // 5, replace=False)
    ids[outside] = rng.choice([-1, -7, E, E + 3, 2 ** 31 - 1], len(outside))
    if dtype == torch.int64 and len(outside) > 1:
        ids[outside[:2]] = [2 ** 31 + 1, -2 ** 40]
    # (in 32 bits whatever does not fit, like anything below 0 of 64, is -1)
    narrow = np.where((ids < 0) | (ids > 2 ** 31 - 1), -1, ids) if dtype == torch.int64 else ids
    flat = np.clip(narrow, 0, E - 1)
    x = torch.randn(T, H, generator=torch.Generator().manual_seed(T)).to(torch.bfloat16).cuda()
    ws = [torch.randn(*s, device="cuda").to(torch.bfloat16) for s in ((E, 8, H), (E, 8, H), (E, H, 8))]
    out, rt = pkg.experts_rows(x, torch.tensor(ids, dtype=dtype, device="cuda"), *ws, return_routing=True)
    order = np.argsort(flat, kind="stable")
    inverse = np.empty_like(order)
    inverse[order] = np.arange(T)
    counts = np.bincount(flat, minlength=E)
    for name, want in (("counts", counts), ("offs", np.concatenate([[0], counts.cumsum()])), ("pos_to_row", order),
                       ("row_to_pos", inverse), ("bad_ids", np.array([(narrow < 0).sum() + (narrow >= E).sum()]))):
        assert np.array_equal(rt[name].cpu().numpy().reshape(-1), want.astype(np.int32)), name
    sorted_out = pkg.experts_rows(x[torch.tensor(order, device="cuda")], torch.tensor(flat[order], device="cuda"), *ws)
    assert torch.equal(out[torch.tensor(order, device="cuda")], sorted_out)


@pytest.mark.parametrize("T,E,k", [
    (65, 8, 8),       # every expert asked for
    (511, 4, 1),      # a lane short of a workgroup's
    (513, 4, 4),      # one token in its second turn
    (682, 8, 3),      # the most rows
    (1024, 8, 2),
    (1024, 4, 2),
    (1025, 8, 1),     # past it: two launches
])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("unaligned", [False, True])  # logits of which a lane cannot read a row at once: two launches
def test_selection_and_places_in_one_launch(pkg, lib, T, E, k, dtype, unaligned):
    print("one launch", T, E, k, dtype, unaligned, flush=True)
    g = torch.Generator().manual_seed(T + E)
    logits = torch.randn(T, E, generator=g).round(decimals=1).to(dtype)  # (ties)
    logits[::7, 0], logits[::5, E - 1] = -float("inf"), float("inf")
    logits[3, 1], logits[4, :] = float("nan"), -float("inf")
    bias = torch.randn(E, generator=g).round(decimals=1)
    x, ws = torch.randn(T, 64, generator=g), [torch.randn(*s, generator=g) * 0.1 for s in ((E, 8, 64), (E, 8, 64), (E, 64, 8))]
    lg = torch.empty(T * E + 1, dtype=dtype, device="cuda")[1:].view(T, E) if unaligned else torch.empty(T, E, dtype=dtype, device="cuda")
    lg.copy_(logits)
    ops, dev = pkg.ops, lambda t: t.to(torch.bfloat16).cuda()
    i32 = lambda n: torch.empty(n, dtype=torch.int32, device="cuda")
    ids, gates, counts, offs, p2r, r2p = i32(T * k), i32(T * k), i32(E), i32(E + 1), i32(T * k), i32(T * k)
    xd, wd, bd, out = dev(x), [dev(w) for w in ws], bias.cuda(), torch.empty(T, 64, dtype=torch.bfloat16, device="cuda")
    xp, act = torch.empty(T * k, 64, dtype=torch.bfloat16, device="cuda"), torch.empty(T * k, 8, dtype=torch.bfloat16, device="cuda")
    scratch = torch.empty(max(lib.cdll.moe_layer_scratch_bytes(T, 64, E, 8, k, 0), 256), dtype=torch.uint8, device="cuda")
    p, bf16 = lambda t: t.data_ptr(), pkg.lib.DT_BF16
    lib.call_layer("moe_layer_forward", ops._FORWARD_ARGS.pack(
        T, 64, E, 8, k, p(xd), bf16, p(lg), bf16 if dtype == torch.bfloat16 else pkg.lib.DT_F32, p(bd), 0, p(wd[0]), p(wd[1]), p(wd[2]),
        0, p(out), bf16, p(ids), p(gates), p(counts), p(offs), p(p2r), p(r2p), 0, p(xp), 0, p(act), p(scratch),
        scratch.numel()), ops._stream())
    want, _ = O.topk_select(logits.float() + bias, k)
    flat = want.reshape(-1)
    order = np.argsort(flat, kind="stable")
    inverse = np.empty_like(order)
    inverse[order] = np.arange(T * k)
    n = np.bincount(flat, minlength=E)
    for name, got, ref in (("ids", ids, flat), ("counts", counts, n), ("offs", offs, np.concatenate([[0], n.cumsum()])),
                           ("pos_to_row", p2r, order), ("row_to_pos", r2p, inverse)):
        assert np.array_equal(got.cpu().numpy(), ref.astype(np.int32)), name
    assert torch.equal(xp.cpu(), xd.cpu()[torch.tensor(order) // k])
    ids_ref, gates_ref = ops.router_topk(lg.clone(), k, bd)  # (the selection by itself)
    assert torch.equal(ids.view(-1), ids_ref.view(-1)) and torch.equal(gates, gates_ref.reshape(-1).view(torch.int32))
