"""fp32 products in three bf16 parts (csrc/f32_split.h) against fp64: where tiles and their quarters end, the smallest widths,
operands whose size changes along the contraction and from row to row or column to column, the ends of the fp32 range,
infinities and NaN.

Bar: an element of a product of K terms may be off by (6 K / 16 + 8) roundings of its accumulator and by the parts that are left
out, 2^-24 of every product: c = (6 K / 16 + 10) 2^-24 times the sum of the sizes of its own products.  Nothing else takes part in
the bar: a small element of a large result is held to its own digits."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
SPLIT = 1


@pytest.fixture
def forced(lib, pkg):
    def force(tile):
        return pkg.lib.load().cdll.moe_f32_gemm_force_tile(tile)
    before = force(SPLIT)
    yield force
    force(before)


def _offs(counts):
    return torch.tensor(np.concatenate([[0], np.cumsum(counts)]), dtype=torch.int32)


def _check(name, got, ref, size, K):
    bar = (6 * K / 16 + 10) * 2.0 ** -24 * size
    off = (got.cpu().double() - ref).abs()
    worst = (off / bar.clamp_min(2.0 ** -149)).max().item()  # (half of the smallest value fp32 has may be lost at the end)
    print("  ", name, K, "share of the bound", worst, flush=True)
    assert worst <= 1.0, name


@pytest.mark.parametrize("counts,H,I", [
    ([1, 0, 33], 4, 4),                              # the smallest widths
    ([65, 0, 130, 31, 97], 100, 36),                 # ragged everything, quarters only
    ([300, 7, 0, 513, 64, 1, 0, 200] * 9, 132, 260),  # more experts than lanes in a wave, a cut last round
    ([700, 650, 500], 1028, 132),                    # contractions that end inside a k-tile
    ([128, 256], 64, 128),                           # whole tiles and k-tiles
])
def test_split_products(pkg, lib, forced, counts, H, I):
    print("split products", len(counts), sum(counts), H, I, flush=True)
    g = torch.Generator().manual_seed(sum(counts) + H)
    E, R, offs = len(counts), sum(counts), _offs(counts)
    r = lambda *s: torch.randn(*s, generator=g) * 0.3
    xp, dyp, w1, w3, w2 = r(R, H), r(R, H), r(E, I, H), r(E, I, H), r(E, H, I)
    ops = pkg.ops
    x_, dy_, w1_, w3_, w2_, o_ = (v.cuda() for v in (xp, dyp, w1, w3, w2, offs))
    g_, u_, a_ = ops.f32_gateup_swiglu(x_, w1_, w3_, o_)
    y_ = ops.f32_gemm_rows(a_, w2_, o_, True)
    d_ = ops.f32_gemm_rows(dy_, w2_, o_, False)
    dg_, du_ = ops.f32_down_swiglu_bwd(dy_, w2_, g_, u_, o_)
    dx_ = ops.f32_gateup_bwd(dg_, du_, w1_, w3_, o_)
    dw = ops.f32_wgrads(dg_, du_, dy_, x_, a_, o_)
    d = lambda t: t.cpu().double()
    rows = [slice(int(offs[e]), int(offs[e + 1])) for e in range(E)]
    per = lambda a, w: (torch.cat([d(a)[s] @ d(w)[e].t() for e, s in enumerate(rows)]),
                        torch.cat([d(a)[s].abs() @ d(w)[e].abs().t() for e, s in enumerate(rows)]))
    back = lambda w: d(w).transpose(1, 2).contiguous()
    for name, got, (ref, size), K in (("g", g_, per(xp, w1), H), ("u", u_, per(xp, w3), H), ("y", y_, per(a_, w2), I),
                                      ("d", d_, per(dyp, back(w2)), H)):
        _check(name, got, ref, size, K)
    one, two = per(dg_, back(w1)), per(du_, back(w3))
    _check("dx", dx_, one[0] + two[0], one[1] + two[1], 2 * I)
    # the epilogues, on the products as the device has them: a few roundings and an exponential
    gd, ud, s = d(g_), d(u_), torch.sigmoid(d(g_))
    for name, got, ref in (("act", a_, gd * s * ud), ("dg", dg_, d(d_) * ud * (s * (1 + gd * (1 - s)))), ("du", du_, d(d_) * gd * s)):
        assert ((d(got) - ref).abs() <= 2.0 ** -20 * (ref.abs() + ref.abs().max())).all(), name
    for name, got, a, b in (("dw1", dw[0], dg_, xp), ("dw3", dw[1], du_, xp), ("dw2", dw[2], dyp, a_)):
        ref = torch.stack([d(a)[q].t() @ d(b)[q] for q in rows])
        size = torch.stack([d(a)[q].abs().t() @ d(b)[q].abs() for q in rows])
        _check(name, got, ref, size, max(counts))
        for e in range(E):
            assert counts[e] or not got[e].any()


@pytest.mark.parametrize("a_size,b_size", [
    (lambda k: 2.0 ** (k // 40), lambda k: 1.0),               # larger and larger: the scale changes again and again
    (lambda k: 2.0 ** -(k // 40), lambda k: 2.0 ** (k // 40)),  # one shrinks as the other grows
    (lambda k: 1e-30 if k < 500 else 1e20, lambda k: 1.0),     # one large change
    (lambda k: 1e6 if k < 512 else 1e-6, lambda k: 1e-6 if k < 512 else 1e7),
    (lambda k: 1e6 if k // 128 % 2 else 1e-6, lambda k: 1e-6 if k // 128 % 2 else 1e6),
    (lambda k: 1e8 if k // 256 % 2 else 1e-8, lambda k: 1e-8 if k // 256 % 2 else 1e8),
    (lambda k: 1e10 if k // 256 % 2 else 1e-10, lambda k: 1e-10 if k // 256 % 2 else 1e10),
    (lambda k: 1e10 if k < 512 else 1e-10, lambda k: 1e-10 if k < 512 else 1e10),
    (lambda k: 1e15 if k % 2 else 1e-15, lambda k: 1e-15 if k % 2 else 1e15),  # from term to term
    (lambda k: 1e15 if k < 16 else 1.0, lambda k: 0.0 if k < 16 else 1.0),     # what is large meets zeros
    (lambda k: 1.0, lambda k: 1.0 if k < 64 else 1e-12),       # the third and fourth k-tile smaller than those before
    (lambda k: 0.0 if k < 300 else 1.0, lambda k: 3e-38),      # zeros first; the smallest normal values
    (lambda k: 1e19, lambda k: 1e16),                          # large ones
    (lambda k: 1e-20, lambda k: 1e-16),
], ids=["growing", "both ways", "one change", "one each", "to and fro", "to and fro 1e8", "to and fro 1e10",
        "shrinking and growing 1e10", "by terms 1e15", "large times zero", "small from the third k-tile on", "zeros first", "large", "small"])
def test_operands_that_change_along_the_contraction(pkg, lib, forced, a_size, b_size):
    R, N, K = 200, 136, 1100
    g = torch.Generator().manual_seed(3)
    a = torch.randn(R, K, generator=g) * torch.tensor([a_size(k) for k in range(K)])
    b = torch.randn(1, N, K, generator=g) * torch.tensor([b_size(k) for k in range(K)])
    o = _offs([R]).cuda()
    ref = a.double() @ b[0].double().t()
    got = pkg.ops.f32_gemm_rows(a.cuda(), b.cuda(), o, True)
    forced(64)
    plain = pkg.ops.f32_gemm_rows(a.cuda(), b.cuda(), o, True)
    forced(SPLIT)
    # the same product with the contraction along the rows of both
    wg = pkg.ops.f32_gemm_wgrad(a.t().contiguous().cuda(), b[0].t().contiguous().cuda(), _offs([K]).cuda(), 1)[0]
    rel = lambda t: ((t.cpu().double() - ref).norm() / ref.norm()).item()
    print("  split", rel(got), "transposed", rel(wg), "fp32", rel(plain), flush=True)
    assert rel(got) <= 1e-6 and rel(wg) <= 1e-6  # (1100 terms: 5e-7)
    size = a.double().abs() @ b[0].double().abs().t()
    _check("rows", got, ref, size, K)
    _check("transposed", wg, ref, size, K)


def test_a_row_does_not_change_the_others(pkg, lib, forced):
    """Rows of very different size in one tile: each has the precision it has alone."""
    R, N, K = 300, 200, 520
    g = torch.Generator().manual_seed(6)
    a, b = torch.randn(R, K, generator=g), torch.randn(1, N, K, generator=g)
    a *= torch.tensor([10.0 ** (i % 61 - 30) for i in range(R)]).unsqueeze(1)
    a[10:20, :200] *= 1e-9  # rows that grow along the contraction, and that shrink
    a[20:30, 200:] *= 1e-9
    for b_k in (True, False):
        w = b if b_k else b.transpose(1, 2).contiguous()
        got = pkg.ops.f32_gemm_rows(a.cuda(), w.cuda(), _offs([R]).cuda(), b_k).cpu().double()
        ref = a.double() @ b[0].double().t()
        assert ((got - ref).norm(dim=1) / ref.norm(dim=1)).max() <= 1e-6  # (520 terms: 3e-7)


@pytest.mark.parametrize("spread", [10, 20, 40, 60])
@pytest.mark.parametrize("first", [1.0, 2.0 ** 20])
def test_rows_and_columns_of_any_size_keep_their_digits(pkg, lib, forced, spread, first):
    """Rows of both operands 2^-spread apart side by side, alone and with the first terms of every sum much larger (and, in
    half of the rows of B, meeting zeros): each element has the digits its own products have, in every launch."""
    R, N, K = 300, 200, 520
    g = torch.Generator().manual_seed(spread)
    a, b = torch.randn(R, K, generator=g), torch.randn(1, N, K, generator=g)
    a *= torch.exp2(torch.arange(R) % 5 * (-spread / 4)).unsqueeze(1)
    b *= torch.exp2(torch.arange(N) % 3 * (-spread / 2)).view(1, N, 1)
    a[:, :8] *= first
    b[:, N // 2:, :8] = 0
    ops, o = pkg.ops, _offs([R]).cuda()
    ref, size = a.double() @ b[0].double().t(), a.double().abs() @ b[0].double().abs().t()
    for b_k in (True, False):
        w = b if b_k else b.transpose(1, 2).contiguous()
        _check("rows", ops.f32_gemm_rows(a.cuda(), w.cuda(), o, b_k), ref, size, K)
    _check("wgrad", ops.f32_gemm_wgrad(a.t().contiguous().cuda(), b[0].t().contiguous().cuda(), _offs([K]).cuda(), 1)[0], ref, size, K)
    # one of gate's and up's weights far below the other's
    small = b * 2.0 ** -spread
    for w1, w3 in ((b, small), (small, b)):
        g_, u_, _ = ops.f32_gateup_swiglu(a.cuda(), w1.cuda(), w3.cuda(), o)
        for name, got, w in (("g", g_, w1), ("u", u_, w3)):
            k = 1.0 if w is b else 2.0 ** -spread
            _check(name, got, ref * k, size * k, K)
    # the two halves of an input gradient
    back = b.transpose(1, 2).contiguous().cuda()
    dx = ops.f32_gateup_bwd(a.cuda(), (a * 2.0 ** -spread).cuda(), back * 2.0 ** -spread, back, o)
    _check("dx", dx, ref * 2.0 ** (1 - spread), size * 2.0 ** (1 - spread), 2 * K)


@pytest.mark.parametrize("a_size,b_size", [(1e-38, 1e30), (1e-41, 1e36), (3e37, 1e-36), (1e38, 1e-38), (2.0 ** -149, 1.0),
                                           (2.0 ** -140, 2.0 ** 100), (2.0 ** 60, 2.0 ** 60)])
def test_the_ends_of_the_range(pkg, lib, forced, a_size, b_size):
    """Denormal values, the smallest and the largest normal ones, results past 2^80."""
    R, N, K = 132, 68, 260
    g = torch.Generator().manual_seed(8)
    a = torch.rand(R, K, generator=g).add_(1).mul_(a_size)
    b = torch.randn(1, N, K, generator=g) * b_size
    ref, size = a.double() @ b[0].double().t(), a.double().abs() @ b[0].double().abs().t()
    _check("rows", pkg.ops.f32_gemm_rows(a.cuda(), b.cuda(), _offs([R]).cuda(), True), ref, size, K)
    dw = pkg.ops.f32_gemm_wgrad(a.t().contiguous().cuda(), b[0].t().contiguous().cuda(), _offs([K]).cuda(), 1)[0]
    _check("wgrad", dw, ref, size, K)


def test_infinities_and_nan(pkg, lib, forced):
    """Rows and columns with values that are not finite, or overflow, become what the fp32 instruction makes of them; the
    others keep their values."""
    R, N, K = 300, 200, 260
    g = torch.Generator().manual_seed(4)
    a, b = torch.randn(R, K, generator=g), torch.randn(1, N, K, generator=g)
    a[5, 7], a[140, 3], a[141, 250] = float("inf"), float("nan"), -float("inf")
    b[0, 77, 9] = float("inf")
    o = _offs([R]).cuda()

    def both(a):
        one = pkg.ops.f32_gemm_rows(a.cuda(), b.cuda(), o, True).cpu()
        forced(64)
        two = pkg.ops.f32_gemm_rows(a.cuda(), b.cuda(), o, True).cpu()
        forced(SPLIT)
        return one, two

    got, want = both(a)
    at, bt = a.t().contiguous(), b[0].t().contiguous()
    for x in (got, pkg.ops.f32_gemm_wgrad(at.cuda(), bt.cuda(), _offs([K]).cuda(), 1)[0].cpu()):
        assert torch.equal(x.isnan(), want.isnan()) and torch.equal(x[x.isinf()], want[want.isinf()])
        ok = want.isfinite()
        assert ok[0].sum() == N - 1 and not ok[5].any()
        assert (x[ok].double() - want[ok].double()).norm() <= 1e-6 * want[ok].double().norm()
    # the bits of elements whose values are all finite are those they have without the others
    rows, cols = torch.ones(R, dtype=torch.bool), torch.ones(N, dtype=torch.bool)
    rows[[5, 140, 141]], cols[77] = False, False
    calm, calm_b = a.nan_to_num(1, 1, 1), b.nan_to_num(1, 1, 1)
    alone = pkg.ops.f32_gemm_rows(calm.cuda(), calm_b.cuda(), o, True).cpu()
    assert torch.equal(got[rows][:, cols], alone[rows][:, cols])
    a[260, :] = 3e38  # sums that overflow or not, by the order of their terms
    got, want = both(a)
    usual = torch.arange(R) != 260
    x, y = got[usual], want[usual]
    ok = y.isfinite()
    assert torch.equal(x.isnan(), y.isnan()) and (x[ok].double() - y[ok].double()).norm() <= 1e-6 * y[ok].double().norm()


@pytest.mark.parametrize("uneven", [False, True])
def test_two_runs_give_the_same_bits(pkg, lib, forced, uneven):
    counts, H, I = [513, 0, 200, 64], 516, 132
    g = torch.Generator().manual_seed(5)
    x, w1, w3 = (torch.randn(*s, generator=g).cuda() for s in ((sum(counts), H), (4, I, H), (4, I, H)))
    if uneven:  # the third and fourth k-tile much smaller than the others
        x[:, 64:128] *= 2.0 ** -30
        w1[:, :, 64:256] *= 2.0 ** -20
    o = _offs(counts).cuda()
    one = pkg.ops.f32_gateup_swiglu(x, w1, w3, o)
    short = torch.ones(8 * 128, 128, device="cuda")  # contractions of few k-tiles on every compute unit between the two
    pkg.ops.f32_gemm_wgrad(short, short, torch.arange(0, 1025, 128, dtype=torch.int32, device="cuda"), 8)
    two = pkg.ops.f32_gateup_swiglu(x, w1, w3, o)
    assert all(torch.equal(p, q) for p, q in zip(one, two))
    dw = [pkg.ops.f32_gemm_wgrad(one[0], x, o, 4) for _ in range(2)]
    assert torch.equal(*dw)
    # added to what is there: the sum of the rounded result and the old value
    old = torch.randn(4, I, H, generator=g).cuda()
    acc = pkg.ops.f32_gemm_wgrad(one[0], x, o, 4, out=old.clone())
    assert torch.equal(acc, torch.where(torch.tensor(counts, device="cuda").view(4, 1, 1) > 0, dw[0] + old, old))


@pytest.mark.parametrize("E,R,N,K", [
    (4, 2176, 2048, 256),    # the shortest contraction the split tiles take where there is work enough
    (4, 2176, 2048, 252),    # shorter: fp32 products
    (32, 2048, 2048, 260),   # experts that fill half a tile
    (32, 2047, 2048, 260),   # ... a row less
    (128, 1020, 2584, 36),   # many large tiles by the bound, of few rows: small ones
])
def test_at_the_lines_of_the_rule(pkg, lib, forced, E, R, N, K):
    forced(0)
    g = torch.Generator().manual_seed(R + K)
    counts = [R // E + (e < R % E) for e in range(E)]
    a, b = torch.randn(R, K, generator=g), torch.randn(E, N, K, generator=g)
    got = pkg.ops.f32_gemm_rows(a.cuda(), b.cuda(), _offs(counts).cuda(), True)
    parts, sizes = a.double().split(counts), a.double().abs().split(counts)
    ref = torch.cat([p @ w.double().t() for p, w in zip(parts, b)])
    size = torch.cat([p @ w.double().abs().t() for p, w in zip(sizes, b)])
    # (either tile: at most a rounding for every product of the contraction, and the parts that the split leaves out)
    assert ((got.cpu().double() - ref).abs() <= (K + 1) * 2.0 ** -24 * size).all()


@pytest.mark.parametrize("E,R,M,N", [
    (8, 1792, 1024, 1024),   # weight gradients: the fewest rows an expert that split tiles take
    (8, 1791, 1024, 1024),   # ... a row less
    (4, 3584, 1024, 1028),   # columns past the tiles
    (4, 3584, 1024, 960),    # fewer tiles than compute units
])
def test_at_the_lines_of_the_weight_gradients(pkg, lib, forced, E, R, M, N):
    forced(0)
    g = torch.Generator().manual_seed(R + N)
    counts = [R // E + (e < R % E) for e in range(E)]
    a, b = torch.randn(R, M, generator=g), torch.randn(R, N, generator=g)
    got = pkg.ops.f32_gemm_wgrad(a.cuda(), b.cuda(), _offs(counts).cuda(), E)
    parts = list(zip(a.double().split(counts), b.double().split(counts)))
    ref = torch.stack([p.t() @ q for p, q in parts])
    size = torch.stack([p.abs().t() @ q.abs() for p, q in parts])
    assert ((got.cpu().double() - ref).abs() <= (max(counts) + 1) * 2.0 ** -24 * size).all()
