"""The float32 product and attention on the matrix cores, against float64 and against themselves under other cuts of
the same rows: a row's bits do not depend on the rows beside it."""
import ctypes
import math

import pytest
import torch

from test_kernels_gpu import FakeCtx, View, dev, f64, ops  # noqa: F401  (the fixture)

pytestmark = pytest.mark.gpu

EPS = 2.0 ** -24


@pytest.mark.parametrize("N,K", [(16, 4), (1000, 20), (65, 132), (1024, 1024), (36, 3076)])
def test_product_at_the_edges_of_its_tiles(ops, N, K):  # noqa: F811
    """Rows on either side of every tile's edge, runs of K that end inside a step of 32 or are empty, a last tile of few
    columns.  A sum of K products in 32 bits, added in any order, is within (K + 1) 2^-24 of sum |a| |w|; the error is
    held to that bound, the row beyond the last is left alone, and a row alone has the bits of the row among others."""
    g = torch.Generator().manual_seed(N + K)
    a = torch.randn(321, K, generator=g)
    w = torch.randn(N, K, generator=g)
    ad, wd = dev(a), dev(w)
    ref, size = f64(a) @ f64(w).T, f64(a).abs() @ f64(w).abs().T
    full = torch.empty(321, N, device="cuda")
    ops.linear(ad, wd, full, "store")
    for M in (1, 15, 16, 17, 33, 64, 65, 80, 81, 161, 320):
        out = torch.full((M + 1, N), 7.0, device="cuda")
        ops.linear(ad[:M], wd, out[:M], "store")
        assert ((f64(out[:M]) - ref[:M]).abs() <= (K + 1) * EPS * size[:M]).all(), M
        assert bool((out[M] == 7.0).all()) and torch.equal(out[:M], full[:M]), M
    last = torch.empty(1, N, device="cuda")
    ops.linear(ad[320:], wd, last, "store")
    assert torch.equal(last[0], full[320])
    for epilogue, want in (("add", full + 1.0), ("relu2", torch.relu(full) ** 2)):
        out = torch.ones(321, N, device="cuda")
        ops.linear(ad, wd, out, epilogue)
        assert torch.equal(out, want), epilogue
    if N % 2 == 0:
        for M in (1, 17, 321):
            out = torch.empty(M, N // 2, device="cuda")
            ops.linear(ad[:M], wd, out, "swiglu")
            gate, up = f64(full[:M, :N // 2]), f64(full[:M, N // 2:])
            want = gate / (1 + torch.exp(-gate)) * up
            assert ((f64(out) - want).abs() <= 16 * EPS * want.abs() + 1e-30).all(), M


# a last tile of few rows and of few columns, columns that are no whole float4, runs of K of 1 to 5 steps, an odd number of steps, rows further apart than K
@pytest.mark.parametrize("swiglu,M,N,K,lda", [(0, 321, 8194, 1056, 1056), (0, 130, 40003, 320, 320), (0, 4000, 8194, 64, 64), (0, 64, 151936, 1024, 1056),
                                              (1, 300, 3072, 1024, 1024), (1, 250, 3039, 1056, 1060)])
def test_product_whose_wavefronts_split_together(ops, swiglu, M, N, K, lda):  # noqa: F811
    """The bits of sixteen rows at a time, which go to the kernel whose wavefronts split for themselves, with every epilogue; infinite, NaN
    and the largest floats among the operands.  Within the bound of a 32-bit sum of float64."""
    choice = ops.lib("gemm_generic").ti_gemm_generic_f32_choice
    choice.argtypes = [ctypes.c_int] * 4 + [ctypes.c_long]
    assert choice(swiglu, M, N, K, lda) == 1 and choice(swiglu, 16, N, K, lda) == 0
    g = torch.Generator(device="cuda").manual_seed(M + N)
    rows = torch.randn(M, lda, device="cuda", generator=g)
    w = torch.randn(N * (1 + swiglu), K, device="cuda", generator=g) * 0.05
    rows[M - 1, K - 1], rows[M // 2, 3], rows[1, K // 2] = float("inf"), float("nan"), 3.39e38
    w[N - 1, 5] = float("-inf")
    a = rows[:, :K]
    bits = lambda t: t.view(torch.int32)                      # noqa: E731
    for epilogue in ("swiglu",) if swiglu else ("store", "add", "relu2"):
        full, parts = torch.full((M + 1, N), 0.5, device="cuda"), torch.full((M, N), 0.5, device="cuda")
        ops.linear(a, w, full[:M], epilogue)
        assert bool((full[M] == 0.5).all())
        for m in range(0, M, 16):
            ops.linear(a[m:m + 16], w, parts[m:m + 16], epilogue)
        same = (bits(full[:M]) == bits(parts)) | (torch.isnan(full[:M]) & torch.isnan(parts))
        assert bool(same.all()), epilogue
        if epilogue == "store":
            m = min(M, 400)
            ref, size = a[:m].double() @ w.double().t().contiguous(), a[:m].double().abs() @ w.double().abs().t().contiguous()
            fine = torch.isfinite(ref) & (ref.abs() < 1e38)
            assert bool(((full[:m].double() - ref).abs() <= (K + 1) * EPS * size)[fine].all())
            assert torch.equal(torch.isnan(full[:m]), torch.isnan(ref))


@pytest.mark.parametrize("swiglu,M,N,K,together", [
    # one workgroup a unit: a round that is nearly full, and one that has just begun; 600 rows begin a fourth round of the dies with the most columns
    (1, 256, 3072, 1024, 1), (1, 512, 3072, 1024, 0), (1, 384, 4864, 896, 1), (1, 600, 4864, 896, 0), (1, 64, 9728, 2560, 1), (1, 100, 9728, 2560, 0),
    # two workgroups a unit
    (0, 512, 4096, 1024, 0), (0, 1000, 4096, 1024, 1), (0, 1280, 4096, 1024, 0), (0, 300, 6144, 4096, 0), (0, 2048, 6144, 4096, 1)])
def test_which_products_split_together(ops, swiglu, M, N, K, together):  # noqa: F811
    """The faster of the two kernels, as measured on either side of the line."""
    choice = ops.lib("gemm_generic").ti_gemm_generic_f32_choice
    choice.argtypes = [ctypes.c_int] * 4 + [ctypes.c_long]
    assert choice(swiglu, M, N, K, K) == together


@pytest.mark.parametrize("M,N,K", [(7, 64, 20), (37, 132, 1056), (300, 96, 260)])
def test_product_of_what_three_bfloat16_do_not_hold(ops, M, N, K):  # noqa: F811
    """Operands from 1e-30 to the largest float, infinite ones and NaN, beside zeros: what float64 gives in 32 bits is what comes out, of
    the same kind where it is not finite, within the bound of a 32-bit sum where it is.  Every row by every weight row's own kind."""
    g = torch.Generator().manual_seed(M + N + K)
    a, w = torch.randn(M, K, generator=g), torch.randn(N, K, generator=g) * 1e-3
    big = torch.finfo(torch.float32).max
    for i, x in enumerate((1e-30, big, -big, float("inf"), float("nan"), 3.39e38)):
        a[(3 * i) % M, (5 * i + 1) % K] = x
    a[M // 2] *= 1e-30
    w[3] *= 1e-6
    w[5, :] = 0.0
    w[7, 6 % K] = float("-inf")
    w[9, K - 1] = float("nan")
    ref = f64(a) @ f64(w).T
    size = f64(a).abs() @ f64(w).abs().T
    out = torch.empty(M, N, device="cuda")
    ops.linear(dev(a), dev(w), out, "store")
    out = f64(out)
    fine = torch.isfinite(ref) & (ref.abs() < big)
    assert fine.any() and not fine.all()
    assert ((out - ref).abs() <= (K + 1) * EPS * size + 1e-36)[fine].all()
    assert torch.equal(torch.isnan(out), torch.isnan(ref))
    assert torch.equal(torch.isposinf(out), torch.isposinf(ref)) and torch.equal(torch.isneginf(out), torch.isneginf(ref))


@pytest.mark.parametrize("M,N,K", [(7, 64, 20), (37, 132, 1056), (300, 96, 260), (1000, 64, 96)])
def test_product_of_the_smallest_floats_and_of_single_ones(ops, M, N, K):  # noqa: F811
    """Tokens, weights and both down to the subnormal floats: the bound of a 32-bit sum, and half the last place of what a subnormal
    result holds.  One token element a row that is not zero: each result is one product, rounded once (2^-24 of it), of whose nine products
    of pieces the three least, 2^-24 of it together, are left out; a zero row gives zeros."""
    g = torch.Generator().manual_seed(M + N + K)
    a, w = torch.randn(M, K, generator=g), torch.randn(N, K, generator=g)
    out = torch.empty(M, N, device="cuda")
    for small_a, small_w in ((1e-36, 1.0), (1e-39, 1.0), (1e-43, 1.0), (1.0, 1e-39), (1e-20, 1e-19)):
        x, y = a * small_a, w * small_w
        ops.linear(dev(x), dev(y), out, "store")
        size = f64(x).abs() @ f64(y).abs().T
        assert ((f64(out) - f64(x) @ f64(y).T).abs() <= (K + 1) * EPS * size + 2.0 ** -150).all(), (small_a, small_w)
    single = torch.zeros(M, K)
    single[torch.arange(M), torch.randint(0, K, (M,), generator=g)] = a[:, 0]
    single[M // 2] = 0.0
    ops.linear(dev(single), dev(w), out, "store")
    ref = f64(single) @ f64(w).T
    assert ((f64(out) - ref).abs() <= 2 * EPS * ref.abs()).all() and not out[M // 2].any()


def case(entries, nh, nkv, hd, P, window, seed):
    """Requests with pages scattered over a pool of rubbish; the queries of a step's last tokens, and float64's result."""
    g = torch.Generator().manual_seed(seed)
    lens = [s + n for n, s in entries]
    each = [-(-n // P) for n in lens]
    pages = sum(each) + 3
    perm = torch.randperm(pages - 1, generator=g) + 1
    pool = torch.full((pages, 2, nkv, P, hd), float("nan"))
    vt = pool[:, 1].reshape(pages, nkv, hd, P)
    table = torch.full((len(lens), max(each) + 1), -1, dtype=torch.int32)
    qs, want, used = [], [], 0
    for e, ((n, start), size) in enumerate(zip(entries, lens)):
        k, v = torch.randn(size, nkv, hd, generator=g), torch.randn(size, nkv, hd, generator=g)
        q = torch.randn(n, nh, hd, generator=g)
        mine = perm[used:used + each[e]]
        used += each[e]
        for t in range(size):
            pool[mine[t // P], 0, :, t % P] = k[t]
            vt[mine[t // P], :, :, t % P] = v[t]
        first = max(0, start - window + 1) // P if window else 0
        table[e, first:each[e]] = mine[first:].to(torch.int32)        # pages behind the window were given back
        i = torch.arange(start, size)[:, None]
        j = torch.arange(size)[None, :]
        hidden = (j > i) | ((i - j >= window) if window else False)
        o = torch.empty(n, nh, hd, dtype=torch.float64)
        for h in range(nh):
            s = (f64(q[:, h]) @ f64(k[:, h * nkv // nh]).T / math.sqrt(hd)).masked_fill(hidden, float("-inf"))
            o[:, h] = torch.softmax(s, -1) @ f64(v[:, h * nkv // nh])
        qs.append(q.reshape(n, nh * hd))
        want.append(o.reshape(n, nh * hd))
    pool[:, 1] = vt.reshape(pages, nkv, P, hd)
    return qs, dev(pool.reshape(pages, 2 * nkv, P, hd).contiguous()), table, want


@pytest.mark.parametrize("nh,nkv,hd,P,window", [(2, 1, 16, 4, None), (6, 2, 48, 12, 37), (16, 8, 128, 16, None), (17, 1, 64, 16, 70),
                                                (5, 5, 256, 4, None)])
def test_attention_under_every_cut_of_a_step(ops, nh, nkv, hd, P, window):  # noqa: F811
    """Portions that start at 0 and in the middle, of one row beyond a tile and of two, beside single tokens, one of them
    alone in its context; rows never written hold NaN.  Within 2e-5 of float64 (a row's weights sum to one; scores of
    some 4 sqrt(hd) / 2^24 and sums of hundreds of keys), and each row taken as a single token has the same bits."""
    entries = [(65, 0), (1, 0), (18, 131), (1, 300), (2, 15), (1, 16)]
    qs, pool, table, want = case(entries, nh, nkv, hd, P, window, seed=nh + hd)
    q = dev(torch.cat(qs))
    out = torch.full_like(q, 7.0)
    args = (nh, nkv, hd, 1.0 / math.sqrt(hd), window)
    ops.attention(FakeCtx(entries), View(dev(table)), q, pool, out, *args)
    assert (f64(out) - torch.cat(want)).abs().max() < 2e-5
    for row_in, e in ((0, 0), (40, 0), (64, 0), (7, 2), (17, 2), (1, 4)):
        row = sum(n for n, _ in entries[:e]) + row_in
        one = torch.empty(1, nh * hd, device="cuda")
        ops.attention(FakeCtx([(1, entries[e][1] + row_in)]), View(dev(table[e:e + 1].contiguous())), q[row:row + 1].contiguous(), pool,
                      one, *args)
        assert torch.equal(one[0], out[row]), (row_in, e)
    try:
        ops.use_fast_attention = False
        rows = torch.empty_like(q)
        ops.attention(FakeCtx(entries), View(dev(table)), q, pool, rows, *args)
    finally:
        ops.use_fast_attention = True
    assert (f64(rows) - f64(out)).abs().max() < 2e-5


@pytest.mark.parametrize("nh,nkv,hd,P,window", [(2, 1, 16, 16, None), (17, 1, 48, 48, 37), (4, 2, 64, 16, 70), (3, 3, 80, 32, None),
                                                (4, 4, 112, 16, 20), (16, 8, 128, 16, None), (2, 2, 128, 64, 37)])
def test_attention_blocks_through_lds_and_straight_from_memory(ops, nh, nkv, hd, P, window):  # noqa: F811
    """Pages of whole blocks, whose keys and values come through LDS, and the same cache in pages of 4 rows, whose come straight from
    memory: the same bits, for heads of every remainder of four slices, contexts of no, one and several blocks a wavefront, and pages
    given back behind a window; rows never written hold NaN."""
    entries = [(65, 0), (1, 0), (18, 131), (1, 300), (2, 15), (130, 3), (1, 16)]
    qs, pool, table, want = case(entries, nh, nkv, hd, P, window, seed=nh + hd + P)
    q, n = dev(torch.cat(qs)), P // 4
    pages = pool.cpu().view(-1, 2, nkv * P * hd)
    k = pages[:, 0].reshape(-1, nkv, n, 4, hd).permute(0, 2, 1, 3, 4).reshape(-1, nkv * 4 * hd)
    v = pages[:, 1].reshape(-1, nkv, hd, n, 4).permute(0, 3, 1, 2, 4).reshape(-1, nkv * hd * 4)
    small = dev(torch.stack((k, v), 1).reshape(-1, 2 * nkv, 4, hd).contiguous())
    ids = torch.where(table[:, :, None] < 0, -1, table[:, :, None] * n + torch.arange(n, dtype=torch.int32)).to(torch.int32)
    args = (nh, nkv, hd, 1.0 / math.sqrt(hd), window)
    staged, straight = torch.full_like(q, 7.0), torch.full_like(q, 8.0)
    ops.attention(FakeCtx(entries), View(dev(table)), q, pool, staged, *args)
    ops.attention(FakeCtx(entries), View(dev(ids.reshape(len(entries), -1).contiguous())), q, small, straight, *args)
    assert (f64(staged) - torch.cat(want)).abs().max() < 2e-5
    assert torch.equal(staged, straight)


def hold(pool, table, P, nkv, hd, e, j, key, value):
    """What the cache holds of request e's token j: its key and its value, the same number everywhere."""
    page = pool[int(table[e, j // P])]
    page[:nkv, j % P] = key
    page[nkv:].view(nkv, hd, P)[:, :, j % P] = value


@pytest.mark.parametrize("hd,P,window", [(16, 4, None), (64, 16, None), (128, 16, 20), (256, 4, 20), (144, 16, 33)])
@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
def test_rows_do_not_feel_what_they_cannot_see(ops, bad, hd, P, window):  # noqa: F811
    """Infinite and not-a-number keys and values of tokens in the middle of a text: rows in front of them, and rows whose
    window has left them behind, keep their bits in every cut of the step; the rows that see them are spoiled."""
    nh, nkv = 4, 2
    entries = [(65, 0), (40, 37), (1, 50)]
    qs, pool, table, _ = case(entries, nh, nkv, hd, P, window, seed=hd)
    q, view, args = dev(torch.cat(qs)), View(dev(table)), (nh, nkv, hd, 1.0 / math.sqrt(hd), window)
    clean, out = torch.empty_like(q), torch.empty_like(q)
    ops.attention(FakeCtx(entries), view, q, pool, clean, *args)
    told = [(0, 9, 0.0, bad), (0, 21, bad, 0.0), (1, 44, 0.0, -bad), (1, 61, bad, bad), (2, 50 - (window or 0) if window else 50, 0.0, bad)]
    for e, j, key, value in told:
        hold(pool, table, P, nkv, hd, e, j, key, value)
    ops.attention(FakeCtx(entries), view, q, pool, out, *args)
    row = 0
    for e, (n, start) in enumerate(entries):
        for p in range(start, start + n):
            seen = any(x == e and j <= p and (not window or p - j < window) for x, j, _, _ in told)
            if seen:
                assert not torch.isfinite(out[row]).any(), (e, p)
            else:
                assert torch.equal(out[row], clean[row]), (e, p)
            row += 1


def test_portions_without_a_list_of_small_tiles(ops):  # noqa: F811
    """A work list that names its portions by tiles of 128 rows alone, beside a single token: every row is written."""
    nh, nkv, hd, P = 4, 2, 64, 16
    entries = [(65, 0), (1, 40)]
    qs, pool, table, want = case(entries, nh, nkv, hd, P, None, seed=3)
    ctx, q = FakeCtx(entries), dev(torch.cat(qs))
    ctx.tiles_small, ctx.n_tiles_small = None, 0
    out = torch.full_like(q, 7.0)
    ops.attention(ctx, View(dev(table)), q, pool, out, nh, nkv, hd, 1.0 / math.sqrt(hd), None)
    assert (f64(out) - torch.cat(want)).abs().max() < 2e-5
