"""The pipelined product's tiles beyond the ones tests of the whole dispatch name, loops shorter than the ring of stages,
the dies' blocks of tiles, split sums and the norm behind them, the q/k/v product in tiles of 64 rows, and what large weights
under few rows and very long rows take."""
import ctypes

import pytest
import torch

from test_kernels_gpu import dev, f64, ops, qkv_prepared_case, ref_linear  # noqa: F401  (the fixture)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K", [64, 128, 192, 320, 448])
@pytest.mark.parametrize("M,N", [(65, 160), (129, 256), (300, 136)])
def test_every_tile_over_few_k_tiles(ops, M, N, K):  # noqa: F811
    """One to seven k-tiles (the rings hold two to five) under every tile: the bits of the 128 x 64 tile, which are the sums in
    ascending steps of 16, within K 2^-24 of float64 for each of the K sums' terms; the row behind the last is left alone."""
    lib = ops.lib("gemm_bf16")
    g = torch.Generator().manual_seed(M + K)
    a = dev((torch.rand(M, K, generator=g) * 2 - 1).to(torch.bfloat16))
    w = dev((torch.rand(N, K, generator=g) * 2 - 1).to(torch.bfloat16))
    ref, size = ref_linear(a.cpu(), w.cpu()), f64(a).abs() @ f64(w).abs().T
    want = {}
    try:
        for tile in (3, 1, 2, 4, 5, 6, 7, 8, 9, 10, 11):
            lib.ti_tuning_set(b"force_tile", tile)
            out = torch.full((M + 1, N), 7.0, device="cuda")
            ops.linear(a, w, out[:M], "store")
            act = torch.full((M + 1, N // 2), 7.0, device="cuda", dtype=torch.bfloat16)
            ops.linear(a, w, act[:M], "swiglu")
            assert bool((out[M] == 7.0).all()) and bool((act[M] == 7.0).all())
            added = torch.ones(M, N, device="cuda")
            ops.linear(a, w, added, "add")
            got = (out[:M], act[:M], added)
            want = want or got
            for x, y in zip(got, want):
                assert torch.equal(x, y), tile
    finally:
        lib.ti_tuning_set(b"force_tile", 0)
    assert ((f64(want[0]) - ref).abs() <= (K + 1) * 2.0 ** -24 * size).all()


@pytest.mark.parametrize("tile", [10, 12])
@pytest.mark.parametrize("M,F,K,shift", [(255, 128, 64, 0), (257, 136, 128, 0), (256, 130, 192, 0), (513, 264, 256, 0), (64, 8, 576, 0), (300, 136, 320, 4)])
def test_tiles_of_256_by_quarters(ops, tile, M, F, K, shift):  # noqa: F811
    """The loop by quarters over one k-tile and more than its two stages, rows and columns a tile, one more and one less, columns in
    whole pieces of 16 bytes and not (130), a result that starts between two pieces (shift): the bits of the 128 x 128 tile."""
    lib = ops.lib("gemm_bf16")
    g = torch.Generator().manual_seed(M + F + K)
    a = dev((torch.rand(M, K, generator=g) * 2 - 1).to(torch.bfloat16))
    w = dev((torch.rand(2 * F, K, generator=g) * 2 - 1).to(torch.bfloat16))
    outs = []
    lib.ti_tuning_set(b"rows_112", 0)
    lib.ti_tuning_set(b"tiled_from", 1)
    try:
        for force in (2, tile):
            lib.ti_tuning_set(b"force_tile", force)
            room = torch.full((M * F + 16,), 7.0, device="cuda", dtype=torch.bfloat16)
            out = room[shift:shift + M * F].view(M, F)
            ops.linear(a, w, out, "swiglu")
            assert bool((room[:shift] == 7.0).all()) and bool((room[shift + M * F:] == 7.0).all())
            outs.append(out.clone())
    finally:
        lib.ti_tuning_reset()
    assert torch.equal(outs[0], outs[1])
    gate, up = (ref_linear(a.cpu(), w[i * F:(i + 1) * F].cpu()) for i in (0, 1))
    want = torch.nn.functional.silu(gate) * up
    # sums of K products within K 2^-24 of their sizes, a result rounded to 8 bits
    assert ((f64(outs[1]) - want).abs() <= 2.0 ** -8 * want.abs() + (K + 8) * 2.0 ** -24 * K * (1 + up.abs() + gate.abs())).all()


@pytest.mark.parametrize("M,F,K,tile", [(2048, 3072, 1024, 10), (2048, 12288, 4096, 12), (512, 3072, 1024, 0), (2000, 2565, 2048, 10)])
def test_which_gate_up_products_go_by_quarters(ops, M, F, K, tile):  # noqa: F811
    """Where the costs say so, and with the bits of what is taken without them: two tile shapes for two ranges of columns, or one."""
    lib = ops.lib("gemm_bf16")
    assert lib.ti_gemm_bf16_quarters_choice(M, F, K) == tile
    g = torch.Generator(device="cuda").manual_seed(M + F)
    a = torch.randn(M, K, device="cuda", generator=g).to(torch.bfloat16)
    w = (torch.randn(2 * F, K, device="cuda", generator=g) * 0.1).to(torch.bfloat16)
    outs = []
    try:
        for on, ranges in ((1, 1), (0, 1), (0, 0)):
            lib.ti_tuning_set(b"tiles_256", on)
            lib.ti_tuning_set(b"two_ranges", ranges)
            outs.append(torch.empty(M, F, device="cuda", dtype=torch.bfloat16))
            ops.linear(a, w, outs[-1], "swiglu")
    finally:
        lib.ti_tuning_reset()
    assert torch.isfinite(outs[0]).all()
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])


# whole rounds by quarters of four or eight wavefronts, the columns left in another tile: of no whole tile and no whole piece of 16 bytes (9717)
@pytest.mark.parametrize("M,F,K", [(1000, 9728, 2560), (800, 9717, 2560), (1792, 9728, 2560), (1300, 6144, 2048), (1300, 12288, 4096), (2304, 12288, 4096)])
def test_gate_up_products_by_quarters_in_two_ranges(ops, M, F, K):  # noqa: F811
    """Rows and weights whose tiles of 256 x 256 are no whole rounds of the units: the bits of one tile of 128 x 128 everywhere."""
    lib = ops.lib("gemm_bf16")
    rest, n_big = ctypes.c_int(), ctypes.c_int()
    tile = lib.ti_gemm_bf16_quarters_ranges(M, F, K, ctypes.byref(rest), ctypes.byref(n_big))
    assert tile in (10, 12) and 0 < n_big.value < F and n_big.value % 128 == 0 and rest.value > 0
    g = torch.Generator(device="cuda").manual_seed(M + F)
    a = torch.randn(M, K, device="cuda", generator=g).to(torch.bfloat16)
    w = (torch.randn(2 * F, K, device="cuda", generator=g) * 0.1).to(torch.bfloat16)
    outs = []
    try:
        for force in (0, 2):
            lib.ti_tuning_set(b"force_tile", force)
            room = torch.full((M * F + 8,), 7.0, device="cuda", dtype=torch.bfloat16)
            ops.linear(a, w, room[:M * F].view(M, F), "swiglu")
            assert bool((room[M * F:] == 7.0).all())
            outs.append(room)
    finally:
        lib.ti_tuning_reset()
    assert torch.isfinite(outs[0]).all() and torch.equal(outs[0], outs[1])


@pytest.mark.parametrize("M,nh,nkv,hd,K,P,norm,rope", [
    (300, 3, 1, 128, 128, 16, True, "table"), (513, 5, 1, 64, 256, 32, True, None), (257, 4, 0, 128, 64, 16, False, "computed"),
    (100, 2, 2, 64, 192, 48, False, "table")])
def test_qkv_product_in_tiles_of_256_by_256(ops, M, nh, nkv, hd, K, P, norm, rope):  # noqa: F811
    """The heads finished in two ranges of 128 columns: whole tiles, a second range beyond the last head, rows that are no
    multiple of the tile.  The bits of the product and the kernel that prepares whole steps."""
    qkv_prepared_case(ops, 512, M, nh, nkv, hd, K, P, norm, rope)


@pytest.mark.parametrize("M,N,K,wide", [
    # both sides of the line: rounds of 256 x 256 nearly full, and ones that have just begun
    (2048, 6144, 2560, 1), (3000, 6144, 2560, 0), (6000, 6144, 2560, 0), (2048, 6144, 4096, 1), (6000, 6144, 4096, 0), (2048, 4096, 2048, 0),
    (3000, 4096, 2048, 1), (6000, 4096, 2048, 0), (4096, 4096, 1024, 1), (2048, 4096, 1024, 0), (3500, 10240, 5120, 0), (2048, 5120, 2048, 1)])
def test_which_qkv_products_take_tiles_of_256_by_256(ops, M, N, K, wide):  # noqa: F811
    """By their costs, at any K."""
    assert ops.lib("gemm_bf16").ti_gemm_bf16_qkv_wide(M, N, K) == wide


@pytest.mark.parametrize("M,nh,nkv,hd,ranges,wide", [(2048, 32, 4, 128, 1, 1), (1900, 70, 5, 64, 1, 1), (3000, 32, 8, 128, 1, 0), (3000, 16, 8, 128, 0, 1)])
def test_qkv_product_as_chosen_with_and_without_tiles_of_256_by_256(ops, M, nh, nkv, hd, ranges, wide):  # noqa: F811
    """Tiles of 256 x 256 where they are chosen, and without them 256-row tiles, with the heads left over in 128-row tiles where `ranges`: the bits
    of the product and the kernel that prepares whole steps."""
    lib, n_big, K = ops.lib("gemm_bf16"), ctypes.c_int(0), 2048
    N = (nh + 2 * nkv) * hd
    assert lib.ti_gemm_bf16_qkv_choice(M, N, K, ctypes.byref(n_big)) == 256 and (0 < n_big.value < N) == ranges
    assert lib.ti_gemm_bf16_qkv_wide(M, N, K) == wide
    try:
        for on in (1, 0):
            lib.ti_tuning_set(b"tiles_256", on)
            qkv_prepared_case(ops, 0, M, nh, nkv, hd, K, 16, True, "table")
    finally:
        lib.ti_tuning_set(b"tiles_256", 1)


@pytest.mark.parametrize("M,N,K", [(1024, 1024, 128), (2048, 512, 128), (512, 2048, 64), (384, 1152, 64)])
def test_dies_blocks_cover_every_tile_once(ops, M, N, K):  # noqa: F811
    """Grids that the eight dies cut by rows, by columns and by both, and one that none of the cuts divides."""
    lib = ops.lib("gemm_bf16")
    g = torch.Generator().manual_seed(M + N)
    a = dev((torch.rand(M, K, generator=g) * 2 - 1).to(torch.bfloat16))
    w = dev((torch.rand(N, K, generator=g) * 2 - 1).to(torch.bfloat16))
    outs = []
    try:
        for tile in (2, 4, 6):
            lib.ti_tuning_set(b"force_tile", tile)
            for order in (0, 1):
                lib.ti_tuning_set(b"die_order", order)
                out = torch.full((M, N), float("nan"), device="cuda")
                ops.linear(a, w, out, "store")
                outs.append(out)
    finally:
        lib.ti_tuning_set(b"force_tile", 0)
        lib.ti_tuning_set(b"die_order", 1)
    for out in outs[1:]:
        assert torch.equal(out, outs[0])
    assert (f64(outs[0]) - ref_linear(a.cpu(), w.cpu())).abs().max() < 2e-5 * K


@pytest.mark.parametrize("M,N,K", [(77, 1024, 3072), (256, 1024, 2048), (512, 2048, 512), (130, 4096, 4096), (700, 1000, 1024),
                                   (2048, 1024, 3072)])
def test_sums_of_a_split_product(ops, M, N, K):  # noqa: F811
    """Products into the residual whose launch is cut into two, four or eight runs of K, or left whole, as their cost says.  The
    norm behind a product whose sums were left adds them to the same bits and has the bits of the norm of their sum."""
    g = torch.Generator().manual_seed(M + N + K)
    a = dev((torch.rand(M, K, generator=g) * 2 - 1).to(torch.bfloat16))
    w = dev((torch.rand(N, K, generator=g) * 2 - 1).to(torch.bfloat16))
    base = dev(torch.randn(M, N, generator=g))
    ref, size = ref_linear(a.cpu(), w.cpu()) + f64(base), f64(a).abs() @ f64(w).abs().T + f64(base).abs()
    for may_defer in (False, True):
        x = base.clone()
        ops.linear(a, w, x, "add", may_defer=may_defer)
        ops.flush()
        assert ((f64(x) - ref).abs() <= (K + 9) * 2.0 ** -24 * size).all()
    nw = dev(torch.rand(N, generator=g) + 0.5)
    normed, want = (torch.empty(M, N, device="cuda", dtype=torch.bfloat16) for _ in range(2))
    ops.rmsnorm(x, nw, 1e-6, want)
    y = base.clone()
    ops.linear(a, w, y, "add", may_defer=True)
    ops.rmsnorm(y, nw, 1e-6, normed)
    assert torch.equal(y, x) and torch.equal(normed, want)


@pytest.mark.parametrize("M,nh,nkv,hd,K", [(65, 16, 8, 128, 64), (129, 6, 2, 64, 128), (200, 4, 1, 128, 320), (512, 16, 8, 128, 192)])
def test_qkv_product_with_prepared_heads_in_tiles_of_64_rows(ops, M, nh, nkv, hd, K):  # noqa: F811
    qkv_prepared_case(ops, 64, M, nh, nkv, hd, K, 16, True, "table")


@pytest.mark.parametrize("M,N,K", [(17, 5120, 17408), (32, 5120, 8192), (64, 5120, 17408)])
def test_large_weights_under_few_rows_keep_eight_runs_of_k(ops, M, N, K):  # noqa: F811
    """17 to 64 rows times a weight that is waited for from memory: eight runs of K, whose sums are within (K + 9) 2^-24 of
    float64 for each of the terms."""
    g = torch.Generator(device="cuda").manual_seed(M)
    a = (torch.rand(M, K, generator=g, device="cuda") * 2 - 1).to(torch.bfloat16)
    w = (torch.rand(N, K, generator=g, device="cuda") * 2 - 1).to(torch.bfloat16)
    x, partial, splits = torch.zeros(M, N, device="cuda"), torch.full((8, M, N), float("nan"), device="cuda"), ctypes.c_int(0)
    lib, ptr = ops.lib("gemm_bf16"), lambda t: ctypes.c_void_p(t.data_ptr())
    rc = lib.ti_gemm_bf16_add_split(ptr(a), ptr(w), ptr(x), M, N, K, ctypes.c_long(K), 1, ptr(partial),
                                    ctypes.c_long(partial.numel() * 4), 1, ctypes.byref(splits), None)
    torch.cuda.synchronize()
    assert rc == 0 and splits.value == 8
    ref, size = a.double() @ w.double().T, a.double().abs() @ w.double().abs().T
    assert ((partial.double().sum(0) - ref).abs() <= (K + 9) * 2.0 ** -24 * size).all()


def test_rows_too_long_for_the_tiled_kernel(ops):  # noqa: F811
    """A row of 2^21 entries: the kernel whose loads have 32-bit offsets inside a tile leaves it to others, split or not.
    Sums of ones and zeros are exact."""
    M, N, K = 17, 64, 1 << 21
    g = torch.Generator(device="cuda").manual_seed(5)
    a = (torch.rand(M, K, generator=g, device="cuda") < 0.5).to(torch.bfloat16)
    w = (torch.rand(N, K, generator=g, device="cuda") < 0.5).to(torch.bfloat16)
    out, partial = torch.empty(M, N, device="cuda"), torch.empty(8, M, N, device="cuda")
    lib, ptr = ops.lib("gemm_bf16"), lambda t: ctypes.c_void_p(t.data_ptr())
    assert lib.ti_gemm_bf16_store_split(ptr(a), ptr(w), ptr(out), M, N, K, ctypes.c_long(K), ptr(partial),
                                        ctypes.c_long(partial.numel() * 4), None) == 3
    ops.linear(a, w, out, "store")
    assert torch.equal(out, (a.float() @ w.float().T).round())
