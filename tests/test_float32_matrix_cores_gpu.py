"""The float32 product and attention on the matrix cores, against float64 and against themselves under other cuts of
the same rows: a row's bits do not depend on the rows beside it."""
import math

import pytest
import torch

from test_kernels_gpu import FakeCtx, View, dev, f64, ops  # noqa: F401  (the fixture)

pytestmark = pytest.mark.gpu

EPS = 2.0 ** -24


@pytest.mark.parametrize("N,K", [(16, 4), (1000, 20), (65, 132), (1024, 1024), (36, 3076)])
def test_product_at_the_edges_of_its_tiles(ops, N, K):  # noqa: F811
    """Rows on either side of every tile's edge, runs of K that end inside a step of 16 or are empty, a last tile of few
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
