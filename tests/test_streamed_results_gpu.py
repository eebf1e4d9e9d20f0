"""Tiled products of many megabytes of float32 results, kept in the caches and sent past them in whole lines: the bits of smaller products and of kept
results, and no element left out or touched twice."""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def rnd(*shape, seed=0):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)).to(DEV, torch.bfloat16)


# features that end in the first and in the second half of a line, on its end, and 2 past a multiple of 4 (quads that are not aligned); rows that
# end in the first and the second eight of a tile of 16
@pytest.mark.parametrize("M,N,K", [(9, 200064, 64), (61, 32772, 64), (64, 32788, 192), (57, 32770, 64), (1999, 1028, 128), (1537, 1024, 64), (1535, 1024, 64),
                                   (2041, 4132, 128), (2047, 4128, 256), (1100, 10880, 64)])
def test_rows_of_many_megabytes(M, N, K):
    from llmx_amd import ops
    a, w = rnd(M, K), rnd(N, K, seed=1)
    held = torch.full((M + 2, N), float("nan"), device=DEV)
    ops.gemm(a, w, held[1:-1])
    assert bool(held[0].isnan().all()) and bool(held[-1].isnan().all())
    c = held[1:-1]
    rows = sorted({0, 7, 8, 15 % M, 63 % M, M // 2, M - 9, M - 8, M - 1})
    few = torch.empty(len(rows), N, device=DEV)
    ops.gemm(a[rows].contiguous(), w, few)
    assert torch.equal(few, c[rows])
    want = a.double() @ w.double().T
    # float32 sums of K exact products of random sign stay about sqrt(K), K roundings of them by up to 2^-24 add up by their square root; 16 times that over
    # all the elements
    assert (c.double() - want).abs().max() <= 4 * 2.0 ** -24 * math.sqrt(K) * math.sqrt(K) * 4


@pytest.mark.parametrize("N,K", [(520, 1536), (388, 1024), (1028, 2048), (514, 1024), (640, 512)])
def test_routed_rows_of_many_megabytes(N, K):
    from llmx_amd import ops
    X = 24
    n = [(0, 1, 7, 8, 63, 64, 65, 129, 300, 500)[i % 10] for i in range(X - 1)]
    n.append(max(4096, (7 << 20) // (4 * N)) - sum(n))
    P = sum(n)
    gen = torch.Generator().manual_seed(N)
    ids = torch.repeat_interleave(torch.arange(X), torch.tensor(n))[torch.randperm(P, generator=gen)].to(torch.int32).view(P, 1).to(DEV)
    found, offsets, active = (torch.zeros(m, dtype=torch.int32, device=DEV) for m in (X, X + 1, X))
    pairs, n_active, ticket, stats = (torch.zeros(m, dtype=torch.int32, device=DEV) for m in (P, 1, 1, 2))
    ops.moe_align(ids, X, found, offsets, pairs, active, n_active, tile_stats=stats, ticket=ticket)
    a, w = rnd(P, K), rnd(X, N, K, seed=1)
    got = []
    for choice, more in ((0, {}), (15, {}), (15, {"ticket": ticket})):
        stats[1] = choice
        c = torch.full((P, N), float("nan"), device=DEV)
        ops.grouped_gemm(a, w, c, offsets, pairs, 1, ops.EPI_STORE, tile_stats=stats, **more)
        got.append(c)
    for e in range(X):
        rows = pairs[int(offsets[e]):int(offsets[e + 1])].long()
        if not len(rows):
            continue
        alone = torch.empty(len(rows), N, device=DEV)
        ops.gemm(a[rows], w[e].contiguous(), alone)       # the expert's own product, in runs of K of the same shape
        for c in got:
            assert torch.equal(c[rows], alone)


FORMS = {"64": {"gemm_tile.64": 1}, "64_deep": {"gemm_tile.64": 1, "gemm_tile.64_deep": 1}, "wide": {"gemm_tile.wide": 1}}


# Every dense form, K in one run and in several, a last one shorter than the others (1,728 values: 3 runs of 448 and one of 384).  The results are `wide`
# features apart: rows of whole lines leave in lines, the same 4 values wider are kept, and so are smaller results.  Features that end in the first and the
# second half of a line and on its end, in a partial tile; rows that end in the first and the second eight of 16.
@pytest.mark.parametrize("M,N,K,runs,wide,form,lines", [
    (1601, 8192, 64, 1, 8192, "wide", True), (1543, 8224, 128, 1, 8256, "wide", True), (1999, 8196, 1536, 4, 8224, "wide", True), (2041, 8212, 1728, 4, 8224, "wide", True),
    (1544, 8224, 1728, 4, 8224, "wide", True), (1535, 8192, 1536, 4, 8192, "wide", False),
    (24, 131076, 2048, 1, 131104, "64", True), (57, 131072, 2048, 2, 131072, "64", True), (191, 22016, 12288, 2, 22016, "64", True), (19, 131072, 2048, 1, 131072, "64", False),
    (250, 12260, 21952, 1, 12288, "64_deep", True), (321, 8208, 32768, 4, 8224, "64_deep", True), (328, 8192, 32768, 8, 8192, "64_deep", True), (319, 8192, 32768, 4, 8192, "64_deep", False)])
def test_every_form_stores_lines(M, N, K, runs, wide, form, lines):
    from llmx_amd import ops
    gen = torch.Generator(device=DEV).manual_seed(M)
    a, w = (torch.randn(n, K, generator=gen, device=DEV, dtype=torch.bfloat16) for n in (M, N))
    got = []
    for ldc in (wide, wide + 4):
        held = torch.full((M + 2, ldc), float("nan"), device=DEV)
        ops.take_launches()
        ops._check(ops.lib().llmx_gemm_tile(a.data_ptr(), w.data_ptr(), held[1:].data_ptr(), ops._code(held.dtype), M, N, K, K, ldc, ops.EPI_STORE, runs, 0, 0, 0, 0, 1, 0, 0, 0, 0,
                                            0, 0, 0, 0.0, 0, 0, 0, ops._stream()), "gemm_tile")
        assert ops.take_launches(details=True) == {**FORMS[form], **({"gemm_tile+lines": 1} if lines and ldc == wide else {})}
        assert bool(held[0].isnan().all()) and bool(held[-1].isnan().all()) and bool(held[:, N:].isnan().all())
        got.append(held[1:-1, :N])
    assert torch.equal(*got)
    cols = torch.tensor(sorted({0, 3, 15, 16, 31, 32, 127, 128, 255, 256, N // 2, N - 33, N - 17, N - 16, N - 5, N - 4, N - 1}), device=DEV)
    exact, sizes = a.double() @ w[cols].double().T, a.double().abs() @ w[cols].double().abs().T
    # K products, exact in float32, and K + runs additions, each of which rounds what it gives by 2^-24 of it at most, and no sum is larger than the sizes'
    assert bool(((got[0][:, cols].double() - exact).abs() <= (K + runs) * 2.0 ** -24 * sizes).all())


# the routed forms: 128 rows by four waves, the wide one with and without tickets, 64 rows; K in one run and in several, a last one that is shorter
@pytest.mark.parametrize("N,K,forms,lines", [
    (640, 512, {"gemm_tile.grouped_128": 3, "gemm_tile.grouped_64": 3}, 6), (544, 1536, {"gemm_tile.grouped_128": 3, "gemm_tile.grouped_64": 3, "gemm_tile.grouped_wide": 0}, 6),
    (512, 1728, {"gemm_tile.grouped_128": 3, "gemm_tile.grouped_64": 3}, 6), (1056, 2048, {"gemm_tile.grouped_wide": 3, "gemm_tile.grouped_64": 3}, 6),
    (1028, 2048, {"gemm_tile.grouped_wide": 3, "gemm_tile.grouped_64": 3}, 0), (480, 1536, {"gemm_tile.grouped_128": 3, "gemm_tile.grouped_64": 3}, 0)])
def test_routed_forms_store_lines(N, K, forms, lines):
    from llmx_amd import ops
    ops.take_launches()
    test_routed_rows_of_many_megabytes(N, K)
    ran = ops.take_launches(details=True)
    assert ran.get("gemm_tile+lines", 0) == lines and {k: ran.get(k, 0) for k in forms} == forms
