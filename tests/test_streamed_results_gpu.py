"""Tiled products whose float32 results go past the caches in whole lines: the bits of smaller products, and no element left out or touched twice."""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def rnd(*shape, seed=0):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)).to(DEV, torch.bfloat16)


# features that end in the first and in the second half of a line, on its end, and 2 past a multiple of 4 (quads that are not aligned); rows that
# end in the first and the second eight of a tile of 16; the 64-row forms, two and three tiles deep, and the wide one; just above and below the bytes
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
    # float32 sums of K exact products of random sign: each addition rounds once
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
