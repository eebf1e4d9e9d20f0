"""Routed tiled products whose workgroups take tile after tile by tickets, against a workgroup a tile: the same bits, and the counter 0 again."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# fewer tiles than CUs and many rounds of them; experts without rows, of one row, of whole tiles and one more, of few and many rows; a last strip that
# is partial; K about the forms' bounds
@pytest.mark.parametrize("N,K", [(256, 1024), (520, 1088), (1024, 2048), (2056, 2560)])
@pytest.mark.parametrize("counts", ["even", "uneven", "few"])
def test_tickets_change_no_bit(counts, N, K):
    from llmx_amd import ops
    X = 40
    gen = torch.Generator().manual_seed(N + K)
    if counts == "even":
        n = [120 + i % 17 for i in range(X)]
    elif counts == "uneven":
        n = [(0, 1, 64, 65, 128, 129, 300, 777)[i % 8] for i in range(X)]
    else:
        n = [0] * X
        n[3], n[39] = 4095, 1
    P = sum(n)
    ids = torch.repeat_interleave(torch.arange(X), torch.tensor(n))[torch.randperm(P, generator=gen)].to(torch.int32).view(P, 1).to(DEV)
    found, offsets, active = (torch.zeros(m, dtype=torch.int32, device=DEV) for m in (X, X + 1, X))
    pairs, n_active, ticket, stats = (torch.full((m,), -7, dtype=torch.int32, device=DEV) for m in (P, 1, 1, 2))
    ops.moe_align(ids, X, found, offsets, pairs, active, n_active, tile_stats=stats, ticket=ticket)
    assert int(ticket) == 0
    held = [c for c in n if c]
    assert int(stats[1]) == ops.lib().llmx_tile_choice_tickets(P, sum(-(-c // 128) for c in n), sum(-(-c // 64) for c in n), len(held))
    a = torch.randn(P, K, generator=gen).to(DEV, torch.bfloat16)
    w = (torch.randn(X, N, K, generator=gen) * 0.05).to(DEV, torch.bfloat16)
    for choice in (15, int(stats[1])):
        stats[1] = choice
        for epi, shape, dtype in ((ops.EPI_STORE, N, torch.float32), (ops.EPI_SWIGLU, N // 2, torch.bfloat16)):
            want, got = (torch.full((P, shape), float("nan"), dtype=dtype, device=DEV) for _ in range(2))
            ops.grouped_gemm(a, w, want, offsets, pairs, 1, epi, tile_stats=stats)
            for _ in range(2):
                got.fill_(float("nan"))
                ops.grouped_gemm(a, w, got, offsets, pairs, 1, epi, tile_stats=stats, ticket=ticket)
                assert int(ticket) == 0
                assert torch.equal(got, want)
            if epi == ops.EPI_STORE:
                rows = pairs[int(offsets[3]):int(offsets[3]) + 64].long()
                exact = a[rows].double() @ w[3].double().T
                # float32 sums of K exact products of random sign
                assert (got[rows].double() - exact).abs().max() <= 4 * 2.0 ** -24 * K ** 0.5 * exact.abs().max() * 4


# groups beyond a wave's lanes and beyond the scan's 512, those about 64 and 512 and the last ones without rows; against the form of 64 rows,
# which finds its groups in another way, and against float64
@pytest.mark.parametrize("X,K", [(65, 1024), (256, 2048), (600, 1024), (1100, 2048)])
def test_the_groups_of_tiles_are_found(X, K):
    from llmx_amd import ops
    N = 520
    gen = torch.Generator().manual_seed(X)
    n = [(9, 0, 130, 1, 64, 0, 17)[i % 7] if X > 100 else 40 + 30 * (i % 4) for i in range(X)]
    for i in (0, 1, 62, 63, 64, 510, 511, 512, 513, X - 2, X - 1):
        if i < X:
            n[i] = 0 if i in (1, 63, 64, 511, 512, X - 1) else 131
    P = sum(n)
    assert P >= ops.TILE_STATS_MIN_PAIRS
    ids = torch.repeat_interleave(torch.arange(X), torch.tensor(n))[torch.randperm(P, generator=gen)].to(torch.int32).view(P, 1).to(DEV)
    found, offsets, active = (torch.zeros(m, dtype=torch.int32, device=DEV) for m in (X, X + 1, X))
    pairs, n_active, ticket, stats = (torch.full((m,), -7, dtype=torch.int32, device=DEV) for m in (P, 1, 1, 2))
    # more groups than the grouping counts tiles for: the numbers are set by hand
    ops.moe_align(ids, X, found, offsets, pairs, active, n_active, tile_stats=stats if X <= 1024 else None, ticket=ticket if X <= 1024 else None)
    assert found.tolist() == n
    ticket.zero_()
    a = torch.randn(P, K, generator=gen).to(DEV, torch.bfloat16)
    w = torch.empty(X, N, K, dtype=torch.bfloat16, device=DEV).normal_(0.0, 0.05, generator=torch.Generator(DEV).manual_seed(X))
    held = [e for e in range(X) if n[e]]
    for epi, width, dtype in ((ops.EPI_STORE, N, torch.float32), (ops.EPI_SWIGLU, N // 2, torch.float32)):
        want, got, plain = (torch.full((P, width), float("nan"), dtype=dtype, device=DEV) for _ in range(3))
        for out, choice, more in ((want, 0, {}), (got, 15, {"ticket": ticket}), (plain, 15, {})):
            stats[1] = choice
            ops.grouped_gemm(a, w, out, offsets, pairs, 1, epi, tile_stats=stats, **more)
            assert int(ticket) == 0
        assert torch.equal(got, want) and torch.equal(plain, want)
        for e in {held[0], held[-1], *(min(held, key=lambda h: abs(h - b)) for b in (62, 65, 510, 513))}:
            rows = pairs[int(offsets[e]):int(offsets[e + 1])].long()
            exact = a[rows].double() @ w[e].double().T
            tol = 4 * 2.0 ** -24 * K ** 0.5 * exact.abs().max()         # float32 sums of K exact products of random sign
            if epi == ops.EPI_SWIGLU:
                gate, up = exact[:, :width], exact[:, width:]
                exact = gate * torch.sigmoid(gate) * up
                tol = tol * (1.1 * up.abs().max() + gate.abs().max()) + 2.0 ** -21 * exact.abs().max()      # |silu'| <= 1.1, |silu(g)| <= |g|; the unit's own roundings
            assert (got[rows].double() - exact).abs().max() <= tol, (epi, e)


def test_a_dense_product_takes_no_tickets():
    """The entry point that takes a ticket, called for a dense product of more tiles than there are CUs: every tile is stored."""
    from llmx_amd import ops
    M, N, K = 2568, 4104, 128
    gen = torch.Generator().manual_seed(1)
    a, w = (torch.randn(n, K, generator=gen).to(DEV, torch.bfloat16) for n in (M, N))
    want, got = (torch.full((M, N), float("nan"), device=DEV) for _ in range(2))
    ticket = torch.zeros(1, dtype=torch.int32, device=DEV)
    ops.gemm(a, w, want)
    args = (M, N, K, K, N, ops.EPI_STORE, ops._split_k(-(-N // 16), K), 0, 0, 0, 0, 1, 0, 0, 0, 0)
    assert ops.lib().llmx_gemm_tile_tickets(a.data_ptr(), w.data_ptr(), got.data_ptr(), ops._code(got.dtype), *args, ticket.data_ptr(), 0, 0, 0, 0, 0.0, 0, 0, 0,
                                            torch.cuda.current_stream().cuda_stream) == 0
    torch.cuda.synchronize()
    assert bool(want.isfinite().all()) and torch.equal(got, want) and int(ticket) == 0
