"""Weight-streaming bf16 products at the edges of their rounds: waves with no pair of steps, one, an odd and an even number, an odd step, a
last step of fewer than 32 values, rows whose lines are not whole, strips that end early."""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def rnd(*shape, seed=0, dtype=torch.bfloat16):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)).to(DEV, dtype)


def close(got, want, K):
    """A float32 sum of K exact products of random sign, each addition rounding once."""
    assert (got.double() - want).abs().max() <= 4 * 2.0 ** -24 * math.sqrt(K) * want.abs().max() + 1e-6


SIZES = [(16, 8), (17, 32), (40, 40), (16, 64), (24, 96), (31, 104), (48, 128), (16, 160), (33, 192), (1000, 320), (264, 640), (130, 1536), (3072, 1536),
         (520, 2688), (96, 2056), (4100, 3072)]


@pytest.mark.parametrize("N,K", SIZES)
@pytest.mark.parametrize("M", [1, 4, 16])
def test_rows_have_the_bits_the_tiles_give(M, N, K):
    from llmx_amd import ops
    a, w = rnd(70, K), rnd(N, K, seed=1)
    many, c = torch.empty(70, N, device=DEV), torch.full((M, N), float("nan"), device=DEV)
    ops.gemm(a, w, many)
    ops.take_launches()
    ops.gemm(a[:M].contiguous(), w, c)
    assert ops.take_launches() == {"gemm_skinny": 1}
    close(c, a[:M].double() @ w.double().T, K)
    assert torch.equal(c, many[:M])
    added = torch.ones(M, N, device=DEV)
    ops.gemm(a[:M].contiguous(), w, added, ops.EPI_ADD)
    assert torch.equal(added, c + 1.0)
    bias = rnd(N, seed=2, dtype=torch.float32)
    ops.gemm(a[:M].contiguous(), w, added, act=(ops.ACT_BIAS, bias))
    assert torch.equal(added, c + bias)
    if N % 2 == 0:
        gated = torch.full((M, N // 2), float("nan"), device=DEV)
        ops.gemm(a[:M].contiguous(), w, gated, ops.EPI_SWIGLU)
        both = a[:M].double() @ w.double().T
        gate, up = both[:, :N // 2], both[:, N // 2:]
        want = gate * torch.sigmoid(gate) * up
        # the two sums' errors (see close), carried on by |silu'| <= 1.1 and |silu(g)| <= |g|, and the unit's own float32 roundings
        bound = 4 * 2.0 ** -24 * math.sqrt(K) * both.abs().max() * (1.1 * up.abs() + gate.abs()) + 2.0 ** -21 * want.abs() + 1e-6
        assert ((gated.double() - want).abs() <= bound).all()
    if M <= 4 and K % 8 == 0 and M * K * 2 <= 32768:
        x, nw = rnd(M, K, seed=3, dtype=torch.float32), rnd(K, seed=4, dtype=torch.float32)
        h, formed = torch.empty(M, K, dtype=torch.bfloat16, device=DEV), torch.full((M, N), float("nan"), device=DEV)
        ops.rmsnorm(x, nw, 1e-6, h)
        ops.gemm(h, w, c)
        ops.gemm(ops.NormedRows(x, nw, 1e-6), w, formed)
        assert torch.equal(formed, c)


# groups without rows, of one row, of several chunks of 16, and lists that end inside a chunk
@pytest.mark.parametrize("N,K", [(16, 8), (40, 96), (48, 192), (130, 320), (256, 1536), (264, 2688), (512, 3072)])
def test_grouped_rows_are_the_dense_ones(N, K):
    from llmx_amd import ops
    G, counts = 6, [1, 0, 17, 2, 0, 33]
    P = sum(counts)
    w, a = rnd(G, N, K, seed=1), rnd(P, K)
    offsets = torch.tensor([0] + torch.tensor(counts).cumsum(0).tolist(), dtype=torch.int32, device=DEV)
    pairs = torch.randperm(P, generator=torch.Generator().manual_seed(5)).to(DEV, torch.int32)
    active = torch.tensor([0, 2, 3, 5, 77777, -5], dtype=torch.int32, device=DEV)      # what lies beyond the groups that have rows is not used
    n_active = torch.tensor([4], dtype=torch.int32, device=DEV)
    c = torch.full((P, N), float("nan"), device=DEV)
    ops.take_launches()
    ops.grouped_gemm(a, w, c, offsets, pairs, 1, ops.EPI_STORE, active, n_active, token_rows=1)
    assert ops.take_launches() == {"gemm_skinny.grouped": 1}
    at = 0
    for g, n in enumerate(counts):
        rows = pairs[at:at + n].long()
        at += n
        if n:
            dense = torch.empty(n, N, device=DEV)
            ops.gemm(a[rows].contiguous(), w[g].contiguous(), dense)
            close(dense, a[rows].double() @ w[g].double().T, K)
            assert torch.equal(c[rows], dense)


# waves with no round, part of one, one and more, lines that are whole and not, strips that end early
@pytest.mark.parametrize("N,K", [(16, 16), (40, 32), (17, 64), (130, 96), (48, 160), (264, 288), (100, 672), (2050, 1344), (4100, 2688)])
@pytest.mark.parametrize("M", [1, 4, 16])
def test_float32_rows_have_the_bits_the_tiles_give(M, N, K):
    from llmx_amd import ops
    a, w = rnd(80, K, dtype=torch.float32), rnd(N, K, seed=1, dtype=torch.float32)
    many, c = torch.empty(80, N, device=DEV), torch.full((M, N), float("nan"), device=DEV)
    ops.gemm(a, w, many)
    ops.take_launches()
    ops.gemm(a[:M].contiguous(), w, c)
    assert ops.take_launches() == {"gemm_generic": 1, "gemm_generic.stream": 1}
    close(c, a[:M].double() @ w.double().T, K)
    assert torch.equal(c, many[:M])
