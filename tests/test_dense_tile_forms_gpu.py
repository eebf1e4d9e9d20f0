"""Dense tiled products at the edges of their forms: three tiles deep, strips handed to XCDs in runs, runs of K apart."""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def rnd(*shape, seed=0):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)).to(DEV, torch.bfloat16)


# K of one, two, three and more tiles of 64 (fewer than the form is deep, as many, more); 512 and 513 tiles of 64 rows; strips in and out
# of multiples of 8, a last one that is partial; rows that end inside a tile; the head's rows about 64
@pytest.mark.parametrize("M,N,K", [(70, 256, 64), (70, 256, 128), (130, 1160, 192), (2048, 2048, 256), (2049, 2048, 256), (1999, 2200, 384),
                                   (700, 10880, 128), (65, 17 * 256 + 8, 768), (64, 65536, 64), (65, 65536, 64), (1600, 3072, 4096), (300, 2048, 8192)])
def test_rows_have_the_bits_they_have_alone(M, N, K):
    from llmx_amd import ops
    a, w = rnd(M, K), rnd(N, K, seed=1)
    c = torch.full((M, N), float("nan"), device=DEV)
    ops.gemm(a, w, c)
    want = a[::37].double() @ w.double().T
    # float32 sums of K exact products of random sign: each addition rounds once
    assert (c[::37].double() - want).abs().max() <= 4 * 2.0 ** -24 * math.sqrt(K) * math.sqrt(K) * 4
    rows = sorted({0, 15, 63, 64 % M, M // 2, M - 2, M - 1})
    few = torch.empty(len(rows), N, device=DEV)
    ops.gemm(a[rows].contiguous(), w, few)
    assert torch.equal(few, c[rows]), "a row's bits depend on the form its product took"
    apart = torch.empty(M, N, device=DEV)
    ops.gemm(a, w, apart, scratch=lambda name, shape, dtype: torch.empty(shape, dtype=dtype, device=DEV))
    assert torch.equal(apart, c)
    if N % 16 == 0:
        gated, few = torch.empty(M, N // 2, dtype=torch.bfloat16, device=DEV), torch.empty(len(rows), N // 2, dtype=torch.bfloat16, device=DEV)
        ops.gemm(a, w, gated, ops.EPI_SWIGLU)
        ops.gemm(a[rows].contiguous(), w, few, ops.EPI_SWIGLU)
        assert torch.equal(few, gated[rows])
