"""The 32-bit path's products on the matrix cores: both forms at the sizes where they can go wrong, against float64."""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def ops():
    from llmx_amd import ops as o
    return o


def rnd(*shape, seed=0):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)).to(DEV)


def close(got, want, K):
    """Each product and each addition of a sum of K terms rounds once: at most (K + 1) 2^-24 of the sum of magnitudes; the sums
    here are of random signs, for which sqrt(K) of that holds with room."""
    assert (got.double() - want).abs().max() <= 4 * 2.0 ** -24 * math.sqrt(K) * want.abs().max()


# rows about a strip (16), a tile (64) and the change of form; features about a strip and both tiles; K of one short step, of an
# odd number of steps, with a last step of 4, 8 and 12 values, and whole runs
@pytest.mark.parametrize("M", [1, 15, 17, 64, 65, 300])
@pytest.mark.parametrize("N,K", [(1, 4), (17, 16), (130, 20), (48, 216), (3072, 2048), (4099, 604), (32768, 48), (2500, 400)])
def test_rows_features_and_runs(M, N, K):
    o = ops()
    a, w = rnd(M, K), rnd(N, K, seed=1)
    o.take_launches()
    c = torch.full((M, N), float("nan"), device=DEV)
    o.gemm(a, w, c)
    ran = o.take_launches()
    assert ran.get("gemm_generic") == 1 and ran.get("gemm_generic.stream", 0) + ran.get("gemm_generic.tiles", 0) == 1
    close(c, a.double() @ w.double().T, K)
    few = torch.empty(1, N, device=DEV)
    o.gemm(a[M - 1:].contiguous(), w, few)
    assert torch.equal(few[0], c[M - 1]), "a row's bits depend on the rows beside it"
    old = rnd(M, N, seed=2)
    added = old.clone()
    o.gemm(a, w, added, o.EPI_ADD)
    assert torch.equal(added, old + c)
    if N % 2 == 0:
        gated = torch.empty(M, N // 2, device=DEV)
        o.gemm(a, w, gated, o.EPI_SWIGLU)
        gate, up = c[:, :N // 2].double(), c[:, N // 2:].double()
        want = gate * torch.sigmoid(gate) * up
        assert (gated.double() - want).abs().max() <= 8 * 2.0 ** -23 * want.abs().max()
    bias = rnd(N, seed=3)
    biased = torch.empty(M, N, device=DEV)
    o.gemm(a, w, biased, act=(o.ACT_BIAS, bias))
    assert torch.equal(biased, c + bias)


@pytest.mark.parametrize("counts", [[1, 0, 3, 16], [0, 0, 17, 1], [70, 0, 200, 130], [64, 129, 65, 63]])
@pytest.mark.parametrize("N,K", [(40, 36), (136, 208), (2688, 2048)])
def test_groups_of_rows(counts, N, K):
    """Groups with no rows, one, a tile's and one more; rows gathered two pairs a row and scattered through the list."""
    o = ops()
    G, pairs = len(counts), sum(counts)
    order = torch.randperm(pairs, generator=torch.Generator().manual_seed(5)).to(torch.int32).to(DEV)
    offsets = torch.tensor([0] + torch.tensor(counts).cumsum(0).tolist(), dtype=torch.int32, device=DEV)
    a, w = rnd((pairs + 1) // 2, K), rnd(G, 2 * N, K, seed=1)
    c, gated = torch.full((pairs, 2 * N), float("nan"), device=DEV), torch.full((pairs, N), float("nan"), device=DEV)
    o.grouped_gemm(a, w, c, offsets, order, 2)
    o.grouped_gemm(a, w, gated, offsets, order, 2, o.EPI_SWIGLU)
    for g in range(G):
        rows = order[int(offsets[g]):int(offsets[g + 1])].long()
        if not len(rows):
            continue
        close(c[rows], a[rows // 2].double() @ w[g].double().T, K)
        alone = torch.empty(len(rows), 2 * N, device=DEV)
        o.gemm(a[rows // 2].contiguous(), w[g], alone)
        assert torch.equal(alone, c[rows]), "a group's rows have other bits than the same product alone"
        gate, up = c[rows, :N].double(), c[rows, N:].double()
        want = gate * torch.sigmoid(gate) * up
        assert (gated[rows].double() - want).abs().max() <= 8 * 2.0 ** -23 * want.abs().max()


def test_operands_that_allow_no_wide_loads_take_the_universal_product():
    o = ops()
    w = rnd(32, 20)
    for a in (rnd(3 * 20 + 1)[1:].view(3, 20), rnd(3, 20)):
        c = torch.empty(3, 32, device=DEV)
        o.take_launches()
        o.gemm(a, w, c)
        ran = o.take_launches()
        assert ("gemm_generic.stream" in ran) == (a.data_ptr() % 16 == 0)
        close(c, a.double() @ w.double().T, 20)
    a, w, c = rnd(5, 30), rnd(32, 30), torch.empty(5, 32, device=DEV)
    o.gemm(a, w, c)
    assert not any(k.startswith("gemm_generic.") for k in o.take_launches())
    close(c, a.double() @ w.double().T, 30)
