"""The grouping's ranks (ballots and a byte a wave) and the choice of tiles it hands on."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("n_experts", [1, 2, 5, 64, 255, 256, 257, 1024])
@pytest.mark.parametrize("T,k", [(1, 1), (63, 1), (64, 1), (65, 1), (128, 8), (129, 8), (700, 5), (2100, 8), (2200, 8)])
def test_pairs_grouped_in_order(n_experts, T, k):
    from llmx_amd import ops
    g = torch.Generator().manual_seed(n_experts + T)
    spread = torch.randint(0, n_experts, (T, k), generator=g)
    crowded = torch.zeros(T, k, dtype=torch.long) + (n_experts - 1)
    none = spread.clone()
    none[torch.rand(T, k, generator=g) < 0.3] = -1
    for ids in (spread, crowded, none):
        flat = ids.flatten()
        counts, offsets = torch.full((n_experts,), -5, dtype=torch.int32, device=DEV), torch.full((n_experts + 1,), -5, dtype=torch.int32, device=DEV)
        pairs = torch.full((T * k,), -5, dtype=torch.int32, device=DEV)
        active, n_active = torch.full((n_experts,), -5, dtype=torch.int32, device=DEV), torch.full((1,), -5, dtype=torch.int32, device=DEV)
        stats = torch.full((2,), -5, dtype=torch.int32, device=DEV)
        ops.moe_align(ids.to(torch.int32).to(DEV), n_experts, counts, offsets, pairs, active, n_active, tile_stats=stats)
        want = torch.bincount(flat[flat >= 0], minlength=n_experts)
        held = int(want.sum())
        assert torch.equal(counts.cpu().long(), want)
        assert torch.equal(offsets.cpu().long(), torch.cat([torch.zeros(1, dtype=torch.long), want.cumsum(0)]))
        assert torch.equal(pairs[:held].cpu().long(), torch.argsort(torch.where(flat >= 0, flat, n_experts), stable=True)[:held])
        assert int(n_active) == int((want > 0).sum()) and torch.equal(active[:int(n_active)].cpu().long(), torch.nonzero(want > 0).flatten())
        if T * k >= ops.TILE_STATS_MIN_PAIRS:
            n128, n64, held = int(((want + 127) // 128).sum()), int(((want + 63) // 64).sum()), int((want > 0).sum())
            assert int(stats[0]) == n128
            assert int(stats[1]) == (0 if 200 * n128 <= 84 * held + 100 * n64 or 100 * n128 <= 61 * n64 else 1 << 30)
