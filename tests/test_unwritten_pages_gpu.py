"""Decode attention over pages of several 16-key tiles: what was never written behind a request's last tile reaches no result."""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# few requests (contexts shared out over many waves or workgroups) and many (a wave walks its context); contexts that end in a page's first
# tile, in its last, at a segment's and a page's edge
@pytest.mark.parametrize("requests,Hkv", [(3, 2), (40, 8)])
@pytest.mark.parametrize("D,page,window", [(64, 32, 0), (128, 64, 0), (128, 48, 200), (160, 64, 0), (208, 16, 0), (224, 64, 0), (240, 16, 0), (256, 32, 100)])
def test_keys_past_the_end_are_not_numbers(requests, Hkv, D, page, window):
    from llmx_amd import ops
    contexts = [(1, 15, 17, 33, 96, 128, 129, 250, 257, 400, 513)[i % 11] for i in range(requests)] if requests > 3 else [5, 145, 390]
    gen = torch.Generator().manual_seed(D + page)
    blocks = [-(-n // page) for n in contexts]
    tables = torch.full((requests, max(blocks)), -1, dtype=torch.int32)
    pages = (torch.randperm(sum(blocks), generator=gen) + 1).to(torch.int32)      # page 0 is nobody's
    k = (torch.randn(1 + sum(blocks), Hkv, page, D, generator=gen) * 0.5).bfloat16()
    v = torch.randn(1 + sum(blocks), Hkv, D, page, generator=gen).bfloat16()
    k_bad, v_bad = k.clone(), v.clone()
    k_bad[0], v_bad[0] = float("nan"), float("inf")
    at = 0
    for i, n in enumerate(contexts):
        tables[i, :blocks[i]] = pages[at:at + blocks[i]]
        at += blocks[i]
        last, written = int(tables[i, blocks[i] - 1]), -(-((n - 1) % page + 1) // 16) * 16
        k_bad[last, :, written:], v_bad[last, :, :, written:] = float("nan"), float("inf")
        if window:      # pages that fell out of the window are given back
            tables[i, :max(0, n - window) // page] = -1
    q = torch.randn(requests, 2 * Hkv * D, generator=gen).to(DEV, torch.bfloat16)
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    plan = ops.attention_plan([1] * requests, contexts, 2 * Hkv, Hkv, DEV, window)
    out = []
    ops.take_launches()
    for kc, vc in ((k, v), (k_bad, v_bad)):
        out.append(torch.full_like(q, float("nan")))
        ops.paged_attention(q, kc.to(DEV), vc.to(DEV), i32([n - 1 for n in contexts]), i32(list(range(requests))), tables.to(DEV), out[-1],
                            1.0 / math.sqrt(D), 2 * Hkv, window, plan=plan)
    ran = ops.take_launches()
    assert ran.get("attention.direct", 0) == (2 if requests > 3 else 0), ran
    assert bool(out[0].isfinite().all()) and torch.equal(out[1], out[0])
    for i in range(0, requests, 7):         # alone a request's context is shared out: the same bits
        one = torch.empty_like(q[:1])
        ops.paged_attention(q[i:i + 1].contiguous(), k.to(DEV), v.to(DEV), i32([contexts[i] - 1]), i32([0]), tables[i:i + 1].contiguous().to(DEV), one,
                            1.0 / math.sqrt(D), 2 * Hkv, window, plan=ops.attention_plan([1], [contexts[i]], 2 * Hkv, Hkv, DEV, window))
        assert torch.equal(one[0], out[0][i]), f"request {i}"
