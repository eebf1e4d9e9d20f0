"""How a decoding step's contexts are shared out over work items: both sides of the lines, and every segment dealt once."""

import pytest


# rows, context, query and KV heads -> items (the plan's segments: a multiple of 8 that holds the context and one more)
@pytest.mark.parametrize("rows,context,heads,kv_heads,items", [
    (1, 40, 2, 1, 8), (1, 4096, 48, 8, 40 * 8), (2, 20011, 48, 8, 160 * 16), (2, 24000, 48, 8, 192 * 16), (2, 24448, 48, 8, 192 * 16),
    (2, 24449, 48, 8, 128 * 16), (2, 40000, 48, 8, 128 * 16), (8, 6016, 48, 8, 48 * 64), (8, 6017, 48, 8, 32 * 64), (39, 700, 48, 8, 8 * 312), (16, 1000, 48, 8, 16 * 128), (16, 3000, 48, 8, 16 * 128),
    (40, 700, 48, 8, 320), (64, 1280, 48, 8, 512)])
def test_segments_are_shared_out(rows, context, heads, kv_heads, items):
    from llmx_amd import ops
    plan = ops.attention_plan([1] * rows, [context] * rows, heads, kv_heads, "cpu")
    assert plan.n_items == items and plan.n_shared == 0
    dealt = {}
    for row, n, head0, _, share, shares, slot, cap in plan.items.tolist():
        assert n == 1 and 0 <= share < shares
        dealt.setdefault((row, head0), []).append(share)
        if shares > 1:
            assert 128 * cap > context and shares <= cap and slot >= 0
    assert len(dealt) == rows * kv_heads and all(sorted(v) == list(range(len(v))) for v in dealt.values())
