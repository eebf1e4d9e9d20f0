"""How a decoding step's contexts are shared out over work items: both sides of the lines, and every segment dealt once."""

import pytest


# rows, context, query and KV heads -> items (the plan's segments: a multiple of 8 that holds the context and one more)
@pytest.mark.parametrize("rows,context,heads,kv_heads,items", [
    (1, 40, 2, 1, 8), (1, 4096, 48, 8, 40 * 8), (2, 20011, 48, 8, 160 * 16), (2, 24000, 48, 8, 192 * 16), (2, 24448, 48, 8, 192 * 16),
    (2, 24449, 48, 8, 128 * 16), (2, 40000, 48, 8, 128 * 16), (8, 6016, 48, 8, 48 * 64), (8, 6017, 48, 8, 32 * 64), (39, 700, 48, 8, 7 * 312), (16, 1000, 48, 8, 16 * 128), (16, 3000, 48, 8, 16 * 128),
    (8, 4096, 48, 8, 32 * 64), (16, 2048, 48, 8, 16 * 128), (16, 2049, 48, 8, 16 * 128), (8, 4737, 48, 8, 40 * 64), (8, 4608, 48, 8, 32 * 64),
    (1, 32640, 48, 8, 256 * 8), (1, 32641, 48, 8, 256 * 8), (2, 80000, 12, 2, 512 * 4),
    (40, 700, 48, 8, 320), (64, 1280, 48, 8, 512)])
def test_segments_are_shared_out(rows, context, heads, kv_heads, items):
    from llmx_amd import ops
    plan = ops.attention_plan([1] * rows, [context] * rows, heads, kv_heads, "cpu")
    assert plan.n_items == items and plan.n_shared == 0
    every_segment_once(plan, rows, context, kv_heads)


def every_segment_once(plan, rows, context, kv_heads):
    dealt = {}
    for row, n, head0, _, share, shares, slot, cap in plan.items.tolist():
        assert n == 1 and 0 <= share < shares
        dealt.setdefault((row, head0), []).append(share)
        if shares > 1:
            assert 128 * cap > context and shares <= cap and slot >= 0
    assert len(dealt) == rows * kv_heads and all(sorted(v) == list(range(len(v))) for v in dealt.values())


# unequal rows, head size and window -> items.  An item a segment only where an eighth of the segments that hold keys would be an item's second and
# there are few items without keys: rows that differ little; not many short rows beside a long one, nor rows whose segments an item each has already
@pytest.mark.parametrize("contexts,window,head_dim,items", [
    ([10200] * 3 + [9100], 0, 128, 88 * 32), ([10200, 8000, 8000, 8000], 0, 128, 64 * 32), ([10200] * 3 + [9100], 0, 112, 64 * 32), ([10200] * 3 + [9100], 0, 256, 88 * 32),
    ([16000] + [1000] * 7, 0, 128, 32 * 64), ([6100] + [1000] * 7, 0, 128, 32 * 64), ([4000] * 7 + [4097], 0, 128, 32 * 64), ([5600, 5630, 5500, 5400, 5390, 5640, 5500, 5400], 0, 128, 48 * 64), ([5200, 5230, 5100, 5000, 4990, 5240, 5100, 5000], 0, 128, 32 * 64),
    ([60000] * 8, 5500, 128, 48 * 64), ([60000] * 8, 4096, 128, 32 * 64), ([60000] * 8, 5500, 64, 32 * 64)])
def test_segments_of_unequal_rows_are_shared_out(contexts, window, head_dim, items):
    from llmx_amd import ops
    plan = ops.attention_plan([1] * len(contexts), contexts, 48, 8, "cpu", window, head_dim)
    assert plan.n_items == items
    every_segment_once(plan, len(contexts), min(max(contexts), window + 128 if window else max(contexts)) - 1, 8)


# the rule counts the segments that hold keys: whatever the rows, items of two segments are left only below the eighth, and no plan is more than
# 1.15 times as large as the segments where it has an item for each
@pytest.mark.parametrize("seed", range(40))
def test_what_an_item_a_segment_needs(seed):
    import random
    from llmx_amd import ops
    r = random.Random(seed)
    contexts = [r.randint(50, r.choice([900, 6000, 24000])) for _ in range(r.randint(1, 39))]
    if seed % 2:
        contexts = [contexts[0] + 3000] * len(contexts)
    base, segments = 8 * len(contexts), [-(-c // 128) for c in contexts]
    splits = ops.attention_plan([1] * len(contexts), contexts, 48, 8, "cpu").n_items // base
    before = min(-(-2048 // base), -(-(max(segments) + 1) // 8) * 8)
    assert splits in (before, -(-(max(segments) + 1) // 8) * 8)
    if splits != before:
        assert 8 * sum(max(0, n - before) for n in segments) >= sum(segments) and 8 * splits * len(contexts) <= 3072 and splits * len(contexts) <= 1.15 * sum(segments)
