"""The delta rule with one decay a key channel: its step of single tokens against preparation and scan as launches of their own,
and the preparation of many rows against that of few."""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


# (heads, key groups, key channels, value channels, taps): key channels at and beside each width of a workgroup (64, 128, 256),
# value channels short of a tile and over several workgroups, no convolution, slots whose size is no multiple of four floats
@pytest.mark.parametrize("H,G,D,V,taps", [(4, 2, 16, 24, 3), (3, 3, 5, 7, 1), (2, 1, 64, 64, 4), (6, 2, 65, 33, 2), (2, 1, 128, 128, 4), (1, 1, 129, 1, 8), (1, 1, 256, 100, 4)])
@pytest.mark.parametrize("entries", [1, 9])
def test_a_single_token_has_the_bits_of_preparation_and_scan(H, G, D, V, taps, entries):
    from llmx_amd import ops

    gen = torch.Generator().manual_seed(H * 1000 + D * 10 + taps)
    rand = lambda *shape: torch.randn(*shape, generator=gen).cuda()
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")
    C, T = 2 * G * D + H * V, entries
    matrix = ops.state_matrix_size(H, D, V)
    stride = -(-(matrix + (taps - 1) * C) // 4) * 4
    pre, conv, low = rand(T, C + H + 3), rand(C, taps) * 0.6, rand(T, H * D + H * V)
    step_pre, dt_bias, a_log = low[:, :H * D], rand(H * D), rand(H) - 1.0
    start = rand(2 * T + 1, stride)
    held, written = i32(range(T)), i32([2 * T - 1 - e for e in range(T)])
    rows, entry = i32([[e, 1] for e in range(T)]), i32(range(T))

    one, apart = start.clone(), start.clone()
    got, want = torch.full((T, H * V), 9.0, device="cuda"), torch.full((T, H * V), 7.0, device="cuda")
    assert ops.delta_step_ok(D, one)
    ops.delta_step(pre, conv, step_pre, dt_bias, a_log, one, matrix, held, written, rows, got, D ** -0.5, G, H, D, V, C)
    q, k, v, decay, beta = (torch.empty(T, w, device="cuda") for w in (G * D, G * D, H * V, H * D, H))
    ops.delta_prep(pre, conv, step_pre, dt_bias, a_log, apart, matrix, held, entry, rows, q, k, v, decay, beta, G, H, D, V, C)
    tail = (pre[:, :C], taps, matrix) if taps > 1 else None
    ops.state_scan(q, k, v, decay, beta, apart, held, written, rows, want, D ** -0.5, H, G, D, V, tail=tail, max_rows=1)
    assert torch.equal(got, want)
    for s in written.tolist():          # what a request keeps; a tile's columns beyond V and the slot's padding are nobody's
        assert torch.equal(ops.state_matrix_plain(one[s], H, D, V), ops.state_matrix_plain(apart[s], H, D, V))
        assert torch.equal(one[s, matrix:matrix + (taps - 1) * C], apart[s, matrix:matrix + (taps - 1) * C])
    assert torch.equal(one[:T], start[:T]) and torch.equal(one[2 * T], start[2 * T])
    assert np.isfinite(got.cpu().numpy()).all()


# heads at each number of channels a lane and beside it, value channels over several units, both ends of the taps that the form for
# many rows takes and one beyond; runs that begin inside a block of 16 rows, and the first number of rows that takes the form
@pytest.mark.parametrize("H,G,D,V,taps", [(4, 2, 16, 24, 3), (2, 1, 64, 100, 2), (3, 3, 65, 33, 4), (2, 1, 128, 128, 4), (1, 1, 129, 1, 2), (2, 2, 256, 40, 4), (2, 1, 32, 32, 5)])
@pytest.mark.parametrize("counts", [(255, 1), (1, 200, 99), (3, 250, 17, 2)])
def test_many_rows_are_prepared_with_the_bits_of_few(H, G, D, V, taps, counts):
    from llmx_amd import ops

    gen = torch.Generator().manual_seed(H * 1000 + D * 10 + taps)
    rand = lambda *shape: torch.randn(*shape, generator=gen).cuda()
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")
    C, T = 2 * G * D + H * V, sum(counts)
    matrix = ops.state_matrix_size(H, D, V)
    pre, conv, low = rand(T, C + H + 3), rand(C, taps) * 0.6, rand(T, H * D + H * V)
    dt_bias, a_log, state = rand(H * D), rand(H) - 1.0, rand(len(counts) + 1, matrix + (taps - 1) * C)

    def prepare(a, b, entries):
        n = b - a
        out = [torch.full((n, w), 9.0, device="cuda") for w in (G * D, G * D, H * V, H * D, H)]
        begins = [sum(counts[:e]) - a for e in entries]
        ops.delta_prep(pre[a:b], conv, low[a:b, :H * D], dt_bias, a_log, state, matrix, i32([e + 1 for e in entries]),
                       i32([i for i, e in enumerate(entries) for _ in range(counts[e])]), i32([[s, counts[e]] for s, e in zip(begins, entries)]), *out,
                       G, H, D, V, C)
        return out

    together = prepare(0, T, list(range(len(counts))))
    apart = [prepare(sum(counts[:e]), sum(counts[:e + 1]), [e]) for e in range(len(counts))]
    for i, got in enumerate(together):
        assert torch.equal(got, torch.cat([x[i] for x in apart])), ("q", "k", "v", "decay", "beta")[i]
