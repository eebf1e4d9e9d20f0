"""The state scan's forms: operands brought 16 bytes or one value at a time, chunks of any size, against float64."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def strided(t, pad):
    """The same values as columns of a wider tensor, `pad` columns in."""
    wide = torch.zeros(t.shape[0], t.shape[1] + 2 * pad, device=DEV)
    wide[:, pad:pad + t.shape[1]] = t
    return wide[:, pad:pad + t.shape[1]]


@pytest.mark.parametrize("D,V", [(4, 1), (36, 13), (64, 8), (100, 24), (128, 128), (132, 9), (256, 16)])
@pytest.mark.parametrize("delta", [True, False])
def test_loads_chunks_and_rows(D, V, delta):
    from llmx_amd import ops
    H, G, n = 4, 2, [1, 17, 2, 33, 16, 15, 31]
    T = sum(n)
    g = torch.Generator().manual_seed(D + V)
    q, k = torch.randn(T, G * D, generator=g).to(DEV), torch.nn.functional.normalize(torch.randn(T, G, D, generator=g), dim=2).view(T, -1).to(DEV)
    v, decay = torch.randn(T, H * V, generator=g).to(DEV), (0.5 + 0.5 * torch.rand(T, H * D, generator=g)).to(DEV)
    beta = torch.rand(T, H, generator=g).to(DEV) if delta else None
    S0 = torch.randn(len(n), H, D, V, generator=g)
    width = ops.state_matrix_size(H, D, V)
    start = torch.zeros(2 * len(n), width + (-width) % 4, device=DEV)
    for e in range(len(n)):
        start[e, :width] = ops.state_matrix_tiled(S0[e]).reshape(-1).to(DEV)
    row0 = [sum(n[:e]) for e in range(len(n))]
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    entries = [[r, c] for r, c in zip(row0, n)]

    def run(qq, kk, vv, gg, which=None, max_rows=0):
        idx = list(range(len(n))) if which is None else which
        state, out = start.clone(), torch.zeros(T, H * V, device=DEV)
        ops.state_scan(qq, kk, vv, gg, beta, state, i32(idx), i32([len(n) + e for e in idx]), i32([entries[e] for e in idx]), out, 0.5, H, G, D, V,
                       max_rows=max_rows)
        return out, state

    out, state = run(q, k, v, decay)
    for e, (r, c) in enumerate(entries):
        S = S0[e].double()
        for t in range(r, r + c):
            kt, qt = (x[t].double().cpu().view(G, D).repeat_interleave(H // G, 0) for x in (k, q))
            S = S * decay[t].double().cpu().view(H, D, 1)
            u = v[t].double().cpu().view(H, V)
            if delta:
                u = beta[t].double().cpu()[:, None] * (u - (S * kt[:, :, None]).sum(1))
            S = S + kt[:, :, None] * u[:, None, :]
            want = 0.5 * (S * qt[:, :, None]).sum(1)
            # every row adds some ten roundings a value to a state that decays: a few hundred units in the last place of its size at most
            assert (out[t].double().cpu().view(H, V) - want).abs().max() <= 256 * 2.0 ** -24 * max(1.0, float(want.abs().max())) * 4
        got = ops.state_matrix_plain(state[len(n) + e, :width].cpu(), H, D, V).double()
        assert (got - S).abs().max() <= 256 * 2.0 ** -24 * max(1.0, float(S.abs().max()))
    for pad in (1, 4):      # heads that start off a 16-byte place and rows of an odd stride; and both aligned
        o2, s2 = run(strided(q, pad), strided(k, pad), strided(v, pad), strided(decay, pad))
        assert torch.equal(o2, out) and torch.equal(s2, state)
    short = [0, 2]          # entries of one or two rows take chunks of two
    o3, s3 = run(q, k, v, decay, short, max_rows=2)
    for e in short:
        r, c = entries[e]
        assert torch.equal(o3[r:r + c], out[r:r + c]) and torch.equal(s3[len(n) + e], state[len(n) + e])
