"""Float32 attention on the float32 matrix instruction: columns, segments, windows and what may not leak, against float64."""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def ops():
    from llmx_amd import ops as o
    return o


def caches(lens, G, D, V, page, seed, window=0):
    """Keys and values [entry][token] and the same in shuffled pages; places no token lies at hold NaN, pages wholly before the
    last row's window are given back (-1)."""
    g = torch.Generator().manual_seed(seed)
    blocks = [-(-L // page) for L in lens]
    order = torch.randperm(sum(blocks) + 2, generator=g).tolist()
    tables = torch.full((len(lens), max(blocks)), -1, dtype=torch.int32)
    k_cache = torch.full((len(order), G, page, D), float("nan"))
    v_cache = torch.full((len(order), G, V, page), float("nan"))
    keys, values = [], []
    for e, L in enumerate(lens):
        k, v = torch.randn(L, G, D, generator=g), torch.randn(L, G, V, generator=g)
        keys.append(k)
        values.append(v)
        for b in range(blocks[e]):
            at = order.pop()
            n = min(page, L - b * page)
            k_cache[at, :, :n] = k[b * page:b * page + n].transpose(0, 1)
            v_cache[at, :, :, :n] = v[b * page:b * page + n].permute(1, 2, 0)
            tables[e, b] = at
    return keys, values, k_cache.to(DEV), v_cache.to(DEV), tables.to(DEV)


def plain(q, k, v, p, scale, window):
    lo = max(0, p - window + 1) if window else 0
    H, G = q.shape[0], k.shape[1]
    kk, vv = (t[lo:p + 1].double().repeat_interleave(H // G, 1) for t in (k, v))
    w = torch.softmax(torch.einsum("hd,shd->hs", q.double(), kk) * scale, 1)
    return torch.einsum("hs,shv->hv", w, vv)


def run(q, kc, vc, pos, ent, tables, H, V, window=0, **more):
    o = ops()
    out = torch.full((q.shape[0], H * V), float("nan"), device=DEV)
    o.take_launches()
    o.paged_attention(q, kc, vc, pos, ent, tables, out, 0.125, H, window, **more)
    ran = o.take_launches()
    split = "scratch" in more and bool(o.lib().llmx_attention_f32_scratch(q.shape[0], H, vc.shape[1], V, kc.shape[2], tables.shape[1]))
    assert ran == {"attention.generic": 1, "attention_f32": 1, **({"attention_f32.merge": 1} if split else {})}
    return out


def fresh(name, shape, dtype):
    return torch.full(shape, float("nan"), dtype=dtype, device=DEV)


def i32(x):
    return torch.tensor(x, dtype=torch.int32, device=DEV)


# heads a KV head: 1, 3 (15 of 16 columns), 4, 16, 20 (two chunks); widths of one tile, all of a form's and one more; values of a
# width of their own; pages of 4 to 48
SIZES = [(4, 4, 16, 16, 4), (6, 2, 64, 64, 8), (8, 2, 128, 128, 16), (16, 1, 80, 48, 16), (20, 1, 64, 160, 32), (4, 2, 256, 256, 48)]


@pytest.mark.parametrize("H,G,D,V,page", SIZES)
@pytest.mark.parametrize("window", [0, 33])
def test_rows_of_several_requests(H, G, D, V, page, window):
    """Prompt rows, a request of one row and rows about the segments' edges in one call, with and without enough rows for tiles of
    neighbouring rows; each row alone gives the same bits; the gates."""
    lens = [31, 300, 1, 65]
    keys, values, kc, vc, tables = caches(lens, G, D, V, page, 3)
    rows = [(0, 30), (2, 0), (3, 31), (3, 32), (3, 63), (3, 64)] + [(1, p) for p in range(0, 300)] + [(0, 0), (0, 15)]
    q = torch.randn(len(rows), H * D, generator=torch.Generator().manual_seed(4)).to(DEV)
    pos, ent = i32([p for _, p in rows]), i32([e for e, _ in rows])
    out = run(q, kc, vc, pos, ent, tables, H, V, window)
    for t, (e, p) in enumerate(rows):
        want = plain(q[t].cpu().view(H, D), keys[e], values[e], p, 0.125, window)
        got = out[t].double().cpu().view(H, V)
        # scores carry sqrt(D) roundings of their size, values and weights about one each
        assert (got - want).abs().max() <= 64 * 2.0 ** -24 * math.sqrt(D) * max(1.0, float(want.abs().max())), (e, p)
    for t in (0, 1, 2, 3, 5, 40, 305, len(rows) - 1):
        alone = run(q[t:t + 1].contiguous(), kc, vc, pos[t:t + 1], ent[t:t + 1], tables, H, V, window)
        assert torch.equal(alone[0], out[t]), "a row's bits depend on the rows beside it"
        shared = run(q[t:t + 1].contiguous(), kc, vc, pos[t:t + 1], ent[t:t + 1], tables, H, V, window, scratch=fresh)
        assert torch.equal(shared[0], out[t]), "sharing the context out changes a row's bits"
    few = run(q[:200].contiguous(), kc, vc, pos[:200].contiguous(), ent[:200].contiguous(), tables, H, V, window)
    assert torch.equal(few, out[:200])
    gate = torch.randn(len(rows), H + 3, generator=torch.Generator().manual_seed(6)).to(DEV)
    gated = run(q, kc, vc, pos, ent, tables, H, V, window, head_gate=gate[:, 3:])
    one = run(q[40:41].contiguous(), kc, vc, pos[40:41], ent[40:41], tables, H, V, window, head_gate=gate[40:41, 3:], scratch=fresh)
    assert torch.equal(one[0], gated[40])
    assert torch.allclose(gated, (out.view(-1, H, V) * torch.sigmoid(gate[:, 3:, None])).reshape(-1, H * V), rtol=1e-6, atol=1e-7)
    wide = torch.randn(len(rows), H * V, generator=torch.Generator().manual_seed(7)).to(DEV)
    gated = run(q, kc, vc, pos, ent, tables, H, V, window, output_gate=wide)
    one = run(q[40:41].contiguous(), kc, vc, pos[40:41], ent[40:41], tables, H, V, window, output_gate=wide[40:41], scratch=fresh)
    assert torch.equal(one[0], gated[40])
    assert torch.allclose(gated, out * torch.sigmoid(wide), rtol=1e-6, atol=1e-7)


def test_rows_in_any_order_and_entries_in_turn():
    H, G, D, V, page = 4, 1, 32, 32, 16
    keys, values, kc, vc, tables = caches([200, 210], G, D, V, page, 8)
    rows = [(t % 2, (97 * t) % 200) for t in range(320)] + [(0, 199 - t) for t in range(40)]
    q = torch.randn(len(rows), H * D, generator=torch.Generator().manual_seed(4)).to(DEV)
    out = run(q, kc, vc, i32([p for _, p in rows]), i32([e for e, _ in rows]), tables, H, V, 0)
    for t in range(0, len(rows), 7):
        e, p = rows[t]
        alone = run(q[t:t + 1].contiguous(), kc, vc, i32([p]), i32([e]), tables, H, V)
        assert torch.equal(alone[0], out[t])
        assert (alone[0].double().cpu().view(H, V) - plain(q[t].cpu().view(H, D), keys[e], values[e], p, 0.125, 0)).abs().max() < 1e-5


@pytest.mark.parametrize("window", [0, 700])
def test_long_contexts_shared_out(window):
    """Decoded rows of unequal contexts of many segments: as one workgroup a row walks them."""
    lens = [5, 2049, 1000, 3]
    keys, values, kc, vc, tables = caches(lens, 2, 128, 128, 16, 11)
    q = torch.randn(4, 8 * 128, generator=torch.Generator().manual_seed(4)).to(DEV)
    pos, ent = i32([n - 1 for n in lens]), i32([0, 1, 2, 3])
    shared = run(q, kc, vc, pos, ent, tables, 8, 128, window, scratch=fresh)
    assert torch.equal(shared, run(q, kc, vc, pos, ent, tables, 8, 128, window))
    for t, n in enumerate(lens):
        want = plain(q[t].cpu().view(8, 128), keys[t], values[t], n - 1, 0.125, window)
        assert (shared[t].double().cpu().view(8, 128) - want).abs().max() < 64 * 2.0 ** -24 * math.sqrt(128)


def test_pages_given_back_and_values_that_are_not_finite():
    """Keys before a window are not read (their pages are gone); an infinite or NaN key or value reaches the rows that see it and
    no other, in tiles of neighbouring rows too."""
    H, G, D, V, page, window = 8, 2, 64, 64, 16, 40
    L = 400
    keys, values, kc, vc, tables = caches([L], G, D, V, page, 9)
    given = tables.clone()
    given[0, :(L - 30 - window) // page] = -1
    q = torch.randn(L, H * D, generator=torch.Generator().manual_seed(4)).to(DEV)
    pos, ent = i32(list(range(L))), i32([0] * L)
    clean = run(q, kc, vc, pos, ent, tables, H, V, window)
    late = run(q[L - 30:].contiguous(), kc, vc, pos[L - 30:].contiguous(), ent[:30].contiguous(), given, H, V, window)
    assert torch.equal(late, clean[L - 30:])
    whole = run(q, kc, vc, pos, ent, tables, H, V)
    spoilt = vc.clone()
    at = 205
    spoilt[int(tables[0, at // page]), 1, 5, at % page] = float("inf")
    spoilt[int(tables[0, at // page]), 0, 6, at % page] = float("nan")
    for w, plain_out in ((0, whole), (window, clean)):
        got = run(q, kc, spoilt, pos, ent, tables, H, V, w).view(L, H, V)
        expected = plain_out.view(L, H, V).clone()
        sees = slice(at, min(L, at + w) if w else L)
        assert bool(torch.isinf(got[sees, 4:, 5]).all()) and bool(torch.isnan(got[sees, :4, 6]).all())
        expected[sees, 4:, 5], expected[sees, :4, 6] = got[sees, 4:, 5], got[sees, :4, 6]
        assert torch.equal(torch.nan_to_num(got), torch.nan_to_num(expected))
    bad_key = kc.clone()
    bad_key[int(tables[0, at // page]), 1, at % page, 3] = float("nan")
    got = run(q, bad_key, vc, pos, ent, tables, H, V).view(L, H, V)
    assert bool(torch.isnan(got[at:, 4:]).all()) and torch.equal(got[:at], whole.view(L, H, V)[:at]) and torch.equal(got[:, :4], whole.view(L, H, V)[:, :4])
