"""x += s1 * y1 (+ s2 * y2): four values a thread where the rows allow it, with the bits of one a thread."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def rnd(*shape, seed=0):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)).to(DEV)


# four values a thread, and one where a row's are no multiple of 4 or do not begin on 16 bytes
@pytest.mark.parametrize("rows,n", [(1, 4), (3, 2048), (129, 1028), (2, 6)])
@pytest.mark.parametrize("two,scaled,copied", [(True, True, torch.bfloat16), (True, False, None), (False, True, torch.float32), (False, False, torch.bfloat16)])
def test_the_scaled_join_of_any_place(rows, n, two, scaled, copied):
    from llmx_amd import ops
    got = []
    for shift in (0, 1):
        place = lambda seed, *shape: rnd(*shape, seed=seed) if not shift else torch.cat([torch.zeros(1, device=DEV), rnd(*shape, seed=seed).flatten()])[1:].view(*shape)
        x, y1, y2, s1, s2 = place(1, rows, n), place(2, rows, n), place(3, rows, n), place(4, n), place(5, n)
        copy = torch.full((rows, n), float("nan"), dtype=copied, device=DEV) if copied is not None else None
        ops.scale_add(x, y1, s1 if scaled else None, y2 if two else None, s2 if scaled and two else None, copy)
        got.append((x.clone(), None if copy is None else copy.float()))
    assert torch.equal(got[0][0], got[1][0]) and (copied is None or torch.equal(got[0][1], got[1][1]))
    want = rnd(rows, n, seed=1).double() + rnd(rows, n, seed=2).double() * (rnd(n, seed=4).double() if scaled else 1.0)
    if two:
        want = want + rnd(rows, n, seed=3).double() * (rnd(n, seed=5).double() if scaled else 1.0)
    # two products and two sums, each rounded once
    assert (got[0][0].double() - want).abs().max() <= 4 * 2.0 ** -24 * 60


# four values a thread only where every operand lies on 16 bytes: each of them moved by one value, alone
@pytest.mark.parametrize("n", [1028, 1030])
@pytest.mark.parametrize("copied", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("moved", [None, "x", "y1", "s1", "y2", "s2", "copy"])
def test_four_values_a_thread(moved, copied, n):
    from llmx_amd import ops
    rows, got = 3, []
    for name in (None, moved):
        held = {}

        def place(which, values):
            space = torch.full((values.numel() + 8,), float("nan"), dtype=values.dtype, device=DEV)
            at = 1 if which == name else 0
            held[which] = (space, at, values.numel())
            view = space[at:at + values.numel()].view(values.shape)
            view.copy_(values)
            return view

        x, y1, y2 = (place(which, rnd(rows, n, seed=i)) for i, which in enumerate(("x", "y1", "y2")))
        s1, s2 = place("s1", rnd(n, seed=3)), place("s2", rnd(n, seed=4))
        copy = place("copy", torch.zeros(rows, n, dtype=copied, device=DEV))
        ops.take_launches()
        ops.scale_add(x, y1, s1, y2, s2, copy)
        assert ops.take_launches(details=True) == {"scale_add": 1, **({"scale_add+four": 1} if name is None and n % 4 == 0 else {})}
        got.append((x.clone(), copy.clone()))
        for space, at, size in held.values():       # nothing beside an operand is touched
            assert bool(space[:at].isnan().all()) and bool(space[at + size:].isnan().all())
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])
