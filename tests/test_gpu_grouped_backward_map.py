"""The grouped backward reading x through a row map gives the bits of the call on the gathered rows."""

import pytest

from __graft_entry__ import load_package

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes,gpw,extra", [((5, 0, 64, 1), 1, 0), ((513, 31, 0, 40, 33, 7), 2, 9), ((0, 300), 1, 1)])
@pytest.mark.parametrize("k,n,rank", [(64, 264, 16), (328, 72, 64), (1032, 40, 5)])
def test_rows_through_a_map(sizes, gpw, extra, k, n, rank):
    import torch

    pkg = load_package()
    w8 = pkg.w8a8_lora
    print(f"[case] grouped backward through a map, sizes={sizes} gpw={gpw} {k}x{n} rank={rank}", flush=True)
    g = torch.Generator(device="cuda:0").manual_seed(k + n + extra)
    rnd = lambda *s: torch.randn(s, generator=g, device="cuda:0").bfloat16()
    groups, m, repeat = len(sizes), sum(sizes) + extra, 3
    tokens = rnd(-(-m // repeat) + 2, k)
    row_map = torch.randint(0, tokens.shape[0] * repeat, (m,), generator=g, device="cuda:0", dtype=torch.int32)
    x = tokens[row_map.long() // repeat].contiguous()
    dy, a, b = rnd(m, n), rnd(groups, k, rank), rnd(groups, rank, n)
    s = torch.linspace(0.5, 2.0, groups, device="cuda:0")
    codes = torch.randint(-127, 128, (groups // gpw, k, n), generator=g, device="cuda:0", dtype=torch.int8)
    w = w8.prepare_grouped_weight(codes, torch.full((groups // gpw, n), 0.01, device="cuda:0"))
    gs = torch.tensor(sizes, dtype=torch.int32, device="cuda:0")
    want = w8.grouped_backward(x, dy, gs, w, a, b, s, groups_per_weight=gpw)
    got = w8.grouped_backward(tokens, dy, gs, w, a, b, s, groups_per_weight=gpw, row_map=row_map, row_repeat=repeat)
    for p, q in zip(got, want):
        assert torch.equal(p.view(torch.int16), q.view(torch.int16))
    # values outside the tokens read the nearest one
    row_map[0], row_map[1] = -7, tokens.shape[0] * repeat + 5
    x[0], x[1] = tokens[0], tokens[-1]
    want = w8.grouped_backward(x, dy, gs, w, a, b, s, groups_per_weight=gpw)
    got = w8.grouped_backward(tokens, dy, gs, w, a, b, s, groups_per_weight=gpw, row_map=row_map, row_repeat=repeat)
    for p, q in zip(got, want):
        assert torch.equal(p.view(torch.int16), q.view(torch.int16))
