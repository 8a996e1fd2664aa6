"""The pull-back's ring of stages from its shortest contraction on (two stages; fewer, as many and more than are asked for ahead),
for every number of row blocks of a tile, on both tile shapes: grouped calls on 128-row tiles against dense calls (the same bits)
and against float64.

Bound: the products dy * bf16(w) are exact in float32, a sum of n of them in any order is off by at most n * 2^-23 * sum |terms|,
and one rounding to bf16 follows (2^-8 relative; an ulp for the neighbour)."""

import numpy as np
import pytest

from __graft_entry__ import load_package

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [8, 64, 104, 128, 160, 192, 232, 256, 320])
def test_short_contractions(n):
    import torch

    w8 = load_package().w8a8_lora
    k, sizes = 1096, [20, 64, 70, 128, 0, 33, 1, 97]
    rng = np.random.default_rng(n)
    codes = torch.from_numpy(rng.integers(-127, 128, (len(sizes), k, n), dtype=np.int8)).cuda()
    scales = torch.from_numpy(rng.uniform(0.001, 0.01, (len(sizes), 1, n)).astype(np.float32)).cuda()
    dy = torch.from_numpy(rng.standard_normal((sum(sizes), n)).astype(np.float32)).cuda().to(torch.bfloat16)
    x = torch.zeros(sum(sizes), k, dtype=torch.bfloat16, device="cuda")
    gw = w8.prepare_grouped_weight(codes, scales)
    gs = torch.tensor(sizes, dtype=torch.int32, device="cuda")
    print(f"[case] pull-back of {n} columns", flush=True)
    got = w8.grouped_backward(x, dy, gs, gw)[0]
    ref = w8.grouped_backward_per_weight(x, dy, gs, gw)[0]
    assert torch.equal(got, ref)
    first = 0
    for g, rows in enumerate(sizes):
        d = dy[first:first + rows].double()
        w = (codes[g].float() * scales[g]).to(torch.bfloat16).double()
        want, magnitude = d @ w.T, d.abs() @ w.abs().T
        off = (got[first:first + rows].double() - want).abs()
        assert bool((off <= 2.0 ** -7 * want.abs() + n * 2.0 ** -23 * magnitude).all()), (g, rows)
        first += rows
