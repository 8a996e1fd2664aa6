"""Adapters that are not finite on the tiles that stand in for 32-row chunks: an infinity in A or B makes the row's values what they are
in float32 and in the chunks (infinite, of its sign), not NaN."""

import pytest

from __graft_entry__ import load_package
import w8a8_cases as wc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,k,n,n_ad,rank", [
    (65, 8192, 136, 3, 16), (49, 4096, 264, 1, 8), (64, 8192, 130, 2, 64),
    (64, 4096, 2560, 9, 16), (33, 8192, 8192, 1, 40),   # a group to a block, in pairs or alone
    (40, 8192, 4104, 8, 16), (90, 8192, 1024, 24, 64), (65, 8192, 8192, 16, 64),
])
@pytest.mark.parametrize("where", ["a", "b", "both"])
def test_infinite_adapters(m, k, n, n_ad, rank, where):
    import torch

    case = wc.make_case(m, k, n, n_adapters=n_ad, rank=rank, seed=m + k)
    t = wc.to_torch(case, "cuda:0")
    spoil = n_ad // 2
    if where != "b":
        t["a"][spoil, 5, rank // 2] = float("inf")
    if where != "a":
        t["b"][spoil, rank // 3, 7] = -float("inf")
        t["b"][spoil, rank // 2, n - 3] = float("inf")
    print(f"[case] infinite {where} {m}x{k}x{n} adapters={n_ad} rank={rank}", flush=True)
    got = load_package().w8a8_lora.ForwardPlan(t["x"], t["weight"], t["a"], t["b"], t["s"], adapter_indices=t["idx"]).run().float()
    torch.cuda.synchronize()
    want = torch.empty(m, n, dtype=torch.float64)
    for g in range(n_ad):
        rows = torch.from_numpy(case["idx"] == g)
        want[rows] = (t["x"].cpu()[rows].double() @ t["a"][g].double().cpu()) @ t["b"][g].double().cpu()
    got = got.cpu()
    assert (torch.isnan(got) == torch.isnan(want)).all()
    assert (torch.isinf(got) == torch.isinf(want)).all()
    assert (torch.sign(got)[torch.isinf(want)] == torch.sign(want)[torch.isinf(want)]).all()
