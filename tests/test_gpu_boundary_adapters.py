"""Rows of several adapters in one block of slots: what another adapter holds does not reach a row.  Calls whose groups lie packed, z in
quarters and packed, on the K-split tiles and (the last) on others."""

import pytest

from __graft_entry__ import load_package
import w8a8_cases as wc

pytestmark = pytest.mark.gpu

CASES = [(228, 4096, 6144, 24, 16),   # quarters of z, tiles one to a CU
         (300, 2560, 6144, 8, 33),    # quarters
         (530, 1544, 3072, 2, 64),    # packed z
         (700, 1040, 6144, 5, 8),     # quarters, tiles in pairs
         (333, 4096, 2560, 40, 8),    # most blocks hold several
         (4200, 520, 1544, 3, 16)]    # beyond the K-split tiles


def both(case, spoil):
    """The call's output as the case is and with the adapter `spoil` not finite."""
    import torch

    t = wc.to_torch(case, "cuda:0")
    outs = []
    for value in (None, float("inf"), float("nan")):
        a = t["a"].clone()
        if value is not None:
            a[spoil, ::7] = value
        plan = load_package().w8a8_lora.ForwardPlan(t["x"], t["weight"], a, t["b"], t["s"], adapter_indices=t["idx"],
                                                    rms_gamma=t.get("gamma"))
        outs.append(plan.run().clone())
    torch.cuda.synchronize()
    return outs


@pytest.mark.parametrize("m,k,n,n_ad,rank", CASES)
def test_an_adapter_without_rows(m, k, n, n_ad, rank):
    import torch

    n_ad += 1
    case = wc.make_case(m, k, n, n_adapters=n_ad, rank=rank, seed=m + n)
    spoil = n_ad // 2
    case["idx"][case["idx"] == spoil] = n_ad - 1
    print(f"[case] boundary {m}x{k}x{n} adapters={n_ad} rank={rank}", flush=True)
    plain, inf, nan = both(case, spoil)
    assert torch.equal(plain.view(torch.int16), inf.view(torch.int16))
    assert torch.equal(plain.view(torch.int16), nan.view(torch.int16))


@pytest.mark.parametrize("m,k,n,n_ad,rank", CASES)
@pytest.mark.parametrize("rms", [False, True])
def test_the_other_rows_of_a_block(m, k, n, n_ad, rank, rms):
    import torch

    case = wc.make_case(m, k, n, n_adapters=n_ad, rank=rank, seed=m + n, rms=rms)
    spoil = n_ad // 2
    print(f"[case] other rows {m}x{k}x{n} adapters={n_ad} rank={rank} rms={rms}", flush=True)
    plain, inf, nan = both(case, spoil)
    others = torch.from_numpy(case["idx"] != spoil).to(plain.device)
    assert torch.equal(plain[others].view(torch.int16), inf[others].view(torch.int16))
    assert torch.equal(plain[others].view(torch.int16), nan[others].view(torch.int16))
    assert not torch.isfinite(inf[~others]).any() and not torch.isfinite(nan[~others]).any()
