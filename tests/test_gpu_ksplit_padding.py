"""Routed calls on the K-split tiles at either side of the lines that decide whether their groups start on block boundaries, and which
tiles that leaves: the bits of the 128 x 128 geometry (which goes by its own rule), and the oracle."""

import pytest

from __graft_entry__ import load_package
import w8a8_cases as wc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,k,n,n_ad,rank", [
    (97, 2560, 6144, 8, 16),    # on boundaries, in pairs
    (300, 2560, 6144, 8, 16),   # packed: 240 tiles instead of 432
    (530, 1536, 3072, 4, 64), (530, 1544, 3072, 2, 64),   # a short K on boundaries, a longer one packed
    (170, 2048, 10960, 8, 32), (170, 2048, 10960, 8, 8),  # behind each other on boundaries, packed in pairs
    (333, 4096, 2560, 40, 8),   # packed, eight rows to a group
    (50, 640, 3000, 64, 16),    # fewer rows than adapters
    (155, 4096, 5120, 24, 64), (240, 4096, 5120, 24, 64),  # rank 64, six rows to a group: on boundaries; ten: packed
    (323, 4096, 6144, 16, 64),  # twenty rows to a group where packed tiles run in pairs: on boundaries
    (1000, 2560, 2048, 40, 64),  # many groups and rows: on boundaries
])
def test_same_bits_as_128x128(m, k, n, n_ad, rank):
    import torch

    pkg = load_package()
    w8, nat = pkg.w8a8_lora, pkg._native
    case = wc.make_case(m, k, n, n_adapters=n_ad, rank=rank, seed=m + n_ad)
    print(f"[case] padding {m}x{k}x{n} adapters={n_ad} rank={rank}", flush=True)
    t = wc.to_torch(case, "cuda:0")
    outs = []
    for flags in (0, nat.FLAG_TILE_128X128):
        plan = w8.ForwardPlan(t["x"], t["weight"], t["a"], t["b"], t["s"], adapter_indices=t["idx"], flags=nat.FLAG_FORCE_TILED | flags)
        outs.append(plan.run().clone())
        outs.append(plan.run(nat.FLAG_LORA_PACK_VALID).clone())
    torch.cuda.synchronize()
    for other in outs[1:]:
        assert torch.equal(outs[0].view(torch.int16), other.view(torch.int16))
    rep = wc.compare(outs[0].float().cpu().numpy(), wc.oracle_forward(case))
    assert rep["violations"] == 0, rep
