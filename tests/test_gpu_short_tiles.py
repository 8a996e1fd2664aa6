"""Tiles of 192 x 256 where they fill the chip's rounds better than 256 x 256: the same bits."""

import pytest

from __graft_entry__ import load_package
import w8a8_cases as wc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,k,n,n_ad,rank,rms,swiglu,residual", [
    (1409, 384, 6144, 0, 0, False, False, False),   # the fewest stages; the last tile starts 65 slots before the end
    (1537, 520, 6144, 4, 64, False, False, True),   # one row in the last tile, groups that meet inside a tile
    (1441, 384, 6140, 8, 33, True, False, False),   # columns that end inside a wave
    (1700, 640, 6160, 3, 16, True, True, False),
    (1729, 384, 6141, 5, 8, False, False, False),   # an odd width
    (3003, 392, 4096, 4, 32, False, False, True),   # exactly one round
    (2048, 384, 10240, 4, 64, True, False, False),  # two rounds in the place of two
])
def test_tiles_of_192_rows_give_the_bits_of_256(m, k, n, n_ad, rank, rms, swiglu, residual):
    import torch

    pkg = load_package()
    w8, nat = pkg.w8a8_lora, pkg._native
    if swiglu:
        n -= n % 2
    case = wc.make_case(m, k, n, n_adapters=n_ad, rank=max(rank, 1), seed=m + n, rms=rms)
    print(f"[case] tiles of 192 rows {m}x{k}x{n} adapters={n_ad} rank={rank} rms={rms} swiglu={swiglu}", flush=True)
    t = wc.to_torch(case, "cuda:0")
    res = torch.randn((m, n), device="cuda:0").bfloat16() if residual else None
    outs = []
    for flags in (0, nat.FLAG_TILE_256X256):
        plan = w8.ForwardPlan(t["x"], t["weight"], t.get("a"), t.get("b"), t.get("s"), adapter_indices=t.get("idx"),
                              rms_gamma=t.get("gamma"), eps=1e-6, flags=flags, swiglu=swiglu, residual=res)
        out = plan.run()
        out.fill_(7.0)
        outs.append(plan.run().clone())
    torch.cuda.synchronize()
    assert torch.equal(outs[0].view(torch.int16), outs[1].view(torch.int16))
