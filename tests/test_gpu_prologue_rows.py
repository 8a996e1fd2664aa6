"""The tiled path's two prologues -- rows held in the LDS, rows read twice behind their statistics -- on the same
problems: a call that lays the LoRA operands out and one that keeps them, groups padded to 32-row blocks and (a
geometry that never pads) packed, take the one or the other (prologue_keeps_rows).  All give the oracle's
codes and the same bits."""

import numpy as np
import pytest

from __graft_entry__ import load_package
import w8a8_cases as wc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,k,n,n_ad,rank,rms", [
    (33, 40, 72, 2, 5, True),            # a K that ends inside a 32-wide block, boundaries inside a half block
    (150, 1000, 260, 3, 16, False), (520, 4608, 132, 7, 33, True),   # sixteen rows in the LDS, the longest
    (41, 4616, 100, 5, 64, True), (90, 9728, 96, 1, 32, False),      # eight rows; four from 9728 on
    (17, 16384, 64, 2, 8, True), (530, 12288, 40, 3, 16, True),      # more than 128 workgroups of four rows
    (70, 5000, 96, 0, 0, False), (1100, 264, 132, 0, 0, True), (4200, 136, 40, 64, 30, False),
])
def test_both_prologues(m, k, n, n_ad, rank, rms):
    import torch

    pkg = load_package()
    w8, nat = pkg.w8a8_lora, pkg._native
    case = wc.make_case(m, k, n, n_adapters=n_ad, rank=max(rank, 1), seed=m + k, rms=rms)
    print(f"[case] prologues {m}x{k}x{n} adapters={n_ad} rank={rank} rms={rms}", flush=True)
    st = wc.oracle_forward(case, return_stages=True)
    t = wc.to_torch(case, "cuda:0")
    results = []
    for flags in (nat.FLAG_FORCE_TILED, nat.FLAG_FORCE_TILED | nat.FLAG_TILE_256X128):
        plan = w8.ForwardPlan(t["x"], t["weight"], t.get("a"), t.get("b"), t.get("s"), adapter_indices=t.get("idx"),
                              rms_gamma=t.get("gamma"), eps=1e-6, flags=flags)
        plan.keep_lora_pack = False
        results.append(plan.run().clone())
        results += [plan.run(nat.FLAG_LORA_PACK_VALID).clone() for _ in range(2)]
        with_aux, aux = wc.gpu_forward(case, flags=flags)
        results.append(torch.from_numpy(with_aux).to("cuda:0", torch.bfloat16))
        np.testing.assert_array_equal(aux["x_codes"], st["x_codes"])
        np.testing.assert_array_equal(aux["x_scales"], st["x_scales"])
        if rms:
            np.testing.assert_array_equal(aux["normalized"], st["normalized"])
    torch.cuda.synchronize()
    rep = wc.compare(results[0].float().cpu().numpy(), st["out"])
    assert rep["violations"] == 0, rep
    for other in results[1:]:
        assert torch.equal(results[0].view(torch.int16).reshape(-1), other.view(torch.int16).reshape(-1))
