"""64 x 128 tiles whose waves split K: the bits of the 128 x 128 geometry at the edges of tiles, k blocks, ranks and columns, one
workgroup to a CU and two, and beyond the rows whose prologue may leave z in quarters."""

import pytest

from __graft_entry__ import load_package
import w8a8_cases as wc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,k,n,n_ad,rank,kind", [
    (33, 128, 130, 1, 1, "plain"), (64, 136, 127, 2, 16, "residual"), (65, 8, 258, 3, 17, "rms"),
    (96, 1032, 1544, 8, 8, "plain"), (97, 640, 129, 1, 33, "residual"), (333, 768, 384, 4, 64, "plain"),
    (40, 2560, 512, 2, 64, "swiglu"), (129, 264, 260, 3, 5, "swiglu"), (70, 4616, 96, 5, 32, "rms"),
    (200, 512, 300, 0, 0, "plain"), (2047, 256, 1030, 3, 40, "rms"),   # 297 tiles of 64 x 128: two workgroups to a CU
    (2100, 384, 1024, 1, 64, "residual"), (1100, 136, 2820, 2, 24, "swiglu"),
])
def test_same_bits_as_128x128(m, k, n, n_ad, rank, kind):
    import torch

    pkg = load_package()
    w8, nat = pkg.w8a8_lora, pkg._native
    case = wc.make_case(m, k, n, n_adapters=n_ad, rank=max(rank, 1), seed=m + n, rms=kind in ("rms", "swiglu"), residual=kind == "residual")
    print(f"[case] k split {m}x{k}x{n} adapters={n_ad} rank={rank} {kind}", flush=True)
    t = wc.to_torch(case, "cuda:0")
    outs = []
    for flags in (nat.FLAG_FORCE_TILED, nat.FLAG_FORCE_TILED | nat.FLAG_TILE_128X128):
        plan = w8.ForwardPlan(t["x"], t["weight"], t.get("a"), t.get("b"), t.get("s"), adapter_indices=t.get("idx"),
                              rms_gamma=t.get("gamma"), eps=1e-6, residual=t.get("residual"), swiglu=kind == "swiglu", flags=flags)
        outs.append(plan.run().clone())
        outs.append(plan.run(nat.FLAG_LORA_PACK_VALID if n_ad else 0).clone())
    torch.cuda.synchronize()
    for other in outs[1:]:
        assert torch.equal(outs[0].view(torch.int16), other.view(torch.int16))
    if kind != "swiglu":
        rep = wc.compare(outs[0].float().cpu().numpy().reshape(m, n), wc.oracle_forward(case))
        assert rep["violations"] == 0, rep
