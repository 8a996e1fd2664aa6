"""Decode plans over several runs: B gathered by the first, regrouped by the second, kept from then on -- the same bits each
time, and the new values after B, the indices or both are written.  Sizes at the edges of the regrouped layout
(rows of 16 and 32 ranks, 1 KiB pieces that end inside a row quad, N off the 16-column units) and calls that
do not keep it."""

import numpy as np
import pytest

from __graft_entry__ import load_package
import w8a8_cases as wc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,k,n,n_ad,rank,form", [
    (16, 64, 4, 1, 16, "plain"), (9, 512, 132, 2, 31, "residual"), (15, 1024, 260, 16, 18, "plain"), (8, 256, 100, 3, 32, "residual"),
    (16, 2048, 128, 64, 16, "rms"), (16, 12288, 144, 5, 17, "residual"), (13, 16384, 64, 4, 29, "plain"),
    (9, 256, 64, 2, 16, "plain"), (17, 256, 64, 2, 32, "plain"), (12, 256, 66, 2, 32, "plain"), (12, 256, 64, 2, 33, "plain"), (16, 256, 64, 2, 32, "swiglu"),
    (16, 256, 16384, 2, 16, "plain"), (16, 256, 16384, 2, 16, "residual"),   # two slices (never kept), one
])
def test_kept_b(m, k, n, n_ad, rank, form):
    import torch

    w8 = load_package().w8a8_lora
    case = wc.make_case(m, k, n, n_adapters=n_ad, rank=rank, seed=m + n, rms=form in ("rms", "swiglu"), swiglu=form == "swiglu",
                        residual=form == "residual")
    t = wc.to_torch(case, "cuda:0")
    print(f"[case] kept B {m}x{k}x{n} adapters={n_ad} rank={rank} {form}", flush=True)
    plan = w8.ForwardPlan(t["x"], t["weight"], t["a"], t["b"], t["s"], adapter_indices=t["idx"], rms_gamma=t.get("gamma"),
                          eps=1e-6, residual=t.get("residual"), swiglu=form == "swiglu")

    def runs(want):
        got = [plan.run().clone() for _ in range(4)]
        rep = wc.compare(got[0].float().cpu().numpy(), wc.oracle_forward(want))
        assert rep["violations"] == 0, rep
        assert all(torch.equal(got[0].view(torch.int16), g.view(torch.int16)) for g in got[1:])

    runs(case)
    idx = ((case["idx"] + 1) % n_ad).astype(np.int32)
    plan.adapter_indices.copy_(torch.from_numpy(idx).to("cuda:0"))
    runs(dict(case, idx=idx))
    t["b"].mul_(-0.5)
    runs(dict(case, idx=idx, b=case["b"] * np.float32(-0.5)))


def test_a_run_by_the_tiled_path_between():
    """Sixteen adapters on block boundaries: the tiled path's codes then reach over the place of the regrouped B."""
    import torch

    p = load_package()
    case = wc.make_case(16, 1024, 4096, n_adapters=16, rank=32, seed=5, residual=False)
    case["idx"] = np.arange(16, dtype=np.int32)
    t = wc.to_torch(case, "cuda:0")
    plan = p.w8a8_lora.ForwardPlan(t["x"], t["weight"], t["a"], t["b"], t["s"], adapter_indices=t["idx"])
    print("[case] kept B, tiled run between", flush=True)
    want = [plan.run().clone() for _ in range(3)]
    plan.run(p._native.FLAG_FORCE_TILED)
    got = [plan.run().clone() for _ in range(3)]
    assert all(torch.equal(want[0].view(torch.int16), g.view(torch.int16)) for g in want[1:] + got)


def test_one_run_reserves_no_room():
    native = load_package()._native
    size = native.load().mi355_w8a8_workspace_bytes
    plain = size(16, 12288, 4096, 16, 32, 0)
    assert size(16, 12288, 4096, 16, 32, native.FLAG_DECODE_B_WRITE) - plain >= 16 * 32 * 4096 * 2
    for m, rank in ((17, 32), (4, 32), (16, 33)):
        assert size(m, 12288, 4096, 16, rank, native.FLAG_DECODE_B_WRITE) == size(m, 12288, 4096, 16, rank, 0)
