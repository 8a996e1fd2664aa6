"""Decode calls whose LoRA B or residual holds an odd number of values: the last one has no whole dword of its own and
is loaded by itself.  Against the oracle; what lies behind the tensors (NaN here) does not show."""

import pytest

from __graft_entry__ import load_package
import w8a8_cases as wc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,k,n,n_ad,rank,residual", [
    (1, 64, 1, 1, 1, True), (3, 256, 17, 1, 5, True), (16, 512, 129, 3, 33, False), (17, 512, 65, 5, 7, True),
    (31, 1032, 33, 1, 63, True), (35, 256, 97, 3, 1, True),   # 35 rows: chunks of 32 and 3
])
def test_odd_sizes(m, k, n, n_ad, rank, residual):
    import torch

    w8 = load_package().w8a8_lora
    case = wc.make_case(m, k, n, n_adapters=n_ad, rank=rank, seed=m + n, residual=residual)
    case["idx"][-1] = n_ad - 1
    t = wc.to_torch(case, "cuda:0")

    def before_nan(v):
        flat = torch.full((v.numel() + 8,), float("nan"), dtype=v.dtype, device=v.device)
        flat[:v.numel()] = v.reshape(-1)
        return flat[:v.numel()].reshape(v.shape)

    print(f"[case] odd decode {m}x{k}x{n} adapters={n_ad} rank={rank}", flush=True)
    got = w8.forward(t["x"], t["weight"], before_nan(t["a"]), before_nan(t["b"]), t["s"], adapter_indices=t["idx"], eps=1e-6,
                     residual=before_nan(t["residual"]) if residual else None)
    rep = wc.compare(got.float().cpu().numpy(), wc.oracle_forward(case))
    assert rep["violations"] == 0, rep
