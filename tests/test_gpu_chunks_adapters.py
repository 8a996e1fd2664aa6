"""32-row chunks or tiles where mi355_w8a8_forward_path says chunks: the adapters of the call decide.  Either side of the lines
against the oracle; tiles in the place of chunks ignore FLAG_LORA_PACK_VALID and refuse the measurement flags as chunks do."""

import pytest

from __graft_entry__ import load_package
import w8a8_cases as wc

pytestmark = pytest.mark.gpu

CASES = [(65, 8192, 136, 3, 16),    # tiles: a third chunk
         (64, 8192, 130, 2, 64),    # tiles: rank 64 beyond 48 rows
         (49, 4096, 264, 1, 8),     # tiles: a short K
         (48, 4096, 264, 5, 33),    # chunks
         (90, 8192, 2200, 28, 16),  # chunks: the tiles would run in pairs
         (40, 8192, 4104, 16, 16),  # chunks: the same of a wider weight
         (40, 8192, 4104, 8, 16),   # tiles
         (70, 8192, 4104, 40, 8),   # chunks: tiles would run behind each other
         (33, 8200, 4104, 0, 0),    # tiles: no adapters, a wide weight
         (40, 8192, 7944, 8, 16),   # chunks: eight groups whose tiles would run in pairs
         (67, 8192, 136, 40, 16)]   # chunks: many groups of few rows


@pytest.mark.parametrize("m,k,n,n_ad,rank", CASES)
def test_against_the_oracle(m, k, n, n_ad, rank):
    nat = load_package()._native
    assert nat.PATH_NAMES[nat.load().mi355_w8a8_forward_path(m, k, n, 0)] == "skinny-chunks"
    case = wc.make_case(m, k, n, n_adapters=n_ad, rank=max(rank, 1), seed=m + n, residual=m % 2 == 0)
    print(f"[case] chunks {m}x{k}x{n} adapters={n_ad} rank={rank}", flush=True)
    st = wc.oracle_forward(case, return_stages=True)
    got, aux = wc.gpu_forward(case)
    for key in ("x_codes", "acc"):
        assert (aux[key] == st[key]).all()
    rep = wc.compare(got, st["out"])
    assert rep["violations"] == 0, rep


@pytest.mark.parametrize("m,k,n,n_ad,rank", CASES[:4] + CASES[6:8])
def test_what_chunks_ignore_and_refuse(m, k, n, n_ad, rank):
    import torch

    pkg = load_package()
    nat = pkg._native
    t = wc.to_torch(wc.make_case(m, k, n, n_adapters=n_ad, rank=rank, seed=5), "cuda:0")
    print(f"[case] ignored {m}x{k}x{n} adapters={n_ad} rank={rank}", flush=True)

    def plan():
        return pkg.w8a8_lora.ForwardPlan(t["x"], t["weight"], t["a"], t["b"], t["s"], adapter_indices=t.get("idx"), keep_lora_pack=False)

    want = plan().run().clone()
    fresh = plan()
    fresh._keep[-1].zero_()  # (the workspace: nothing has been written there)
    got = fresh.run(nat.FLAG_LORA_PACK_VALID)
    torch.cuda.synchronize()
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))
    for flag in (nat.FLAG_SKIP_PROLOGUE, nat.FLAG_SKIP_GEMM):
        with pytest.raises(RuntimeError, match="UNSUPPORTED"):
            plan().run(flag)
