"""Both forms of z in front of the K-split tiles, quarters where their prologue pays and packed elsewhere, one workgroup to a CU and
in pairs: the bits of the 128 x 128 geometry.  A workspace without room for the quarters takes packed z and gives the same bits; one
byte below that is refused."""

import pytest

from __graft_entry__ import load_package
import w8a8_cases as wc

pytestmark = pytest.mark.gpu


def _plan(t, flags=0):
    pkg = load_package()
    return pkg.w8a8_lora.ForwardPlan(t["x"], t["weight"], t["a"], t["b"], t["s"], adapter_indices=t.get("idx"),
                                     rms_gamma=t.get("gamma"), eps=1e-6, flags=pkg._native.FLAG_FORCE_TILED | flags)


@pytest.mark.parametrize("m,k,n,n_ad,rank,rms", [
    (97, 2056, 384, 4, 64, False),   # quarters
    (97, 2040, 384, 4, 64, True),    # packed: K below the line
    (1100, 2056, 200, 1, 50, False),  # packed: too many rows for the K
    (290, 2048, 7000, 2, 48, True),  # quarters in pairs (275 tiles)
    (530, 2048, 4000, 1, 64, False),  # packed in pairs
    (200, 200, 136, 3, 20, True), (208, 200, 136, 3, 32, False),   # rank 32: either side of K = m
    (1300, 512, 1700, 3, 16, False),  # rank 16: quarters in pairs
])
def test_same_bits_as_128x128(m, k, n, n_ad, rank, rms):
    import torch

    case = wc.make_case(m, k, n, n_adapters=n_ad, rank=rank, seed=m + k, rms=rms)
    print(f"[case] z forms {m}x{k}x{n} adapters={n_ad} rank={rank}", flush=True)
    t = wc.to_torch(case, "cuda:0")
    got = _plan(t).run().clone()
    want = _plan(t, load_package()._native.FLAG_TILE_128X128).run().clone()
    torch.cuda.synchronize()
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))


@pytest.mark.parametrize("m,k,n,n_ad,rank", [(97, 2560, 392, 4, 64), (70, 640, 258, 1, 16), (1300, 512, 1700, 3, 16)])
def test_workspace_without_room_for_the_quarters(m, k, n, n_ad, rank):
    import torch

    case = wc.make_case(m, k, n, n_adapters=n_ad, rank=rank, seed=7)
    t = wc.to_torch(case, "cuda:0")
    quarters = -(-(m + 31 * min(n_ad, m)) // 32) * 32 * (1 if rank <= 16 else 2 if rank <= 32 else 4) * 256
    print(f"[case] short workspace {m}x{k}x{n} adapters={n_ad} rank={rank}", flush=True)
    want = _plan(t).run().clone()
    for short in (256, quarters):
        plan = _plan(t)
        plan.problem.workspace_bytes -= short
        assert torch.equal(plan.run().view(torch.int16), want.view(torch.int16))
    plan = _plan(t)
    plan.problem.workspace_bytes -= quarters + 1
    with pytest.raises(RuntimeError, match="WORKSPACE"):
        plan.run()
    torch.cuda.synchronize()
