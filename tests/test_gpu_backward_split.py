"""The pull-back's tiles split along the contraction (N >= 2048, tiles that do not fill whole rounds of the chip):
few rows, rows and k that end inside a tile, adapters that meet inside a 32-row block, whole tiles in front of
split ones.  Reference: float32 products of the bf16 operands on the same GPU (the rule of the oracle, which
these sizes would keep busy for minutes)."""

import pytest

from __graft_entry__ import load_package

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,k,n,n_ad,rank", [
    (1, 136, 2048, 1, 8), (70, 264, 2056, 3, 5), (300, 520, 4096, 2, 33), (257, 1032, 6144, 4, 64), (500, 2048, 2304, 0, 0),
    (4400, 4096, 2048, 2, 16),   # 288 tiles: 256 whole ones, 32 split
])
def test_split_pull_back(m, k, n, n_ad, rank):
    import torch

    pkg = load_package()
    w8, ql = pkg.w8a8_lora, pkg.quantized_lora
    print(f"[case] split pull-back {m}x{k}x{n} adapters={n_ad} rank={rank}", flush=True)
    g = torch.Generator(device="cuda:0").manual_seed(m + n)
    rnd = lambda *s: torch.randn(s, generator=g, device="cuda:0")
    codes = torch.randint(-127, 128, (k, n), generator=g, device="cuda:0", dtype=torch.int8)
    scales = (torch.rand((1, n), generator=g, device="cuda:0") * 0.8 + 0.2) / (127 * n ** 0.5)
    w = ql.GroupQuantizedWeight(codes, scales, k, k, 8, k)
    dy = rnd(m, n).bfloat16()
    want = dy.float() @ (codes.float() * scales).bfloat16().float().T
    lora = idx = x = None
    if n_ad:
        a, b = (rnd(n_ad, k, rank) * 0.1).bfloat16(), (rnd(n_ad, rank, n) / n ** 0.5).bfloat16()
        s = torch.linspace(0.5, 2.0, n_ad, device="cuda:0")
        idx = torch.randint(0, n_ad, (m,), generator=g, device="cuda:0", dtype=torch.int32)
        x = rnd(m, k).bfloat16()
        lora = (a, b, s)
        for ad in range(n_ad):
            rows = (idx == ad).nonzero().flatten()
            want[rows] += ((dy[rows].float() @ b[ad].float().T) * s[ad]) @ a[ad].float().T
    got = w8.backward(x, dy, w, *(lora or (None, None, None)), adapter_indices=idx)[0].float()
    torch.cuda.synchronize()
    # one bf16 rounding (2^-8 of the value) and float32 sums of n terms in another order (n * 2^-24 of the terms' size)
    bound = want.abs() * 2.0 ** -8 + n * 2.0 ** -24 * 4 * want.abs().mean()
    assert ((got - want).abs() <= bound).all(), ((got - want).abs() / bound).max().item()
    again = w8.backward(x, dy, w, *(lora or (None, None, None)), adapter_indices=idx)[0].float()
    assert torch.equal(got, again)
