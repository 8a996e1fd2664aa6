"""The four-wave pull-back at the edges of its tile: rows that end inside a row block, at the line between the loop over four and
over eight row blocks and behind it, k that ends inside a wave's 64 and 32 and 8, whole tiles and split ones, every rank width.
Reference: float32 products of the bf16 operands on the same GPU."""

import pytest

from __graft_entry__ import load_package

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [1, 32, 128, 129, 255, 300])
@pytest.mark.parametrize("k,n,n_ad,rank", [(8, 256, 1, 16), (264, 8, 3, 17), (328, 520, 0, 0), (584, 2056, 2, 64)])
def test_edges(m, k, n, n_ad, rank):
    import torch

    pkg = load_package()
    w8, ql = pkg.w8a8_lora, pkg.quantized_lora
    print(f"[case] wide pull-back {m}x{k}x{n} adapters={n_ad} rank={rank}", flush=True)
    g = torch.Generator(device="cuda:0").manual_seed(m + n + k)
    rnd = lambda *s: torch.randn(s, generator=g, device="cuda:0")
    codes = torch.randint(-127, 128, (k, n), generator=g, device="cuda:0", dtype=torch.int8)
    scales = (torch.rand((1, n), generator=g, device="cuda:0") * 0.8 + 0.2) / (127 * n ** 0.5)
    w = ql.GroupQuantizedWeight(codes, scales, k, k, 8, k)
    dy = rnd(m, n).bfloat16()
    want = dy.float() @ (codes.float() * scales).bfloat16().float().T
    lora, idx, x = (None, None, None), None, None
    if n_ad:
        a, b = (rnd(n_ad, k, rank) * 0.1).bfloat16(), (rnd(n_ad, rank, n) / n ** 0.5).bfloat16()
        s = torch.linspace(0.5, 2.0, n_ad, device="cuda:0")
        idx = torch.randint(0, n_ad, (m,), generator=g, device="cuda:0", dtype=torch.int32)
        x, lora = rnd(m, k).bfloat16(), (a, b, s)
        for ad in range(n_ad):
            rows = (idx == ad).nonzero().flatten()
            want[rows] += ((dy[rows].float() @ b[ad].float().T) * s[ad]) @ a[ad].float().T
    got = w8.backward(x, dy, w, *lora, adapter_indices=idx)[0].float()
    torch.cuda.synchronize()
    # one bf16 rounding (2^-8 of the value) and float32 sums of n terms in another order (n * 2^-24 of the terms' size)
    bound = want.abs() * 2.0 ** -8 + n * 2.0 ** -24 * 4 * want.abs().mean()
    assert ((got - want).abs() <= bound).all(), ((got - want).abs() / bound).max().item()
