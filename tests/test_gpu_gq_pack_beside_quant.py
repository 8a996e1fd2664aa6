"""One adapter's A packed by the group quantizer's launch: the bits of a call whose routing launch packs it, and float64."""

import pytest

from __graft_entry__ import load_package

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,k,n,group,rank", [
    (33, 32, 64, 32, 1), (33, 2048, 72, 128, 64), (40, 72, 136, 32, 8), (63, 1000, 64, 64, 33), (300, 640, 128, 128, 32), (1100, 96, 64, 32, 16),
])
def test_same_bits_as_behind_the_routing_launch(m, k, n, group, rank):
    import torch

    pkg = load_package()
    gq, ql = pkg.gq_linear, pkg.quantized_lora
    print(f"[case] packed beside the quantizer {m}x{k}x{n} group={group} rank={rank}", flush=True)
    g = torch.Generator(device="cuda:0").manual_seed(m + k)
    rand = lambda *s: torch.randn(s, generator=g, device="cuda:0")  # noqa: E731
    x, a, b = rand(m, k).bfloat16(), rand(k, rank).bfloat16(), rand(rank, n).bfloat16()
    w = ql.quantize_frozen_weight(rand(k, n), bits=8, group_size=group)
    got = gq.forward(x, w, a, b, 0.5)
    two_a, two_b = torch.stack((a, -a)), torch.stack((b, b))
    factors = torch.full((2,), 0.5, device="cuda:0")
    want = gq.forward(x, w, two_a, two_b, factors, adapter_indices=torch.zeros(m, dtype=torch.int32, device="cuda:0"))
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))
    # two adapters and no indices: the first for every row, both packed
    assert torch.equal(gq.forward(x, w, two_a, two_b, factors).view(torch.int16), want.view(torch.int16))
    # against float64: the low-rank product alone, its float32 sums added to the base and rounded to bf16 (half an ulp, 2^-9 of the value)
    base = gq.forward(x, w).double()
    full = base + 0.5 * ((x.double() @ a.double()) @ b.double())
    bound = full.abs() * 2.0**-8 + base.abs() * 2.0**-8 + 1e-5 * (k * rank) ** 0.5 * 16
    assert bool(((got.double() - full).abs() <= bound).all())
