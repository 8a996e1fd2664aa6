"""128 x 128 tiles of the staged group-scaled product (8-bit codes in groups beyond 256, a long K, more than 896 tiles of 64 x
128): ragged rows and columns, stages that leave a remainder in the ring, several adapters; bit for bit the direct kernel's."""

import pytest

from __graft_entry__ import load_package

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,k,n,group,n_ad,rank", [
    (1825, 6144, 3990, 384, 0, 0),    # last tile: one row, 22 columns
    (1920, 6208, 4096, 6208, 9, 17),  # one group; 97 stages of a ring of four
    (1953, 6656, 4001, 512, 2, 64),   # B value by value; the last tile's second half has one row
    (5200, 6144, 2560, 320, 1, 5),    # beyond 1600 tiles; a group is five stages
])
def test_same_bits_as_the_direct_kernel(m, k, n, group, n_ad, rank):
    import torch

    pkg = load_package()
    dev = torch.device("cuda:0")
    k_pad = -(-k // group) * group
    gen = torch.Generator(device=dev).manual_seed(m + n)
    normal = lambda *s: torch.randn(s, generator=gen, device=dev).to(torch.bfloat16)
    codes = torch.randint(-128, 128, (k_pad, n), generator=gen, device=dev, dtype=torch.int8)
    scales = torch.rand((k_pad // group, n), generator=gen, device=dev) * 0.01 + 0.001
    w = pkg.quantized_lora.GroupQuantizedWeight(codes, scales, k, k_pad, 8, group)
    args, kw = [normal(m, k), w], dict(activation_bits=8, return_aux=True)
    if n_ad:
        args += [normal(n_ad, k, rank) * 0.05, normal(n_ad, rank, n) * 0.05, torch.rand(n_ad, generator=gen, device=dev) + 0.5]
        kw["adapter_indices"] = torch.randint(0, n_ad, (m,), generator=gen, device=dev, dtype=torch.int32)
    print(f"[case] gq tall m={m} k={k} n={n} group={group} adapters={n_ad} rank={rank}", flush=True)
    staged, aux_s = pkg.gq_linear.forward(*args, **kw)
    direct, aux_d = pkg.gq_linear.forward(*args, flags=pkg._native.FLAG_GQ_DIRECT, **kw)
    torch.cuda.synchronize()
    assert torch.equal(aux_s["base"].view(torch.int32), aux_d["base"].view(torch.int32))
    assert torch.equal(staged.view(torch.int16), direct.view(torch.int16))
