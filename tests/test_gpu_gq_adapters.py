"""The staged group-scaled kernel's low-rank sums: batches of up to eight adapters that two row blocks of 32 share, each
block taking its own adapters; bit for bit the direct kernel's, which has neither batches nor the LDS."""

import numpy as np
import pytest

from __graft_entry__ import load_package

pytestmark = pytest.mark.gpu


def _indices(kind, m, n_ad, rng):
    if kind == "random":
        return rng.integers(0, n_ad, m)
    if kind == "halves":   # the row blocks of a tile share no adapter
        return (np.arange(m) // 32 % 2) * (n_ad // 2) + rng.integers(0, n_ad // 2, m)
    if kind == "last":     # none of the first 64
        return rng.integers(64, n_ad, m)
    return np.where(np.arange(m) % 64 < 40, 0, n_ad - 1)  # "ends"


@pytest.mark.parametrize("m,k,n,bits,group,n_ad,rank,kind", [
    (64, 128, 128, 8, 64, 8, 64, "random"),    # one whole batch per step
    (65, 128, 136, 4, 64, 9, 17, "random"),    # a second batch of one, the last step of one rank
    (200, 128, 264, 8, 128, 18, 48, "halves"),
    (127, 192, 130, 4, 64, 3, 33, "ends"),     # B value by value
    (96, 64, 72, 8, 64, 70, 16, "last"),
    (97, 64, 200, 4, 64, 130, 8, "random"),    # three masks
    (40, 512, 24, 8, 512, 2, 1, "halves"),
])
def test_batches_of_adapters(m, k, n, bits, group, n_ad, rank, kind):
    import torch

    pkg = load_package()
    dev = torch.device("cuda:0")
    rng = np.random.default_rng(m + n + rank)
    stored = (rng.integers(-128, 128, (k // 2, n)).astype(np.uint8) if bits == 4 else rng.integers(-127, 128, (k, n)).astype(np.int8))
    scales = rng.uniform(0.001, 0.01, (k // group, n)).astype(np.float32)
    w = pkg.quantized_lora.GroupQuantizedWeight(torch.from_numpy(stored).to(dev), torch.from_numpy(scales).to(dev), k, k, bits,
                                                group)
    bf = lambda v: torch.from_numpy(v.astype(np.float32)).to(dev).to(torch.bfloat16)
    args = [bf(rng.standard_normal((m, k))), w, bf(rng.standard_normal((n_ad, k, rank)) * 0.05),
            bf(rng.standard_normal((n_ad, rank, n)) * 0.05), torch.from_numpy(rng.uniform(0.5, 2.0, n_ad).astype(np.float32)).to(dev)]
    kw = dict(activation_bits=8, adapter_indices=torch.from_numpy(_indices(kind, m, n_ad, rng).astype(np.int32)).to(dev))
    print(f"[case] gq adapters m={m} k={k} n={n} W{bits} group={group} adapters={n_ad} rank={rank} {kind}", flush=True)
    staged = pkg.gq_linear.forward(*args, **kw)
    direct = pkg.gq_linear.forward(*args, flags=pkg._native.FLAG_GQ_DIRECT, **kw)
    torch.cuda.synchronize()
    assert torch.equal(staged.view(torch.int16), direct.view(torch.int16))
