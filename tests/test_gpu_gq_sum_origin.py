"""Edges of the staged group-scaled kernel: sums at the ends of the range that starts at a float32 bit pattern (groups up
to 256), the first longer group, more adapters than one mask holds, LoRA B off a 16-byte boundary, ragged 64 x 128 tiles."""

import numpy as np
import pytest

from __graft_entry__ import load_package

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,k,n,bits,group,n_ad,shift", [
    (64, 256, 128, 8, 256, 0, 0), (65, 512, 129, 4, 256, 0, 0), (127, 640, 160, 8, 320, 0, 0), (33, 64, 40, 4, 64, 0, 0),
    (193, 192, 136, 8, 64, 70, 0), (65, 192, 136, 4, 192, 3, 1), (40, 192, 264, 8, 64, 1, 1)])
def test_staged_kernel_at_the_ends_of_its_range(m, k, n, bits, group, n_ad, shift):
    """Whole columns of the most negative and the largest codes against rows of the largest activation codes: the
    float32 base is the direct kernel's bit for bit, so the integer sums arrived whole."""
    import torch

    pkg = load_package()
    dev = torch.device("cuda:0")
    rng = np.random.default_rng(m + n)
    low, high = (-128, 127) if bits == 8 else (-8, 7)
    codes = rng.integers(low, high + 1, (k, n)).astype(np.int32)
    codes[:, 0::4], codes[:, 1::4] = low, high
    if bits == 4:
        stored = ((codes[0::2] & 15) | ((codes[1::2] & 15) << 4)).astype(np.uint8)
    else:
        stored = codes.astype(np.int8)
    scales = rng.uniform(0.001, 0.01, (k // group, n)).astype(np.float32)
    w = pkg.quantized_lora.GroupQuantizedWeight(torch.from_numpy(stored).to(dev), torch.from_numpy(scales).to(dev), k, k, bits,
                                                group)
    x = rng.standard_normal((m, k)).astype(np.float32)
    x[0::3], x[1::3] = 3.0, -3.0
    args = [torch.from_numpy(x).to(dev).to(torch.bfloat16), w]
    kw = dict(activation_bits=8, return_aux=True)
    if n_ad:
        a = torch.from_numpy(rng.standard_normal((n_ad, k, 8)).astype(np.float32) * 0.05).to(dev).to(torch.bfloat16)
        b = torch.from_numpy(rng.standard_normal((n_ad, 8, n)).astype(np.float32) * 0.05).to(dev).to(torch.bfloat16)
        flat = torch.empty(b.numel() + 8, dtype=torch.bfloat16, device=dev)
        b = flat[shift:shift + b.numel()].view(b.shape).copy_(b)
        args += [a, b, torch.from_numpy(rng.uniform(0.5, 2.0, n_ad).astype(np.float32)).to(dev)]
        kw["adapter_indices"] = torch.from_numpy(rng.integers(0, n_ad, m).astype(np.int32)).to(dev)
    print(f"[case] gq ends m={m} k={k} n={n} W{bits} group={group} adapters={n_ad}", flush=True)
    staged, aux_s = pkg.gq_linear.forward(*args, **kw)
    direct, aux_d = pkg.gq_linear.forward(*args, flags=pkg._native.FLAG_GQ_DIRECT, **kw)
    torch.cuda.synchronize()
    assert torch.equal(aux_s["base"].view(torch.int32), aux_d["base"].view(torch.int32))
    assert torch.equal(staged.view(torch.int16), direct.view(torch.int16))
