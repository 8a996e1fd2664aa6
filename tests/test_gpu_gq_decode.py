"""Group-scaled calls of up to 32 rows at the edges of the streaming kernel and of its prologue: one and two row
halves, shares of K that are empty, shorter or longer than the steps in flight, N off the 16-column units, rank
tiles, K slices that end inside a step of the projection.

Bounds: the float32 base adds the oracle's own terms in another order, T of them off by at most T * 2^-23 * sum
|terms|; the low-rank term's two float32 sums likewise; the output is rounded once to bf16 (2^-8 relative)."""

import numpy as np
import pytest

from oracle import w8a8_oracle as o

pytestmark = pytest.mark.gpu
F32 = np.float32

CASES = [  # m, k, n, weight bits, activation bits, group, rank, adapters
    (1, 64, 16, 8, 8, 64, 1, 1),             # one step, fifteen waves without a share
    (16, 2560, 40, 4, 8, 128, 17, 1),        # N ends inside a 16-column unit; a second rank tile of one rank
    (17, 1160, 48, 8, 4, 64, 33, 1),         # second row half of one row; K padded; K slices end inside a step
    (32, 8192, 24, 4, 4, 64, 64, 1),         # eight groups a wave: rounds beyond the steps in flight
    (9, 12288, 136, 8, 8, 64, 8, 1),
    (31, 1024, 72, 4, 8, 512, 16, 3),        # long groups; several adapters
]


@pytest.mark.parametrize("m,k,n,wb,ab,group,rank,n_ad", CASES)
def test_group_scaled_decode(m, k, n, wb, ab, group, rank, n_ad):
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from __graft_entry__ import load_package

    pkg, dev = load_package(), torch.device("cuda:0")
    rng = np.random.default_rng(m + k + n)
    x = o.bf16_round(rng.standard_t(4, (m, k)).astype(F32))
    w = o.quantize_frozen_weight((rng.standard_normal((k, n)) * 0.05).astype(F32), bits=wb, group_size=group,
                                 scale_dtype="f32")
    base = o.quantized_frozen_linear_f32(x, w, activation_bits=ab)
    a = o.bf16_round((rng.standard_normal((n_ad, k, rank)) * 0.05).astype(F32))
    b = o.bf16_round((rng.standard_normal((n_ad, rank, n)) * 0.05).astype(F32))
    s = rng.uniform(0.5, 2.0, n_ad).astype(F32)
    idx = rng.integers(0, n_ad, m).astype(np.int32)
    bf = lambda v: torch.from_numpy(np.ascontiguousarray(v)).to(dev).to(torch.bfloat16)
    wt = pkg.quantized_lora.GroupQuantizedWeight(torch.from_numpy(w.codes).to(dev), torch.from_numpy(w.scales).to(dev),
                                                 w.original_in_features, w.padded_in_features, wb, group)
    got, aux = pkg.gq_linear.forward(bf(x), wt, bf(a), bf(b), torch.from_numpy(s).to(dev), activation_bits=ab,
                                     adapter_indices=torch.from_numpy(idx).to(dev), return_aux=True)
    torch.cuda.synchronize()
    terms = -(-k // group)
    deq = np.abs(pkg.quantized_lora.dequantize_frozen_weight(wt).cpu().numpy().astype(np.float64))[:k]
    xa = np.abs(x).astype(np.float64)
    amax = np.abs(x).max()  # a dequantized activation is off x by at most half a step of its group's scale
    size = (xa + amax / (14 if ab == 4 else 254)) @ deq
    eps = 2.0 ** -23
    assert (np.abs(aux["base"].cpu().numpy() - base) <= (terms + 2) * eps * size).all()
    a64, b64 = a.astype(np.float64)[idx], b.astype(np.float64)[idx]
    low = s[idx, None] * np.einsum("mr,mrn->mn", np.einsum("mk,mkr->mr", x.astype(np.float64), a64), b64)
    low_size = s[idx, None] * np.einsum("mr,mrn->mn", np.einsum("mk,mkr->mr", xa, np.abs(a64)), np.abs(b64))
    want = base.astype(np.float64) + low
    bound = (terms + 2) * eps * size + (k + rank + 4) * eps * low_size + 2.0 ** -8 * np.abs(want)
    assert (np.abs(got.to(torch.float32).cpu().numpy() - want) <= bound + 1e-30).all()
