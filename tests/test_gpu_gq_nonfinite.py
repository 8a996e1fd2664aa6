"""Infinities and NaN through the group-scaled backward.  The rule is float32 products and sums, so every entry of the
cotangents has the class (finite, either infinity, NaN) that plain products in float64 give it: an infinite
gradient spoils its row of dx and its column of dB, not the columns beside it."""

import pytest

from __graft_entry__ import load_package

pytestmark = pytest.mark.gpu
INF, NAN = float("inf"), float("nan")

PLACES = {  # operand -> [(row, column, value)]
    "none": {},
    "dy_inf": {"dy": [(3, 37, INF)]},
    "dy_two": {"dy": [(3, 37, INF), (3, 5, -INF), (36, 71, -INF)]},
    "dy_nan": {"dy": [(39, 0, NAN), (0, 8, INF)]},
    "x_inf": {"x": [(7, 131, -INF)]},
    "a_inf": {"a": [(129, 0, INF)]},
    "b_inf": {"b": [(0, 40, -INF)]},
}


@pytest.mark.parametrize("rank", [1, 33])
@pytest.mark.parametrize("bits,group,scale", [(8, 32, "float32"), (4, 128, "bfloat16")])
@pytest.mark.parametrize("place", PLACES)
def test_classes_of_the_cotangents(place, bits, group, scale, rank):
    import torch

    pkg = load_package()
    ql, gq = pkg.quantized_lora, pkg.gq_linear
    m, k, n, s = 40, 136, 72, 0.75
    gen = torch.Generator().manual_seed(rank + bits)
    rnd = lambda *shape: (torch.randn(*shape, generator=gen) * 0.5).to(torch.bfloat16)
    ops = {"x": rnd(m, k), "dy": rnd(m, n), "a": rnd(k, rank), "b": rnd(rank, n)}
    for name, entries in PLACES[place].items():
        for row, col, value in entries:
            ops[name][row, col] = value
    w = ql.quantize_frozen_weight(torch.randn(k, n, generator=gen), bits=bits, group_size=group, scale_dtype=getattr(torch, scale))
    x, dy, a, b = (t.double() for t in ops.values())
    rs, z = (dy @ b.T) * s, x @ a
    want = (dy @ ql.dequantize_frozen_weight(w).double().T + rs @ a.T, x.T @ rs, (z.T @ dy) * s, (dy * (z @ b)).sum().reshape(1))
    wt = ql.GroupQuantizedWeight(w.codes.cuda(), w.scales.cuda(), w.original_in_features, w.padded_in_features, bits, group)
    print(f"[case] {place} bits={bits} rank={rank}", flush=True)
    dev = {name: t.cuda() for name, t in ops.items()}
    got = gq.backward(dev["x"], dev["dy"], wt, dev["a"], dev["b"], s)
    only_dx = gq.backward(dev["x"], dev["dy"], wt, dev["a"], dev["b"], s, need_lora_grads=False)[0]
    for name, g, r in zip(("dx", "dA", "dB", "ds", "dx alone"), (*got, only_dx), (*want, want[0])):
        g = g.double().cpu()
        assert torch.equal(g.isnan(), r.isnan()), name
        inf = r.isinf()
        assert torch.equal(g.isinf(), inf) and torch.equal(g[inf], r[inf]), name
        fin = r.isfinite()  # one rounding to bf16, float32 sums (2^-23 of a few hundred terms of size below 4)
        assert ((g - r)[fin].abs() <= 2.0 ** -8 * r[fin].abs() + 2.0 ** -12).all(), name


def test_a_product_beyond_float32_beside_an_infinity():
    """x * rs beyond the largest float32 is finite in the sum: the infinity of another row decides."""
    import torch

    pkg = load_package()
    m, k, n, s = 40, 64, 64, 1.0
    gen = torch.Generator().manual_seed(9)
    rnd = lambda *shape: (torch.randn(*shape, generator=gen) * 0.5).to(torch.bfloat16)
    x, dy, a, b = rnd(m, k).abs() + 1, torch.zeros(m, n, dtype=torch.bfloat16), rnd(k, 8), torch.zeros(8, n, dtype=torch.bfloat16)
    x[3] = 4.0
    b[2, 40], dy[3, 40], dy[7, 41], b[2, 41] = 2e38, 1.0, -INF, 1.0  # rs[3] = 2e38, times 4 beyond float32; rs[7] = -inf
    wt = pkg.quantized_lora.quantize_frozen_weight(torch.randn(k, n, generator=gen).cuda(), bits=8, group_size=32)
    print("[case] product beyond float32 beside an infinity", flush=True)
    da = pkg.gq_linear.backward(x.cuda(), dy.cuda(), wt, a.cuda(), b.cuda(), s)[1].double().cpu()
    rs = (dy.double() @ b.double().T) * s
    want = x.double().T @ rs
    assert torch.equal(da.isnan(), want.isnan()) and torch.equal(da.isinf(), want.isinf())
    assert torch.equal(da[want.isinf()], want[want.isinf()])
