"""The group-scaled backward kernels at the edges of their tiles and dispatch: rows, K and N off the tile sizes,
each code width, group size and scale type, whole and split pull-back tiles.

Bound: every product dy * (code * scale) is exact and the float32 sum of T terms in any order is off by at most
T * 2^-23 * sum |terms|; the cotangents are rounded once to bf16 (2^-8 relative, two ulps allowed)."""

import numpy as np
import pytest

from oracle import w8a8_oracle as o

pytestmark = pytest.mark.gpu
F32 = np.float32


@pytest.fixture(scope="module")
def pkg():
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from __graft_entry__ import load_package

    p = load_package()
    p._native.load()
    return p


CASES = [  # m, k, n, bits, group, scale type, rank
    (1, 32, 8, 8, 32, "f32", 1),
    (257, 136, 40, 8, 64, "bf16", 32),       # K cut inside a group, a second row tile of one row, N off 32
    (40, 264, 200, 4, 32, "f32", 33),        # rank beyond 32, a third k tile of eight columns
    (300, 128, 264, 4, 128, "bf16", 17),
    (130, 384, 2056, 8, 128, "bf16", 8),     # N over 2048: tiles split along the contraction
    (520, 320, 4096, 4, 64, "f32", 64),
]


@pytest.mark.parametrize("m,k,n,bits,group,scale,rank", CASES)
def test_group_scaled_backward(pkg, m, k, n, bits, group, scale, rank):
    import torch

    dev = torch.device("cuda:0")
    rng = np.random.default_rng(m * 7 + n)
    w = o.quantize_frozen_weight((rng.standard_normal((k, n)) * 0.05).astype(F32), bits=bits, group_size=group,
                                 scale_dtype=scale)
    sw = torch.from_numpy(np.asarray(w.scales, dtype=F32)).to(dev)
    wt = pkg.quantized_lora.GroupQuantizedWeight(torch.from_numpy(w.codes).to(dev),
                                                 sw.to(torch.bfloat16) if scale == "bf16" else sw,
                                                 w.original_in_features, w.padded_in_features, bits, group)
    x, dy = (o.bf16_round(rng.standard_normal(s).astype(F32)) for s in ((m, k), (m, n)))
    a, b = (o.bf16_round((rng.standard_normal(s) * 0.05).astype(F32)) for s in ((k, rank), (rank, n)))
    s = 0.75
    bf = lambda v: torch.from_numpy(v).to(dev).to(torch.bfloat16)
    assert pkg.gq_linear.has_native_backward(wt)
    got = pkg.gq_linear.backward(bf(x), bf(dy), wt, bf(a), bf(b), s)
    torch.cuda.synchronize()
    deq = pkg.quantized_lora.dequantize_frozen_weight(wt).cpu().numpy().astype(np.float64)
    x, dy, a, b = (v.astype(np.float64) for v in (x, dy, a, b))
    rs, z = (dy @ b.T) * s, x @ a
    dot = lambda p, q: (p @ q, np.abs(p) @ np.abs(q))
    base, base_abs = dot(dy, deq.T)
    low, low_abs = dot(rs, a.T)
    r_abs, z_abs = (np.abs(dy) @ np.abs(b.T)) * s, np.abs(x) @ np.abs(a)
    want = {
        "dx": (base + low, base_abs + r_abs @ np.abs(a.T), n + rank),
        "dA": (x.T @ rs, np.abs(x.T) @ r_abs, m + n),
        "dB": ((z.T @ dy) * s, (z_abs.T @ np.abs(dy)) * s, m + k),
    }
    for (name, (ref, magnitude, terms)), t in zip(want.items(), got):
        t = t.to(torch.float32).cpu().numpy().astype(np.float64)
        bound = 2.0 ** -7 * np.abs(ref) + terms * 2.0 ** -23 * magnitude
        over = np.abs(t - ref) - bound
        assert t.shape == ref.shape and np.all(over <= 0), (name, float(over.max()), float(np.abs(t - ref).max()))
    ds, ds_abs = float((dy * (z @ b)).sum()), float((np.abs(dy) * (z_abs @ np.abs(b))).sum())
    assert abs(float(got[3]) - ds) <= 2.0 ** -23 * (k + n + rank) * ds_abs


def test_parts_that_are_not_asked_for(pkg):
    """dx alone and the LoRA cotangents alone carry the same bits as the whole call."""
    import torch

    dev = torch.device("cuda:0")
    g = torch.Generator(device="cpu").manual_seed(3)
    bf = lambda *shape: (torch.randn(*shape, generator=g) * 0.1).to(torch.bfloat16).to(dev)
    w = pkg.quantized_lora.quantize_frozen_weight(torch.randn(192, 128, generator=g).to(dev), bits=4, group_size=64)
    x, dy, a, b = bf(70, 192), bf(70, 128), bf(192, 16), bf(16, 128)
    whole = pkg.gq_linear.backward(x, dy, w, a, b, 2.0)
    only_dx = pkg.gq_linear.backward(x, dy, w, a, b, 2.0, need_lora_grads=False)
    only_lora = pkg.gq_linear.backward(x, dy, w, a, b, 2.0, need_dx=False)
    torch.cuda.synchronize()
    assert torch.equal(whole[0], only_dx[0]) and only_dx[1:] == (None, None, None)
    assert only_lora[0] is None and all(torch.equal(p, q) for p, q in zip(whole[1:], only_lora[1:]))


@pytest.mark.parametrize("m,k,n,bits", [(70, 192, 128, 4), (300, 264, 2056, 8)])  # whole tiles, split ones
def test_replays_under_capture(pkg, m, k, n, bits):
    """Captured once, replayed with new operands in the same buffers and eager work between: the eager call's bits."""
    import torch

    dev = torch.device("cuda:0")
    g = torch.Generator(device="cpu").manual_seed(m)
    bf = lambda *shape: (torch.randn(*shape, generator=g) * 0.1).to(torch.bfloat16).to(dev)
    w = pkg.quantized_lora.quantize_frozen_weight(torch.randn(k, n, generator=g).to(dev), bits=bits, group_size=32 if k % 64 else 64)
    operands = [bf(m, k), bf(m, n), bf(k, 16), bf(16, n)]
    scaling = torch.full((), 1.5, device=dev)
    x, dy, a, b = operands
    run = lambda: pkg.gq_linear.backward(x, dy, w, a, b, scaling)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        run()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = run()
    for i in range(4):
        for t in operands:
            t.copy_(bf(*t.shape))
        x[0, 0] = float("inf") if i == 1 else 1.0  # the look at operands that are not finite starts anew each time
        want = run()
        for t in got:
            t.fill_(7.0)
        junk = torch.randn(512, 512, device=dev)
        assert bool(torch.isfinite((junk @ junk).sum()))
        graph.replay()
        torch.cuda.synchronize()
        for p, q in zip(got, want):
            assert torch.equal(torch.nan_to_num(p.float(), nan=3e38), torch.nan_to_num(q.float(), nan=3e38)), i
