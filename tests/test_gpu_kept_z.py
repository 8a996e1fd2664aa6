"""x @ A as the forward leaves it for the backward (mi355_w8a8_problem_z): its values on every prologue that writes it, and the
backward that takes it against the one that forms it again.

Bounds: a product of bf16 values is exact in float32; a sum of k of them in any order is off by at most k * 2^-23 * sum |terms|.  dB
sums m products of z and dy on top and is rounded once to bf16 (2^-8 relative; an ulp for the neighbour)."""

import ctypes

import numpy as np
import pytest

from __graft_entry__ import load_package
import w8a8_cases as wc

pytestmark = pytest.mark.gpu


def _project(x, a, group):
    import torch

    z, mag = (torch.empty(x.shape[0], a.shape[2], dtype=torch.float64, device=x.device) for _ in range(2))
    for g in range(a.shape[0]):
        rows = group == g
        z[rows] = x[rows].double() @ a[g].double()
        mag[rows] = x[rows].double().abs() @ a[g].double().abs()
    return z, mag


def _compare(with_z, without, z_mag, dy, group, k, s):
    import torch

    assert torch.equal(with_z[0], without[0]) and torch.equal(with_z[1], without[1])
    for g in range(with_z[2].shape[0]):
        rows = group == g
        m = int(rows.sum())
        bound = 2.0 ** -6 * without[2][g].double().abs() + 2 * (k + m) * 2.0 ** -23 * (z_mag[rows].T @ dy[rows].double().abs()) * s[g].double().abs()
        assert bool(((with_z[2][g].double() - without[2][g].double()).abs() <= bound).all()), g
    torch.testing.assert_close(with_z[3], without[3], rtol=1e-3, atol=1e-2)


@pytest.mark.parametrize("m,k,n,n_ad,rank,rms", [
    (2048, 512, 4096, 4, 16, False),    # groups on block boundaries
    (1500, 256, 6144, 3, 5, True),      # odd rank
    (3003, 128, 8200, 24, 32, False),   # blocks of several groups
    (4100, 6144, 4104, 2, 64, False),   # K beyond the rows that the LDS holds
    (2100, 320, 4096, 1, 64, True),
])
def test_dense(m, k, n, n_ad, rank, rms):
    import torch

    w8 = load_package().w8a8_lora
    case = wc.make_case(m, k, n, n_adapters=n_ad, rank=rank, rms=rms, seed=m)
    t = wc.to_torch(case, "cuda:0")
    idx = t["idx"] if n_ad > 1 else None
    kw = dict(rms_gamma=t["gamma"], want_normalized=True) if rms else {}
    print(f"[case] kept z {m}x{k}x{n} adapters={n_ad} rank={rank}", flush=True)
    plan = w8.ForwardPlan(t["x"], t["weight"], t["a"], t["b"], t["s"], adapter_indices=idx, want_z=True, **kw)
    assert plan.z is not None
    plan.z.fill_(float("nan"))
    out = plan.run().clone()
    first = plan.z.clone()
    plan.run()   # (the operands kept: another prologue where the rows fit the LDS)
    plain = w8.ForwardPlan(t["x"], t["weight"], t["a"], t["b"], t["s"], adapter_indices=idx, **kw)
    assert torch.equal(out, plain.run())
    x = plan.aux["normalized"] if rms else t["x"].reshape(m, k)
    group = idx.reshape(-1) if idx is not None else torch.zeros(m, dtype=torch.int32, device="cuda")
    want, mag = _project(x, t["a"], group)
    for z in (first, plan.z):
        assert bool(((z.double() - want).abs() <= k * 2.0 ** -23 * mag).all())
    dy = torch.randn(m, n, device="cuda", generator=torch.Generator("cuda").manual_seed(m)).to(torch.bfloat16)
    args = (x, dy, t["weight"], t["a"], t["b"], t["s"])
    got = w8.BackwardPlan(*args, adapter_indices=idx, z=first).run()
    _compare(got, w8.BackwardPlan(*args, adapter_indices=idx).run(), mag, dy, group, k, t["s"])


@pytest.mark.parametrize("sizes,k,n,rank,gpw,repeat", [([5, 0, 300, 17], 256, 512, 8, 1, 0), ([40, 70, 0, 3, 260, 1], 384, 776, 16, 2, 3),
                                                      ([33] * 8, 200, 264, 5, 1, 0), ([64, 129, 1, 127], 1096, 264, 64, 1, 2)])
def test_grouped(sizes, k, n, rank, gpw, repeat):
    import torch

    w8 = load_package().w8a8_lora
    rng = np.random.default_rng(k)
    m, g = sum(sizes), len(sizes)
    f = lambda *shape: torch.from_numpy(rng.standard_normal(shape).astype(np.float32)).cuda().to(torch.bfloat16)
    gw = w8.prepare_grouped_weight(torch.from_numpy(rng.integers(-127, 128, (g // gpw, k, n), dtype=np.int8)).cuda(),
                                   torch.rand(g // gpw, n, device="cuda") * 0.01)
    rows = -(-m // repeat) if repeat else m
    x, a, b, s, dy = f(rows, k), f(g, k, rank) * 0.1, f(g, rank, n) * 0.1, torch.rand(g, device="cuda") + 0.5, f(m, n)
    kw = {}
    if repeat:
        kw = dict(row_map=torch.from_numpy(rng.permutation(rows * repeat)[:m].astype(np.int32)).cuda(), row_repeat=repeat)
    gs = torch.tensor(sizes, dtype=torch.int32, device="cuda")
    print(f"[case] kept z, groups {sizes} k={k} rank={rank} repeat={repeat}", flush=True)
    plan = w8.GroupedForwardPlan(x, gs, gw, a, b, s, groups_per_weight=gpw, want_z=True, **kw)
    out = plan.run()
    assert torch.equal(out, w8.grouped_forward(x, gs, gw, a, b, s, groups_per_weight=gpw, **kw))
    xs = x[(kw["row_map"] // repeat).long()] if repeat else x
    group = torch.repeat_interleave(torch.arange(g, device="cuda"), gs.long())
    want, mag = _project(xs, a, group)
    assert bool(((plan.z.double() - want).abs() <= k * 2.0 ** -23 * mag).all())
    got = w8.GroupedBackwardPlan(x, dy, gs, gw, a, b, s, groups_per_weight=gpw, z=plan.z, **kw).run()
    _compare(got, w8.grouped_backward(x, dy, gs, gw, a, b, s, groups_per_weight=gpw, **kw), mag, dy, group, k, s)


def test_refused_where_the_path_has_no_place_for_it():
    import torch

    pkg = load_package()
    w8, nat = pkg.w8a8_lora, pkg._native
    for m, n in ((16, 4096), (333, 2560)):
        t = wc.to_torch(wc.make_case(m, 512, n, n_adapters=2, rank=16, seed=m), "cuda:0")
        plan = w8.ForwardPlan(t["x"], t["weight"], t["a"], t["b"], t["s"], adapter_indices=t["idx"], want_z=True)
        assert plan.z is None
        z = torch.empty(m, 16, device="cuda")
        p = nat.problem_struct(nat.Problem, nat.ProblemZ, z)
        for name, _ in nat.Problem._fields_[1:]:
            setattr(p, name, getattr(plan.problem, name))
        assert nat.STATUS[nat.load().mi355_w8a8_forward_v1(ctypes.byref(p), None)] == "ERR_UNSUPPORTED"
    with pytest.raises(ValueError):
        w8.BackwardPlan(t["x"], torch.zeros(m, n, dtype=torch.bfloat16, device="cuda"), t["weight"], t["a"], t["b"], t["s"],
                        adapter_indices=t["idx"], z=z[:5])
