"""The host module's forward calls against the plans': the same bits, and the general way for whatever is out of the ordinary."""

import pytest

from __graft_entry__ import load_package
import w8a8_cases as wc

pytestmark = pytest.mark.gpu


def _plan(w8, *args, **kw):
    return w8.ForwardPlan(*args, keep_lora_pack=False, **kw).run()


@pytest.mark.parametrize("m,k,n,n_ad,rank,rms,swiglu,residual", [
    (1, 64, 72, 3, 8, False, False, False), (33, 264, 130, 1, 64, True, False, True), (48, 128, 256, 0, 0, False, True, False),
    (600, 512, 384, 4, 16, True, True, False),
])
def test_same_bits_as_the_plan(m, k, n, n_ad, rank, rms, swiglu, residual):
    import torch

    pkg = load_package()
    w8 = pkg.w8a8_lora
    print(f"[case] host call {m}x{k}x{n} adapters={n_ad} rank={rank}", flush=True)
    case = wc.make_case(m, k, n, n_adapters=n_ad, rank=max(rank, 1), seed=m, rms=rms)
    t = wc.to_torch(case, "cuda:0")
    res = torch.randn((m, n), device="cuda:0").bfloat16() if residual else None
    kw = dict(adapter_indices=t.get("idx"), rms_gamma=t.get("gamma"), residual=res, swiglu=swiglu)
    args = (t["x"], t["weight"], t.get("a"), t.get("b"), t.get("s"))
    want = _plan(w8, *args, **kw)
    calls = []
    real = pkg._native.host().dense

    class Counting:
        @staticmethod
        def dense(*a):
            out = real(*a)
            calls.append(out is not None)
            return out

    saved, pkg._native._host = pkg._native._host, Counting
    try:
        got = w8.forward(*args, **kw)
        assert calls == [True] and tuple(got.shape) == tuple(want.shape)
        assert torch.equal(got.view(torch.int16), want.view(torch.int16))
        # what the module leaves to the plan: indices of another type, operands that are not contiguous, a gradient, no version of its own
        odd = []
        if n_ad:
            odd.append(dict(kw, adapter_indices=t["idx"].long()))
        odd.append(dict(kw, eps=1e-6))
        for o in odd:
            assert torch.equal(w8.forward(*args, **o).view(torch.int16), want.view(torch.int16))
        if n_ad:
            assert calls[1:] == [False, True]
        wide = torch.zeros((m, 2 * k), device="cuda:0", dtype=torch.bfloat16)
        wide[:, :k] = t["x"]
        assert torch.equal(w8.forward(wide[:, :k], *args[1:], **kw).view(torch.int16), want.view(torch.int16))
        leaf = t["x"].clone().requires_grad_(True)
        assert torch.equal(w8.forward(leaf, *args[1:], **kw).view(torch.int16), want.view(torch.int16))
        assert calls[-2:] == [m == 1, False]  # (one row is contiguous)
        with torch.inference_mode():
            assert torch.equal(w8.forward(*args, **kw).view(torch.int16), want.view(torch.int16))
        # one index per example
        if n_ad and m % 3 == 0:
            per = t["idx"].reshape(-1, 3)[:, 0].contiguous()
            rows = per.repeat_interleave(3)
            assert torch.equal(w8.forward(*args, **dict(kw, adapter_indices=per)).view(torch.int16),
                               _plan(w8, *args, **dict(kw, adapter_indices=rows)).view(torch.int16))
        with pytest.raises(ValueError):
            w8.forward(t["x"][:, :k - 8], *args[1:], **kw)
        with pytest.raises(TypeError):
            w8.forward(t["x"].float(), *args[1:], **kw)
    finally:
        pkg._native._host = saved


@pytest.mark.parametrize("m,k,n,bits,group,rank", [(1, 256, 72, 4, 64, 8), (40, 384, 136, 8, 128, 32), (7, 100, 64, 8, 50, 0)])
def test_group_scaled_calls(m, k, n, bits, group, rank):
    import torch

    pkg = load_package()
    gq, ql = pkg.gq_linear, pkg.quantized_lora
    print(f"[case] group-scaled host call {m}x{k}x{n} bits={bits} group={group} rank={rank}", flush=True)
    g = torch.Generator(device="cuda:0").manual_seed(m)
    x = torch.randn((m, k), generator=g, device="cuda:0").bfloat16()
    w = ql.quantize_frozen_weight(torch.randn((k, n), generator=g, device="cuda:0"), bits=bits, group_size=group)
    a = torch.randn((k, rank), generator=g, device="cuda:0").bfloat16() if rank else None
    b = torch.randn((rank, n), generator=g, device="cuda:0").bfloat16() if rank else None
    want, _ = gq.forward(x, w, a, b, 0.5, return_aux=True)
    got = gq.forward(x, w, a, b, 0.5)
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))
    assert tuple(gq.forward(x[0], w, a, b, 0.5).shape) == (n,)
    assert torch.equal(gq.forward(x.t().contiguous().t(), w, a, b, torch.tensor(0.5, device="cuda:0")).view(torch.int16), want.view(torch.int16))


@pytest.mark.parametrize("examples,rows,k,n,n_ad,rank,rms", [
    (3, 7, 256, 384, 3, 16, False), (2, 48, 4096, 256, 4, 32, False), (5, 13, 256, 520, 5, 8, True), (9, 37, 4096, 2560, 4, 64, False),
    (64, 17, 128, 256, 64, 16, True), (3, 700, 512, 4096, 2, 16, True), (1, 300, 256, 256, 1, 8, False),
])
def test_an_index_per_example(examples, rows, k, n, n_ad, rank, rms):
    """Decode, 32-row chunks, K-split, padded and packed groups: the bits of a call with the index written out per row, out-of-range
    indices among them, from an array that is 16-byte aligned and from one that is not."""
    import torch

    pkg = load_package()
    w8 = pkg.w8a8_lora
    m = examples * rows
    print(f"[case] index per example {examples}x{rows}x{k}x{n} adapters={n_ad} rank={rank}", flush=True)
    t = wc.to_torch(wc.make_case(m, k, n, n_adapters=n_ad, rank=rank, seed=m, rms=rms), "cuda:0")
    args = (t["x"], t["weight"], t["a"], t["b"], t["s"])
    g = torch.Generator(device="cuda:0").manual_seed(m)
    store = torch.randint(-2, n_ad + 2, (examples + 1,), generator=g, device="cuda:0", dtype=torch.int32)
    for per in (store[:examples], store[1:]):
        got = w8.forward(*args, adapter_indices=per, rms_gamma=t.get("gamma"))
        want = _plan(w8, *args, adapter_indices=per.repeat_interleave(rows), rms_gamma=t.get("gamma"))
        assert torch.equal(got.view(torch.int16), want.view(torch.int16))


def test_rows_per_index_that_does_not_fit_is_refused():
    """The C call: a count that does not divide the rows, one without indices, one on the decode path."""
    import ctypes
    import torch

    pkg = load_package()
    w8, native = pkg.w8a8_lora, pkg._native
    for m, per, indices, status in ((40, 3, True, -2), (40, 8, False, -2), (32, 8, True, -7)):  # (-2 SHAPE, -7 UNSUPPORTED)
        t = wc.to_torch(wc.make_case(m, 128, 256, n_adapters=2, rank=8, seed=m), "cuda:0")
        plan = w8.ForwardPlan(t["x"], t["weight"], t["a"], t["b"], t["s"], adapter_indices=t["idx"])
        whole = native.ProblemZ(call=plan.problem, rows_per_index=per)
        whole.call.struct_size = ctypes.sizeof(native.ProblemZ)
        if not indices:
            whole.call.adapter_indices = None
        got = native.load().mi355_w8a8_forward_v1(ctypes.byref(whole.call), torch.cuda.current_stream().cuda_stream)
        assert got == status
