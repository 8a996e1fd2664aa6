"""Autograd rule of the group-scaled linear: which calls the kernels may take.  The kernels' results carry no
graph, so a backward that is itself recorded (create_graph) has to run as torch operations.  On the CPU the
native calls are replaced by stand-ins without a graph; the GPU test runs the real ones."""

import contextlib
import types

import pytest
import torch

from __graft_entry__ import load_package

pkg = load_package()
ql, gq = pkg.quantized_lora, pkg.gq_linear


def _setup(dev, m=5, k=64, n=24, rank=8, seed=0):
    g = torch.Generator().manual_seed(seed)
    rnd = lambda *s: torch.randn(*s, generator=g).to(torch.bfloat16).to(dev)
    w = ql.quantize_frozen_weight(torch.randn(k, n, generator=g).to(dev), bits=8, group_size=32)
    x, a, b = (t.requires_grad_() for t in (rnd(m, k), rnd(k, rank), rnd(rank, n)))
    return w, x, a, b


def _rule(w, x, a, b, s):
    """The straight-through forward whose derivative the rule is, in the operands' precision."""
    deq = ql.dequantize_frozen_weight(w).to(x.dtype).to(x.device)
    return x @ deq + ((x @ a) @ b) * s


@pytest.fixture
def stand_ins(monkeypatch):
    calls = []

    def forward(x, weight, lora_a=None, lora_b=None, lora_scaling=None, *, activation_bits=8):
        with torch.no_grad():
            return _rule(weight, x.float(), lora_a.float(), lora_b.float(), float(lora_scaling)).to(torch.bfloat16)

    def backward(x, dy, weight, lora_a, lora_b, lora_scaling, *, need_dx=True, need_lora_grads=True):
        calls.append(tuple(dy.shape))
        with torch.no_grad():
            f = [t.float() for t in (x, dy, lora_a, lora_b)]
            r = (f[1] @ f[3].T) * float(lora_scaling)
            z = f[0] @ f[2]
            return ((f[1] @ ql.dequantize_frozen_weight(weight).T + r @ f[2].T).to(x.dtype), (f[0].T @ r).to(x.dtype),
                    ((z.T @ f[1]) * float(lora_scaling)).to(x.dtype), (f[1] * (z @ f[3])).sum().reshape(1))

    monkeypatch.setattr(gq, "forward", forward)
    monkeypatch.setattr(gq, "backward", backward)
    monkeypatch.setattr(gq, "has_native_backward", lambda *args: True)
    return calls


def _penalised(w, x, a, b, y):
    """Gradients of a loss that holds the square of another gradient."""
    dx, = torch.autograd.grad(y.float().sum(), x, create_graph=True)
    assert dx.requires_grad
    return torch.autograd.grad(y.float().sum() + dx.float().pow(2).sum(), (a, b))


def _reference(w, x, a, b, s):
    leaves = [t.detach().cpu().double().requires_grad_() for t in (x, a, b)]
    w64 = ql.GroupQuantizedWeight(w.codes.cpu(), w.scales.cpu(), w.original_in_features, w.padded_in_features, w.bits,
                                  w.group_size)
    return _penalised(w64, *leaves, _rule(w64, *leaves, s))


def _close(got, want):
    for g, r in zip(got, want):  # products of bf16 values; dx is rounded to bf16 (2^-9) before it is squared
        assert (g.detach().cpu().double() - r).norm() <= 2.0 ** -6 * r.norm()


def test_recorded_backward_keeps_its_graph(stand_ins):
    w, x, a, b = _setup("cpu")
    y = ql.quantized_lora_linear(x, w, a, b, 0.5)
    _close(_penalised(w, x, a, b, y), _reference(w, x, a, b, 0.5))


def test_plain_backward_takes_the_kernels(stand_ins):
    w, x, a, b = _setup("cpu")
    ql.quantized_lora_linear(x, w, a, b, 0.5).float().sum().backward()
    assert stand_ins == [(5, 24)]


@pytest.mark.gpu
def test_second_derivatives_on_the_gpu():
    w, x, a, b = _setup("cuda:0", m=40, k=128, n=72)
    y = ql.quantized_lora_linear(x, w, a, b, 0.5)
    _close(_penalised(w, x, a, b, y), _reference(w, x, a, b, 0.5))


def _shifted(t, by=1):
    """The same values as a contiguous view that starts `by` elements into its storage (a flat parameter buffer)."""
    flat = torch.zeros(t.numel() + by, dtype=t.dtype, device=t.device)
    flat[by:] = t.detach().reshape(-1)
    return flat[by:].reshape(t.shape)


def test_operands_reach_the_kernels_aligned(monkeypatch):
    """The entry point refuses operands off a 16-byte boundary; the forward takes them, so the backward has to."""
    w, x, a, b = _setup("cpu")
    seen = {}

    def entry(ref, stream):
        p = ref._obj
        seen.update({f: getattr(p, f) for f in ("x", "dy", "w_packed", "w_scales", "lora_a", "lora_b", "dx", "d_lora_a", "d_lora_b")})
        return 0

    lib = types.SimpleNamespace(mi355_w8a8_gq_bwd_workspace_bytes=lambda *dims: 256, mi355_w8a8_gq_linear_bwd_v1=entry)
    monkeypatch.setattr(gq._native, "load", lambda: lib)
    monkeypatch.setattr(gq, "_require_cuda", lambda *args: None)
    monkeypatch.setattr(gq, "_on", lambda dev: contextlib.nullcontext())
    monkeypatch.setattr(gq, "_stream_ptr", lambda dev: 0)
    pw = gq.PackedGroupWeight(torch.zeros(64 * 24, dtype=torch.uint8), _shifted(w.scales.float()), 64, 64, 24, 8, 32)
    gq.backward(_shifted(x), _shifted(torch.zeros(5, 24, dtype=torch.bfloat16)), pw, _shifted(a, 3), _shifted(b), torch.tensor(0.5))
    assert seen and all(ptr % 16 == 0 for ptr in seen.values()), seen


@pytest.mark.gpu
def test_operands_at_odd_offsets():
    w, x, a, b = _setup("cuda:0", m=40, k=128, n=72)
    w = ql.GroupQuantizedWeight(w.codes, _shifted(w.scales.float()), w.original_in_features, w.padded_in_features, w.bits,
                                w.group_size)
    dy = torch.randn(40, 72, device="cuda:0").to(torch.bfloat16)
    grads = []
    for shift in (lambda t: t.detach().clone(), _shifted):
        leaves = [shift(t).requires_grad_() for t in (x, a, b)]
        y = ql.quantized_lora_linear(leaves[0], w, leaves[1], leaves[2], 0.5)
        grads.append(torch.autograd.grad(y, leaves, shift(dy)))
    assert all(torch.equal(p, q) for p, q in zip(*grads))


@pytest.mark.parametrize("m,k,n,group,rank,covered", [
    (4096, 12288, 4096, 128, 32, True),
    (350_000, 12288, 512, 128, 32, False),   # m * k beyond 32-bit offsets
    (350_000, 512, 12288, 128, 32, False),   # m * n
    (3, 60, 24, 32, 8, False), (3, 64, 20, 32, 8, False),  # K, N off a multiple of 8
    (0, 64, 24, 32, 8, False),
])
def test_which_calls_the_kernels_cover(m, k, n, group, rank, covered):
    if not pkg._native.LIB_PATH.exists():
        pytest.skip("libmi355_w8a8.so not built (run __graft_entry__.build())")
    k_pad = -(-k // group) * group
    pw = gq.PackedGroupWeight(torch.empty(0), torch.empty(0), k, k_pad, n, 8, group)
    assert gq.has_native_backward(pw, m, rank) is covered


def test_calls_beyond_the_kernels_take_the_library(stand_ins, monkeypatch):
    """The rule decides on the call at hand, rows and rank included."""
    asked = []
    monkeypatch.setattr(gq, "has_native_backward", lambda weight, rows, rank: asked.append((rows, rank)))
    w, x, a, b = _setup("cpu", m=6)
    y = ql.quantized_lora_linear(x.reshape(2, 3, 64), w, a, b, 0.5)
    got = torch.autograd.grad(y.float().sum(), (a, b))
    leaves = [t.detach().double().requires_grad_() for t in (x, a, b)]
    _close(got, torch.autograd.grad(_rule(w, *leaves, 0.5).sum(), leaves[1:]))
    assert asked == [(6, 8)] and not stand_ins
