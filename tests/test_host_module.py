"""The host module is an extension of one torch: where it is missing or another torch's, calls go the general way, as they did without it."""

import warnings

import pytest

from __graft_entry__ import load_package


@pytest.fixture
def native(monkeypatch):
    n = load_package()._native
    if not n.LIB_PATH.exists():
        pytest.skip("libmi355_w8a8.so not built (run __graft_entry__.build())")
    monkeypatch.setattr(n, "_host", None)
    monkeypatch.setattr(n, "_host_tried", False)
    return n


def test_the_built_module_is_this_torchs(native):
    import torch

    with warnings.catch_warnings():
        warnings.simplefilter("error")
        module = native.host()
    assert module.torch_version == torch.__version__ and native.host() is module


def test_a_missing_module_is_reported_once(native, monkeypatch, tmp_path):
    monkeypatch.setattr(native, "HOST_PATH", tmp_path / "mi355_w8a8_host.so")
    with pytest.warns(RuntimeWarning, match="mi355_w8a8_host.so"):
        assert native.host() is None
    with warnings.catch_warnings():
        warnings.simplefilter("error")
        assert native.host() is None


def test_another_torchs_module_is_not_used(native, monkeypatch):
    import torch

    monkeypatch.setattr(torch, "__version__", "0.0")
    with pytest.warns(RuntimeWarning, match="built against"):
        assert native.host() is None


@pytest.mark.gpu
def test_calls_without_it(native, monkeypatch):
    import torch
    import w8a8_cases as wc

    pkg = load_package()
    print("[case] calls without the host module", flush=True)
    t = wc.to_torch(wc.make_case(33, 264, 136, n_adapters=2, rank=8, seed=3), "cuda:0")
    args, kw = (t["x"], t["weight"], t["a"], t["b"], t["s"]), dict(adapter_indices=t["idx"])
    w = pkg.quantized_lora.quantize_frozen_weight(torch.randn((256, 72), device="cuda:0"), bits=4, group_size=64)
    x = torch.randn((5, 256), device="cuda:0").bfloat16()
    want = pkg.w8a8_lora.forward(*args, **kw), pkg.gq_linear.forward(x, w)
    assert native.host() is not None
    monkeypatch.setattr(native, "_host", None)
    for got, ref in zip((pkg.w8a8_lora.forward(*args, **kw), pkg.gq_linear.forward(x, w)), want):
        assert torch.equal(got.view(torch.int16), ref.view(torch.int16))
