"""Codes of decode rows whose scale is not an ordinary number, whose quotients lie on ties, or that hold a NaN or an infinity,
against the rule in float64 (exact for bf16 values): clamp(rint(float32(v / scale)), -127, 127), a NaN at the lower limit."""

import numpy as np
import pytest

from __graft_entry__ import load_package
import w8a8_cases as wc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,k", [(1, 32), (7, 2560), (16, 8224), (32, 12288)])
def test_codes_of_every_kind_of_row(m, k):
    import torch

    case = wc.make_case(m, k, 64, seed=m + k)
    x = torch.from_numpy(np.random.default_rng(k).standard_normal((m, k)).astype(np.float32)).to(torch.bfloat16)
    for row in range(m):
        kind = (row + m // 16) % 8
        if kind == 1: x[row] *= 2.0 ** -120     # (a scale below what the reciprocal serves)
        elif kind == 2: x[row] *= 2.0 ** 110
        elif kind == 3: x[row] = (torch.arange(k) % 255 - 127) * 0.5   # half integers over a scale of 1/2 .. 1
        elif kind == 4: x[row] = 0.0
        elif kind == 5: x[row, k // 3] = float("nan")
        elif kind == 6: x[row, k // 2] = float("inf")
        elif kind == 7: x[row] = torch.where(torch.arange(k) % 2 == 0, 64.0, -0.25 * (torch.arange(k) % 256))
    t = wc.to_torch(case, "cuda:0")
    _, aux = load_package().w8a8_lora.forward(x.cuda(), t["weight"], return_aux=True, flags=load_package()._native.FLAG_FORCE_SKINNY)
    v = x.float().numpy()
    amax = np.nanmax(np.abs(v), axis=1)
    scale = np.where(amax > 0, amax / np.float32(127), np.float32(1)).astype(np.float32)
    with np.errstate(invalid="ignore"):
        q = (v / scale[:, None]).astype(np.float32)
    codes = np.clip(np.rint(np.where(np.isnan(q), np.float32(-127), q)), -127, 127).astype(np.int8)
    np.testing.assert_array_equal(aux["x_scales"].cpu().numpy(), scale)
    np.testing.assert_array_equal(aux["x_codes"].cpu().numpy(), codes)


@pytest.mark.parametrize("t,e,k", [(1, 8, 8), (3, 64, 64), (5, 70, 9), (9, 1000, 64)])
def test_route_of_equal_and_missing_probabilities(t, e, k):
    """Few distinct logits, minus infinities (probability zero) and top_k up to the experts: the selection is the stable order."""
    import torch

    pkg = load_package()
    logits = torch.from_numpy(np.random.default_rng(e).integers(0, 4, (t, e)).astype(np.float32))
    logits[:, 1::3] = float("-inf")
    weights, selected = pkg.w8a8_lora.moe_route(logits.cuda(), k, False)[:2]
    prob = torch.softmax(logits, dim=-1)
    order = torch.argsort(prob, dim=-1, descending=True, stable=True)[:, :k]
    torch.testing.assert_close(selected.cpu().long(), order, rtol=0, atol=0)
    # both softmaxes round the exponential, a sum of at most e terms and the quotient
    torch.testing.assert_close(weights.cpu(), torch.gather(prob, 1, order), rtol=(e + 4) * 2.0 ** -24, atol=0)


@pytest.mark.parametrize("m,k", [(33, 64), (130, 2560), (600, 8224)])
def test_codes_of_every_kind_of_row_on_tiles(m, k):
    """The tiled prologues: a NaN takes the row's scale to 1, its own code and a value's below -128 are -128, above 127 127."""
    import torch

    pkg = load_package()
    case = wc.make_case(m, k, 64, n_adapters=3, rank=8, seed=m + k)
    x = torch.from_numpy(np.random.default_rng(k).standard_normal((m, k)).astype(np.float32)).to(torch.bfloat16)
    for row in range(m):
        kind = (row * 5) % 8
        if kind == 1: x[row] *= 2.0 ** -120
        elif kind == 2: x[row] *= 2.0 ** 110
        elif kind == 3: x[row] = (torch.arange(k) % 255 - 127) * 0.5
        elif kind == 4: x[row] = 0.0
        elif kind == 5: x[row] *= 100.0; x[row, k // 3] = float("nan")
        elif kind == 6: x[row, k // 2] = float("inf")
        elif kind == 7: x[row] = torch.where(torch.arange(k) % 2 == 0, 64.0, -0.25 * (torch.arange(k) % 256))
    t = wc.to_torch(case, "cuda:0")
    v = x.float().numpy()
    nan = np.isnan(v).any(axis=1)
    amax = np.nanmax(np.abs(v), axis=1)
    scale = np.where(nan | (amax == 0), np.float32(1), amax / np.float32(127)).astype(np.float32)
    with np.errstate(invalid="ignore"):
        q = (v / scale[:, None]).astype(np.float32)
    codes = np.clip(np.rint(np.where(np.isnan(q), np.float32(-128), q)), -128, 127).astype(np.int8)
    for lora in (False, True):
        args = (t["a"], t["b"], t["s"]) if lora else ()
        _, aux = pkg.w8a8_lora.forward(x.cuda(), t["weight"], *args, adapter_indices=t["idx"] if lora else None, return_aux=True,
                                       flags=pkg._native.FLAG_FORCE_TILED)
        np.testing.assert_array_equal(aux["x_scales"].cpu().numpy(), scale)
        np.testing.assert_array_equal(aux["x_codes"].cpu().numpy(), codes)
