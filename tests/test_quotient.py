"""The quantizers form codes without a division: q0 = v * r, corrected by its exact remainder.  Every bf16 significand of v
against every one of the largest value, for eight and four bits: the codes of the correctly rounded quotient."""

import numpy as np
import pytest

from __graft_entry__ import load_package

F = np.float32


def _significands():
    return (np.arange(128, 256) / 128.0).astype(F)


def _values():
    """Every bf16 significand at the exponents a code can come from (and some below)."""
    return (_significands()[None, :] * (2.0 ** np.arange(-20, 1))[:, None]).astype(F).reshape(-1)


@pytest.mark.parametrize("qmax", [127.0, 7.0])
def test_corrected_product_gives_the_codes_of_the_division(qmax):
    every = _values()
    for amax in _significands():
        v = every[every <= amax]
        scale = F(amax / F(qmax))
        want = np.rint(v / scale)
        near = F(1) / scale
        for r in (near, np.nextafter(near, F(2e9)), np.nextafter(near, F(0)), np.nextafter(np.nextafter(near, F(2e9)), F(2e9)),
                  np.nextafter(np.nextafter(near, F(0)), F(0))):  # the hardware reciprocal is within one unit
            q0 = v * r
            # (products of two float32 are exact in float64, and so is this difference)
            rem = (v.astype(np.float64) - q0.astype(np.float64) * np.float64(scale)).astype(F)
            q = (q0.astype(np.float64) + rem.astype(np.float64) * np.float64(r)).astype(F)
            code = (q + F(12582912.0)).view(np.uint32).astype(np.uint8).view(np.int8)
            np.testing.assert_array_equal(code, want.astype(np.int8))


def _rows(lead, group):
    """Rows whose groups start with the largest value: (rows, k) float32 with every pair of significands."""
    every = _values()
    per = group - 1
    groups = -(-every.size // per)
    rows = np.zeros((lead.size, groups, group), F)
    flat = np.zeros(groups * per, F)
    flat[:every.size] = every
    rows[:, :, 1:] = flat.reshape(groups, per)[None]
    rows[:, :, 0] = lead[:, None]
    rows[np.abs(rows) > lead[:, None, None]] = 0.0
    rows[:, :, 1::2] *= -1.0
    return rows.reshape(lead.size, -1)


def _expected(rows, group, qmax):
    r = rows.reshape(rows.shape[0], -1, group)
    amax = np.abs(r).max(axis=-1, keepdims=True)
    with np.errstate(invalid="ignore"):
        scale = np.where(amax > 0, amax / F(qmax), F(1)).astype(F)
    return np.rint(r / scale).astype(np.int8).reshape(rows.shape), scale[..., 0]


@pytest.mark.gpu
@pytest.mark.parametrize("bits", [8, 4])
@pytest.mark.parametrize("group", [32, 64, 128, 256])
def test_group_scaled_codes_of_every_pair(bits, group):
    import torch

    pkg = load_package()
    print(f"[case] codes of every pair, groups of {group}, {bits} bits", flush=True)
    lead = np.concatenate([_significands(), np.zeros(1, F)])
    rows = _rows(lead, group)
    want, scales = _expected(rows, group, 127.0 if bits == 8 else 7.0)
    x = torch.from_numpy(rows).to("cuda:0", torch.bfloat16)
    assert torch.equal(x.float().cpu(), torch.from_numpy(rows))
    w = pkg.quantized_lora.quantize_frozen_weight(torch.randn((rows.shape[1], 64), device="cuda:0"), bits=8, group_size=group)
    _, aux = pkg.gq_linear.forward(x, w, activation_bits=bits, return_aux=True)
    np.testing.assert_array_equal(aux["x_codes"].cpu().numpy(), want)
    np.testing.assert_array_equal(aux["x_scales"].cpu().numpy(), scales)


@pytest.mark.gpu
@pytest.mark.parametrize("flags", ["FLAG_FORCE_TILED", "FLAG_FORCE_TILED|FLAG_TILE_256X128"])
def test_per_channel_codes_of_every_pair(flags):
    import torch

    pkg = load_package()
    nat = pkg._native
    print(f"[case] per-channel codes of every pair {flags}", flush=True)
    values = _values()
    lead = np.concatenate([_significands(), np.zeros(3, F), _significands()[:5] * F(127.0)])
    rows = _rows(lead, values.size + 1)[:, :2688]
    want, scales = _expected(rows, rows.shape[1], 127.0)
    x = torch.from_numpy(rows).to("cuda:0", torch.bfloat16)
    rows = x.float().cpu().numpy()  # (127 times a significand has no bf16 value: what the call sees)
    want, scales = _expected(rows, rows.shape[1], 127.0)
    k = rows.shape[1]
    weight = pkg.quantized_lora.GroupQuantizedWeight(torch.ones((k, 64), dtype=torch.int8, device="cuda:0"),
                                                     torch.ones((1, 64), device="cuda:0"), k, k, 8, k)
    value = 0
    for name in flags.split("|"):
        value |= getattr(nat, name)
    _, aux = pkg.w8a8_lora.forward(x, weight, None, None, None, flags=value, return_aux=True)
    np.testing.assert_array_equal(aux["x_codes"].cpu().numpy(), want)
    np.testing.assert_array_equal(aux["x_scales"].cpu().numpy().reshape(-1), scales.reshape(-1))


@pytest.mark.gpu
@pytest.mark.parametrize("m,k", [(33, 512), (4400, 2560)])  # rows kept in the LDS, and read again
def test_codes_beside_a_nan(m, k):
    """A row with a NaN has scale one.  Its other values are clipped as int8, whatever else the wave holds: 127.5 is a bf16 value
    that rounds to 128."""
    import torch

    pkg = load_package()
    print(f"[case] codes beside a NaN {m}x{k}", flush=True)
    rows = np.zeros((m, k), F)
    rows[:, 1::4] = np.array([127.5, -127.5, 127.0, 126.5, -126.5, 0.5, 1.5, -0.5], F)[np.arange(k // 4) % 8]
    rows[3, 64:96:2] = 300.0  # (beyond the range, in one piece of the row only)
    rows[5, 96:128:2] = -300.0
    nan = [0, 3, 5, 18, m - 1]
    rows[nan, 0] = np.nan
    x = torch.from_numpy(rows).to("cuda:0", torch.bfloat16)
    w = pkg.quantized_lora.GroupQuantizedWeight(torch.ones((k, 64), dtype=torch.int8, device="cuda:0"), torch.ones((1, 64), device="cuda:0"),
                                                k, k, 8, k)
    _, aux = pkg.w8a8_lora.forward(x, w, None, None, None, flags=pkg._native.FLAG_FORCE_TILED, return_aux=True)
    want = np.clip(np.rint(np.where(np.isnan(rows[nan]), F(-128), rows[nan])), -128, 127).astype(np.int8)
    np.testing.assert_array_equal(aux["x_codes"][nan].cpu().numpy(), want)
    assert (aux["x_scales"].reshape(-1)[nan] == 1.0).all()
