"""The grouped call's copies of codes and scales are what its GEMM multiplied, row for row -- for rows with a NaN too, where
the scale rule leaves a choice -- and rows beyond the groups get their own."""

import pytest

from __graft_entry__ import load_package

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mapped", [False, True])
def test_copies_are_what_was_multiplied(mapped):
    import torch

    w8 = load_package().w8a8_lora
    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(4)
    e, k, n, sizes = 3, 136, 72, [5, 0, 40]
    m = sum(sizes) + 4
    x = torch.randn(m, k, device=dev, generator=g).to(torch.bfloat16)
    x[2, 7], x[30, 135], x[31, 0] = float("nan"), float("nan"), float("inf")
    codes = torch.randint(-127, 128, (e, k, n), device=dev, generator=g, dtype=torch.int8)
    gw = w8.prepare_grouped_weight(codes, torch.rand(e, n, device=dev, generator=g) * 0.01)
    kw = {"row_map": torch.arange(m, device=dev, dtype=torch.int32) * 2, "row_repeat": 2} if mapped else {}
    _, aux = w8.grouped_forward(x, torch.tensor(sizes, dtype=torch.int32), gw, return_aux=True, **kw)
    xc, r0 = aux["x_codes"].cpu().long(), 0
    for gi, rows in enumerate(sizes):
        want = xc[r0:r0 + rows] @ codes[gi].cpu().long()
        assert torch.equal(aux["acc"].cpu().long()[r0:r0 + rows], want)
        r0 += rows
    assert aux["x_scales"][2] == 1.0  # (no maximum: the comparison amax > 0 fails)
    plain, scales = w8.dynamic_quantize_rows(x)
    rest = [i for i in range(m) if i not in (2, 30, 31)]
    assert torch.equal(aux["x_codes"][rest], plain[rest]) and torch.equal(aux["x_scales"][rest], scales[rest])
