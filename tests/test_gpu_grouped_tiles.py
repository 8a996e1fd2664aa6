"""The grouped GEMM's row tiles: groups at the edges of a 32-row block and of a tile of either height, groups cut
into several tiles, fewer and more tiles than workgroups, the shortest K of either height, ragged N, and
ranks on both sides of the staged epilogue -- each against the oracle."""

import numpy as np
import pytest

from __graft_entry__ import load_package
from oracle import w8a8_oracle as o

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes,k,n,rank,swiglu", [
    ([1, 0, 31, 32, 33, 0, 127, 128, 129], 128, 264, 16, False),      # two k steps: low tiles only
    ([255, 1, 256, 257, 96], 256, 520, 16, True),                      # tall (forced below) at the shortest K they take
    ([520, 3, 260], 320, 257, 9, False),                               # three and two tall tiles of a group, odd N
    ([700, 2], 192, 130, 16, True),                                    # six low tiles of a group
    ([0, 0, 5], 256, 36, 8, False), ([100, 0, 200], 640, 300, 40, False),
    ([2] * 45, 256, 1792, 16, True), ([100] * 40, 256, 2048, 12, False), ([100] * 40, 256, 2048, 20, False),  # more tiles than workgroups
    ([0, 0], 256, 64, 16, False),
])
def test_row_tiles(sizes, k, n, rank, swiglu):
    import torch

    w8 = load_package().w8a8_lora
    rng = np.random.default_rng(len(sizes) * 1000 + k + n)
    e, m = len(sizes), sum(sizes) + 3
    x = o.bf16_round(rng.standard_normal((m, k)).astype(np.float32))
    codes = rng.integers(-127, 128, (e, k, n), dtype=np.int8)
    scales = rng.uniform(0.001, 0.01, (e, n)).astype(np.float32)
    a = o.bf16_round((rng.standard_normal((e, k, rank)) * 0.02).astype(np.float32))
    b = o.bf16_round((rng.standard_normal((e, rank, n)) * 0.02).astype(np.float32))
    s = np.float32(1.5)
    xc, _ = o.quantize_rows(x)
    pre, acc = np.zeros((m, n), np.float32), np.zeros((m, n), np.int32)
    r0 = 0
    for g, rows in enumerate(sizes):
        r1 = r0 + rows
        if rows:
            w = o.GroupQuantizedWeight(codes[g], scales[g:g + 1], k, k, 8, k)
            pre[r0:r1] = o.quantized_lora_linear_f32(x[r0:r1], w, a[g], b[g], s)
            acc[r0:r1] = o.int_matmul(xc[r0:r1], codes[g])
        r0 = r1
    want = o.bf16_round(pre)
    want = o.swiglu_from_interleaved(want) if swiglu else want
    dev = torch.device("cuda:0")
    bf = lambda t: torch.from_numpy(t).to(dev).to(torch.bfloat16)
    gw = w8.prepare_grouped_weight(torch.from_numpy(codes).to(dev), torch.from_numpy(scales).to(dev))
    print(f"[case] grouped tiles {sizes[:6]} x{e} k={k} n={n} rank={rank} swiglu={swiglu}", flush=True)
    out, aux = w8.grouped_forward(bf(x), torch.tensor(sizes, dtype=torch.int32), gw, bf(a), bf(b), float(s),
                                  swiglu=swiglu, return_aux=True)
    for flag in (256, 512):  # low and tall tiles
        same = w8.grouped_forward(bf(x), torch.tensor(sizes, dtype=torch.int32), gw, bf(a), bf(b), float(s), swiglu=swiglu,
                                  flags=flag)
        assert torch.equal(same.view(torch.int16), out.view(torch.int16))
    got = out.float().cpu().numpy()
    np.testing.assert_array_equal(aux["acc"].cpu().numpy(), acc)
    assert np.all(got[sum(sizes):] == 0)
    ok = o.within_tolerance(got, want)
    assert ok.all(), int((~ok).sum())


@pytest.mark.parametrize("m,x_rows,repeat,k,rank", [
    (40, 5, 8, 136, 16), (300, 700, 1, 512, 24), (4100, 513, 8, 320, 8), (4097, 5000, 1, 256, 0), (24, 24, 3, 1032, 40),
    (4097, 600, 7, 256, 40), (8193, 1100, 8, 136, 0),
])
def test_mapped_rows_equal_gathered_rows(m, x_rows, repeat, k, rank):
    """Rows read through a map -- fewer source rows than rows (their statistics are taken per source row) and more,
    repeated and out of range entries, both workgroup sizes of the quantizer -- against the same rows gathered."""
    import torch

    w8 = load_package().w8a8_lora
    dev, e, n = torch.device("cuda:0"), 5, 264
    gen = torch.Generator(device=dev).manual_seed(m + k)
    x = torch.randn(x_rows, k, device=dev, generator=gen).to(torch.bfloat16)
    rmap = torch.randint(-3, x_rows * repeat + 9, (m,), device=dev, generator=gen, dtype=torch.int32)
    gw = w8.prepare_grouped_weight(torch.randint(-127, 128, (e, k, n), device=dev, generator=gen, dtype=torch.int8),
                                   torch.rand(e, n, device=dev, generator=gen) * 0.01)
    a = (torch.randn(e, k, rank, device=dev, generator=gen) * 0.02).to(torch.bfloat16) if rank else None
    b = (torch.randn(e, rank, n, device=dev, generator=gen) * 0.02).to(torch.bfloat16) if rank else None
    sizes = torch.tensor([m // 3, 0, m // 4, 7, m // 5], dtype=torch.int32)
    src = torch.div(rmap.clamp(min=0), repeat, rounding_mode="floor").clamp(max=x_rows - 1).long()
    print(f"[case] mapped rows m={m} x_rows={x_rows} repeat={repeat} k={k} rank={rank}", flush=True)
    want, want_aux = w8.grouped_forward(x[src], sizes, gw, a, b, 1.0 if rank else None, return_aux=True)
    got, aux = w8.grouped_forward(x, sizes, gw, a, b, 1.0 if rank else None, row_map=rmap, row_repeat=repeat, return_aux=True)
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))
    for name in ("x_codes", "x_scales", "acc"):
        assert torch.equal(aux[name], want_aux[name])
