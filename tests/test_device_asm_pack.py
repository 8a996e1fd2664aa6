"""The loads of B in bwd_pack_dy_kernel rely on the buffer's range check for the rank rows that do not exist.  The check compares the
lane's offset with the buffer's size less the scalar offset, so the scalar offset has to be zero (no GPU: the compiled code is read)."""

import re
import subprocess

import pytest

from __graft_entry__ import PKG_DIR, _load_build_module, load_package


def test_the_whole_offset_is_checked(tmp_path):
    build = _load_build_module()
    try:
        hipcc = build.find_hipcc()
    except RuntimeError as e:  # pragma: no cover - the image ships hipcc
        pytest.skip(str(e))
    flags = [f for f in build.HIPCC_FLAGS if f not in ("-shared", "-fPIC") and not f.startswith("-Wl,")]
    tu = tmp_path / "pack.hip"
    tu.write_text('#include "w8a8_backward.h"\nusing namespace w8a8;\n' +
                  "".join(f"template __global__ void w8a8::bwd_pack_dy_kernel<{rb}>(BwdPackDyArgs);\n" for rb in (1, 2)))
    proc = subprocess.run([hipcc, *flags, "--cuda-device-only", "-S", "-I", str(PKG_DIR / "csrc"), str(tu), "-o", str(tmp_path / "pack.s")],
                          capture_output=True, text=True)
    assert proc.returncode == 0, proc.stderr[-2000:]
    kernels = re.findall(r"^(_ZN4w8a8\d+bwd_pack_dy_kernel\S+):(.*?)^\.Lfunc_end", (tmp_path / "pack.s").read_text(), re.M | re.S)
    assert len(kernels) == 2
    for name, text in kernels:
        loads = re.findall(r"buffer_load_dwordx4 v\[\d+:\d+\], (\S+), s\[\d+:\d+\], (\S+) offen", text)
        assert len(loads) >= 8 and {scalar for _, scalar in loads} == {"0"}, name


@pytest.mark.gpu
@pytest.mark.parametrize("rank", [1, 33, 64])
@pytest.mark.parametrize("n", [8, 40, 264, 312, 2056])
def test_nothing_behind_b_is_read(rank, n):
    """B at the front of a buffer whose rest is infinite: a rank row or column that does not exist would spoil dx, dA and dB."""
    import torch

    pkg = load_package()
    w8, ql = pkg.w8a8_lora, pkg.quantized_lora
    m, k, n_ad, dev = 70, 72, 2, "cuda:0"
    print(f"[case] pack dy {m}x{k}x{n} rank={rank}", flush=True)
    g = torch.Generator(device=dev).manual_seed(n + rank)
    rnd = lambda *s: torch.randn(s, generator=g, device=dev)
    codes = torch.randint(-127, 128, (k, n), generator=g, device=dev, dtype=torch.int8)
    scales = (torch.rand((1, n), generator=g, device=dev) + 0.5) / 127
    w = ql.GroupQuantizedWeight(codes, scales, k, k, 8, k)
    x, dy, a = rnd(m, k).bfloat16(), rnd(m, n).bfloat16(), (rnd(n_ad, k, rank) * 0.1).bfloat16()
    room = torch.full((n_ad * rank * n + 64 * n + 1024,), float("inf"), device=dev, dtype=torch.bfloat16)
    b = room[:n_ad * rank * n].view(n_ad, rank, n)
    b.copy_(rnd(n_ad, rank, n))
    s = torch.tensor([0.5, 2.0], device=dev)
    idx = torch.randint(0, n_ad, (m,), generator=g, device=dev, dtype=torch.int32)
    dx, da, db, _ = w8.backward(x, dy, w, a, b, s, adapter_indices=idx)
    d = dy.double()
    deq = (codes.float() * scales).bfloat16().double()
    want, size = d @ deq.T, d.abs() @ deq.abs().T
    for ad in range(n_ad):
        rows = (idx == ad).nonzero().flatten()
        ax, bx, xr, dr, sc = a[ad].double(), b[ad].double(), x[rows].double(), d[rows], s[ad].double()
        rs, rs_size = (dr @ bx.T) * sc, (dr.abs() @ bx.abs().T) * sc
        want[rows] += rs @ ax.T
        size[rows] += rs_size @ ax.abs().T
        # one rounding to bf16 and float32 sums of the terms in any order
        for got, ref, mag, terms in ((da[ad], xr.T @ rs, xr.abs().T @ rs_size, m + n),
                                     (db[ad], ((xr @ ax).T @ dr) * sc, ((xr.abs() @ ax.abs()).T @ dr.abs()) * sc, m + k)):
            assert ((got.double() - ref).abs() <= 2.0 ** -8 * ref.abs() + terms * 2.0 ** -23 * mag).all()
    assert ((dx.double() - want).abs() <= 2.0 ** -8 * want.abs() + (n + rank) * 2.0 ** -23 * size).all()
