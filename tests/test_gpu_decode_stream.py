"""The forms of the weight-streaming decode kernel: one or two column slices per workgroup (two: fused SwiGLU
and wide outputs), one or two row halves, every step count a wave keeps in flight (by K) and the rounds beyond
it, odd N and ranks (whose B rows start in the middle of a dword), each against the oracle."""

import numpy as np
import pytest

from __graft_entry__ import load_package
import w8a8_cases as wc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,k,n,n_ad,rank,form", [
    (1, 2048, 520, 2, 64, "swiglu"), (16, 4096, 264, 16, 32, "swiglu"), (17, 4104, 136, 3, 64, "swiglu"),
    (32, 2048, 96, 4, 7, "swiglu"), (5, 8192, 260, 0, 0, "swiglu"),
    (3, 256, 16402, 2, 12, "plain"), (20, 512, 16384, 3, 33, "plain"),      # two slices, no SwiGLU
    (9, 6144, 97, 5, 5, "residual"), (31, 16384, 33, 3, 9, "plain"),        # odd N; K in more than one round
    (16, 16384, 129, 4, 33, "rms"), (18, 12288, 64, 2, 64, "residual"), (2, 1024, 17, 1, 3, "rms"),
])
def test_decode_stream_forms(m, k, n, n_ad, rank, form):
    pkg = load_package()
    case = wc.make_case(m, k, n, n_adapters=n_ad, rank=max(rank, 1), seed=m * 7 + n, rms=form in ("swiglu", "rms"),
                        swiglu=form == "swiglu", residual=form == "residual")
    st = wc.oracle_forward(case, return_stages=True)
    print(f"[case] decode {m}x{k}x{n} adapters={n_ad} rank={rank} {form}", flush=True)
    got, aux = wc.gpu_forward(case, flags=pkg._native.FLAG_FORCE_SKINNY)
    np.testing.assert_array_equal(aux["x_codes"], st["x_codes"])
    np.testing.assert_array_equal(aux["acc"], st["acc"])
    rep = wc.compare(got, st["out"])
    assert rep["violations"] == 0, rep
