"""The tiled path's prologue without auxiliary outputs (the normalized rows then exist in registers only):
K tails inside a 32-wide block and a 128-wide step, rows of one and of several 8 KiB pieces, every rank block
count, ranks and widths that are no multiple of four, adapters in one and in several 1024-row passes of the
sort -- against the oracle, and bit for bit against the call that writes the normalized rows."""

import numpy as np
import pytest

from __graft_entry__ import load_package
import w8a8_cases as wc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,k,n,n_ad,rank,rms", [
    (33, 40, 72, 2, 5, True), (150, 1000, 260, 3, 16, True), (70, 4104, 129, 1, 33, True),
    (2100, 264, 132, 64, 30, True), (97, 5000, 96, 0, 0, True), (41, 12288, 100, 5, 64, True),
    (1025, 136, 131, 7, 8, False), (64, 16384, 64, 2, 32, False),
])
def test_prologue_without_aux_outputs(m, k, n, n_ad, rank, rms):
    nat = load_package()._native
    case = wc.make_case(m, k, n, n_adapters=n_ad, rank=max(rank, 1), seed=m + k, rms=rms)
    print(f"[case] prologue {m}x{k}x{n} adapters={n_ad} rank={rank} rms={rms}", flush=True)
    st = wc.oracle_forward(case, return_stages=True)
    got = wc.gpu_forward(case, flags=nat.FLAG_FORCE_TILED, return_aux=False)
    rep = wc.compare(got, st["out"])
    assert rep["violations"] == 0, rep
    with_aux, aux = wc.gpu_forward(case, flags=nat.FLAG_FORCE_TILED)
    np.testing.assert_array_equal(aux["x_codes"], st["x_codes"])
    np.testing.assert_array_equal(got.view(np.uint32), with_aux.view(np.uint32))
