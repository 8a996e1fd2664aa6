"""Workspace of the backward calls: what the partial tiles of the split pull-back take."""

import pytest

from __graft_entry__ import load_package

MIB = 1 << 20


@pytest.fixture(scope="module")
def lib():
    native = load_package()._native
    if not native.LIB_PATH.exists():
        pytest.skip("libmi355_w8a8.so not built (run __graft_entry__.build())")
    return native.load()


def test_partial_tiles_follow_the_rows(lib):
    """4096 -> 4096: sixteen tiles of one row band over 128 workgroups, 32 KiB for every 32 rows of at most 144 partial tiles."""
    sizes = [lib.mi355_w8a8_bwd_workspace_bytes(m, 4096, 4096, 1, 16, 0) for m in (1, 32, 33, 256)]
    assert sizes[0] <= 10 * MIB
    assert sizes[1] - sizes[0] < MIB and sizes[2] - sizes[1] <= 5 * MIB
    assert sizes[3] <= 42 * MIB


@pytest.mark.parametrize("m,k,n", [(1, 4096, 4096), (256, 4096, 4096), (1536, 12288, 4096)])
def test_group_scaled_partial_tiles_are_half_the_size(lib, m, k, n):
    """Tiles of 128 k: at most 256 workgroups and 255 tiles, 128 KiB a whole tile; everything else as large as the
    operands it is a copy of."""
    total = lib.mi355_w8a8_gq_bwd_workspace_bytes(m, k, k, n, 64, 32)
    rows = -(-m // 256) * 256
    operands = rows * n * 2 + 2 * 32 * 4 * (k + n) * (m // 512 + 2) + rows * 64 * 4 * 12 + 2 * MIB
    blocks = min(8, -(-m // 32))
    assert total <= operands + (256 + 255) * blocks * MIB // 64
