"""The expert sort at the edges of a chunk and of the one-launch form, against a stable sort."""

import pytest

from __graft_entry__ import load_package

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pairs,groups,repeat", [
    (1, 1, 1), (64, 1024, 8), (1023, 128, 1), (1024, 3, 8), (1025, 128, 5), (16384, 128, 8), (16385, 1024, 1), (40000, 60, 8),
    (32768, 2, 8), (32769, 2, 1),
])
def test_sort_is_stable(pairs, groups, repeat):
    import torch

    w8 = load_package().w8a8_lora
    dev = torch.device("cuda:0")
    gen = torch.Generator(device=dev).manual_seed(pairs)
    idx = torch.randint(-2, groups + 2, (pairs,), device=dev, generator=gen, dtype=torch.int32)  # clamped into range
    adapters = torch.randint(0, 9, (pairs // repeat,), device=dev, generator=gen, dtype=torch.int32)
    print(f"[case] sort pairs={pairs} groups={groups} repeat={repeat}", flush=True)
    _, sizes, order, inverse, ads = w8.moe_dispatch(None, idx, groups, repeat=repeat, adapter_indices=adapters)
    host = idx.cpu().clamp(0, groups - 1).long()
    want = torch.sort(host, stable=True).indices
    assert torch.equal(order.cpu().long(), want)
    assert torch.equal(inverse.cpu().long()[want], torch.arange(pairs))
    assert torch.equal(sizes.cpu().long(), torch.bincount(host, minlength=groups))
    assert torch.equal(ads.cpu(), adapters.cpu()[torch.div(want, repeat, rounding_mode="floor")])
