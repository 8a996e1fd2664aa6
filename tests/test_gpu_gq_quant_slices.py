"""The group-scaled quantizer deals a row's groups to a number of waves that follows from the rows and K: the codes and scales
are those of the same rows in a call of 16, where sixteen waves share a row."""

import pytest

from __graft_entry__ import load_package

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [352, 353, 705, 1408, 2817])
@pytest.mark.parametrize("k,group", [(3072, 128), (3136, 64), (6400, 128), (9216, 3072)])
def test_codes_do_not_depend_on_the_slices(m, k, group):
    import torch

    pkg = load_package()
    print(f"[case] gq quantizer m={m} k={k} group={group}", flush=True)
    g = torch.Generator(device="cuda:0").manual_seed(m + k)
    x = torch.randn((m, k), generator=g, device="cuda:0").bfloat16()
    w = pkg.quantized_lora.quantize_frozen_weight(torch.randn((k, 64), generator=g, device="cuda:0"), bits=8, group_size=group)
    kw = dict(activation_bits=8, return_aux=True)
    _, aux = pkg.gq_linear.forward(x, w, **kw)
    for lo in (0, m // 2, m - 16):
        _, few = pkg.gq_linear.forward(x[lo:lo + 16].contiguous(), w, **kw)
        assert torch.equal(aux["x_codes"][lo:lo + 16], few["x_codes"])
        assert torch.equal(aux["x_scales"][lo:lo + 16], few["x_scales"])
