"""The attention input stage at head widths about the 256 that one piece a lane holds, sums not divided by a power of two, and
fewer units than a workgroup has waves; the oracle comparisons (and bounds) of the two directions' own tests."""

import pytest

import test_gpu_qkv as forward
import test_gpu_qkv_backward as backward
from test_gpu_qkv import dev, pkg  # noqa: F401  (fixtures)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hq,hkv,d,rot,rows", [(1, 1, 252, 40, 7), (2, 1, 260, 8, 5), (5, 5, 384, 256, 9), (1, 1, 512, 128, 3), (3, 1, 12, 8, 65)])
def test_head_widths(dev, pkg, hq, hkv, d, rot, rows):  # noqa: F811
    forward.test_split_norm_rope_matches_oracle(dev, pkg, hq, hkv, d, rot, rows)
    backward.test_split_norm_rope_backward_matches_oracle(dev, pkg, hq, hkv, d, rot, rows)


@pytest.mark.parametrize("d,offset", [(256, 0), (130, 0), (260, 8), (64, 3)])
def test_bf16_norm_weights(dev, pkg, d, offset):  # noqa: F811
    """The model's bf16 weights read as they are, or converted where they do not lie on 16 bytes: the bits of their float32 copies."""
    import torch

    w8 = pkg.w8a8_lora
    cfg = w8.Qwen35QKVStageConfig(4, 2, d, d // 4 * 2, 10_000.0, 1e-6)
    g = torch.Generator("cuda").manual_seed(d)
    rand = lambda *shape: torch.randn(*shape, device=dev, generator=g).to(torch.bfloat16)
    fused, pos = rand(9, cfg.fused_width), torch.arange(9, device=dev)
    q_w, k_w = (rand(d + offset)[offset:] * 0.1 if not offset else rand(d + offset)[offset:] for _ in range(2))
    cots = (rand(9, 4, d), rand(9, 2, d), rand(9, 2, d), rand(9, 4 * d))
    for p, q in zip(w8.qkv_split_norm_rope(fused, q_w, k_w, pos, cfg), w8.qkv_split_norm_rope(fused, q_w.float(), k_w.float(), pos, cfg)):
        assert torch.equal(p, q)
    for need in (False, True):
        got, want = (w8.qkv_split_norm_rope_backward(fused, a, b, pos, cfg, *cots, need_norm_weight_grads=need)
                     for a, b in ((q_w, k_w), (q_w.float(), k_w.float())))
        for p, q in zip(got, want):
            assert (p is None and q is None) or torch.equal(p, q)
