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
