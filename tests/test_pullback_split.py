"""The weight blocks that the group-scaled pull-back reads, walked on the host for every segment of the split rule: dy is
padded to whole tiles of 256 columns, the packed weight ends with its last block of 32."""

import shutil
import subprocess

import pytest

from __graft_entry__ import PKG_DIR, load_package

WALK = r"""
#include <cstdio>
#include "w8a8_bwd_split.h"
using namespace w8a8;
int main() {
  long walked = 0, beyond = 0;
  for (uint32_t tiles_m = 1; tiles_m <= 5; ++tiles_m)
    for (uint32_t tiles_k = 1; tiles_k <= 128; ++tiles_k)
      for (uint32_t weight_nb = 1; weight_nb <= 200; ++weight_nb) {
        const uint32_t NB = (weight_nb + 7u) / 8u * 8u;
        const BwdDxSplit split = bwd_dx_split(tiles_m, tiles_k, NB, 1u);
        auto walk = [&](uint32_t nb0, uint32_t len) {  // as gq_bwd_dx_wide_kernel's issue()
          uint32_t block = gq_bwd_first_block(nb0, weight_nb);
          for (uint32_t nb = nb0;; ) {
            const uint32_t want = nb < weight_nb ? nb : weight_nb - 1u;
            if (block != want || block >= weight_nb) {
              std::printf("tiles %u x %u, %u blocks: segment from %u reads block %u for %u\n", tiles_m, tiles_k, weight_nb, nb0, block, nb);
              return false;
            }
            if (++nb >= nb0 + len) break;
            block += gq_bwd_next_block(nb, weight_nb) ? 1u : 0u;
          }
          ++walked;
          beyond += nb0 >= weight_nb;
          return true;
        };
        if (split.direct_tiles && !walk(0u, NB)) return 1;
        const uint32_t total = (tiles_m * tiles_k - split.direct_tiles) * NB;
        for (uint32_t w = 0; w < split.sk_wgs; ++w)  // as bwd_dx_schedule
          for (uint32_t s0 = w * split.sk_q, s1 = s0 + split.sk_q < total ? s0 + split.sk_q : total; s0 < s1;) {
            const uint32_t nb0 = s0 % NB, len = s1 - s0 < NB - nb0 ? s1 - s0 : NB - nb0;
            if (!walk(nb0, len)) return 1;
            s0 += len;
          }
      }
  std::printf("%ld segments, %ld from beyond the weight\n", walked, beyond);
  return beyond > 0 ? 0 : 2;
}
"""


def test_no_segment_reads_beyond_the_packed_weight(tmp_path):
    cxx = shutil.which("g++") or shutil.which("clang++")
    if cxx is None:
        pytest.skip("no C++ compiler")
    (tmp_path / "walk.cc").write_text(WALK)
    exe = tmp_path / "walk"
    subprocess.run([cxx, "-std=c++17", "-O2", f"-I{PKG_DIR / 'csrc'}", str(tmp_path / "walk.cc"), "-o", str(exe)], check=True)
    run = subprocess.run([str(exe)], capture_output=True, text=True)
    assert run.returncode == 0, run.stdout
    kernel = (PKG_DIR / "csrc" / "w8a8_gq_bwd.h").read_text()
    assert "gq_bwd_first_block((uint32_t)nb0, a.weight_nb) * w_stride" in kernel and "gq_bwd_next_block((uint32_t)nb_load, a.weight_nb)" in kernel


@pytest.mark.gpu
@pytest.mark.parametrize("m,k,n,bits", [(64, 12288, 2568, 8), (64, 12288, 2568, 4)])
def test_segments_from_beyond_the_weight(m, k, n, bits):
    """81 blocks of the weight, 88 of dy, workgroups of 34 stages: segments begin at blocks 82, 84 and 86."""
    import torch

    pkg = load_package()
    print(f"[case] pull-back {m} x {k} <- {n}, {bits} bits", flush=True)
    g = torch.Generator(device="cuda:0").manual_seed(n)
    w = pkg.quantized_lora.quantize_frozen_weight(torch.randn((k, n), generator=g, device="cuda:0") * 0.02, bits=bits, group_size=64)
    dy = torch.randn((m, n), generator=g, device="cuda:0").to(torch.bfloat16)
    x, a, b = (torch.zeros(shape, device="cuda:0", dtype=torch.bfloat16) for shape in ((m, k), (k, 8), (8, n)))
    got = pkg.gq_linear.backward(x, dy, w, a, b, 1.0, need_lora_grads=False)[0].double()
    deq = pkg.quantized_lora.dequantize_frozen_weight(w).double()
    want, size = dy.double() @ deq.T, dy.double().abs() @ deq.abs().T
    # one rounding to bf16, float32 sums of n exact products in any order
    assert ((got - want).abs() <= 2.0 ** -8 * want.abs() + n * 2.0 ** -23 * size).all()
