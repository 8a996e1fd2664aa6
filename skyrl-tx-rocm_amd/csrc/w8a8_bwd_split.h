// The pull-backs' division of work, as plain arithmetic: the host's rule and what the kernels derive from it.
#pragma once
#include <cstdint>

namespace w8a8 {

// How the pull-back's tiles of 256 x 256 are spread over the chip: whole tiles while they come in full rounds of
// 256 workgroups, the rest split along the contraction so that the last round takes its share of the time
// and not all of it (sk_wgs workgroups of sk_q stages each; 0: no split).
struct BwdDxSplit { uint32_t direct_tiles, sk_q, sk_wgs; };

// Costs in stage times (0.98 us: 256 whole tiles of 128 stages 125 us in either kernel, of 768 754; the group-scaled one's stages have
// as many MFMAs): a split adds the partial tiles' way through memory, 256 KiB written and read again for every workgroup and split tile
// (about 0.11 each at 4.7 TB/s), and a launch.  The weights were taken with kernels of eight waves, 1.05 and 1.1 us a stage.
// Pull-back + finish, us, those kernels whole / split, and split as it is now: 2048 x 2560, N = 10240 (80 tiles of 320
// stages) 339 / 135 + 22, 105 + 15; 3003 x 4096, N = 24576 (192 of 768) 800 / 657 + 29, 535 + 22; 3003 x 12288, N = 4096 (64 of 576
// left over) 278 + 13 now.  Group-scaled, with what goes before the pull-back, whole / split, and the two alone now: 200 x 4096 <- 4096
// 150 / 57, 23 + 7; 800 x 12288 <- 4096 (128 tiles left over of 384) 285 / 230, 172 + 8; 1536 x 12288 <- 4096 (64 of 576) 434 / 355,
// 272 + 8; 1536 x 2560 <- 6144 221 / 142, 86 + 11.
// Calls of fewer than 64 stages (N < 2048) stay whole: little to gain, and a grouped call over the same rows
// then gives the same bits.
// k_blocks: k blocks of a wave's tile (2; 1 in the group-scaled kernel, whose partial tiles are half the size).
inline BwdDxSplit bwd_dx_split(uint32_t tiles_m, uint32_t tiles_k, uint32_t NB, uint32_t k_blocks = 2u) {
  const uint32_t ntile = tiles_m * tiles_k, rem = ntile % 256u;
  BwdDxSplit best{ntile, 0u, 0u};
  if (rem == 0u || NB < 64u) return best;
  double cost = 0.9 * NB;
  for (uint32_t wgs = 64u; wgs <= 256u; wgs += 64u) {
    uint32_t q = (rem * NB + wgs - 1u) / wgs;
    q = ((q < 16u ? 16u : q) + 1u) / 2u * 2u;
    const double c = q + 0.055 * k_blocks * (wgs + rem) + 8.0;
    if (c < cost) {
      cost = c;
      best.direct_tiles = ntile - rem; best.sk_q = q;
      best.sk_wgs = ((rem * NB + q - 1u) / q + 7u) / 8u * 8u;
    }
  }
  return best;
}

// The packed block that the group-scaled pull-back reads for n block nb.  dy is padded to n blocks beyond the packed weight's
// weight_nb, and a split segment may begin there: those read the last block again (dy is zero).
constexpr uint32_t gq_bwd_first_block(uint32_t nb, uint32_t weight_nb) { return nb < weight_nb ? nb : weight_nb - 1u; }
// whether n block nb reads the packed block behind that of nb - 1
constexpr bool gq_bwd_next_block(uint32_t nb, uint32_t weight_nb) { return nb < weight_nb; }

}  // namespace w8a8
