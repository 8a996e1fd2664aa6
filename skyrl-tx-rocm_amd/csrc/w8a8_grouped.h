// Grouped int8 GEMM of the ragged expert call: group g multiplies its own rows with its own weight.
// Arithmetic and epilogue are those of w8a8_gemm.h (gemm_epilogue_block).
//
// Bound by the weights' way from HBM while a group has fewer than some 200 rows.  A tile is therefore as tall as the
// group allows (up to kRB 32-row blocks; a group of more blocks is cut into tiles of even height), so that
// every weight byte crosses L2 -> LDS once, and 256 columns wide: the tiles of 128 experts then come in many
// small pieces that fill whole rounds of the 256 CUs.  The tile table counts the tiles that exist; a workgroup
// takes its tiles from them alone, each XCD a contiguous range (the column tiles of one expert run side by side
// and find the activation panel in that L2).
//  * Workgroup = 8 waves, 4 along M x 2 along N.  Wave row w takes the tile's row blocks w and w + 4 (32 x 128
//    each): blocks that the tile lacks cost no MFMAs.  kRB = 4 (tiles of up to 128 rows) leaves LDS for six stages of 24 KiB,
//    kRB = 8 has four of 32 KiB.
//  * K advances in steps of 64 through that ring of LDS stages.  The loads are assembly statements with counted
//    waits: behind the load builtin the compiler drains every counter before an LDS read, which left one
//    stage in flight instead of all.  The ring runs on across tiles: the next tile's first stages travel
//    through this tile's last stages and its epilogue.
//  * Up to rank 16 the epilogue's operands (z, B, the rows' scales and places, the columns' scales) are one more
//    stage of the ring behind the tile's last k step.  Loaded by the epilogue itself they waited for the
//    next tile's stages in front of them and then for each other.
//  * Every wave issues at least the same number of loads per stage whatever the tile's height (row blocks beyond it repeat
//    the last one's lines, which the L1 has), so the waits stay compile-time constants: with at most
//    (stages - 2) * loads outstanding, the stage wanted has landed, whatever stores are counted too.
//  * The weight's loads are non-temporal: 128 experts, 2048 x 1536, 16384 rows 108 -> 101 us, 128 rows 61 -> 58 us.
// Measured (gate/up with SwiGLU 2048 x 1536 / down 768 x 2048, 128 experts, rank 16), against tiles of 64 or 128 x 512
// dealt out over the tiles that there might be (which left two XCDs without any):
//   2048 tokens x 8: 138 -> 101 us (4.0 TB/s of weight) / 107 -> 71;  16 tokens x 8, 82 experts hit: 79 -> 58 (4.5 TB/s) / 55 -> 32.
#pragma once
#include "w8a8_gemm.h"

namespace w8a8 {

constexpr uint32_t kGroupedTileN = 256;
constexpr uint32_t kGroupedThreads = 512;
constexpr int grouped_stages(int rb) { return rb == 4 ? 6 : 4; }
constexpr int grouped_stage_bytes(int rb) { return (rb + 8) * 2 * kBlockBytes; }  // A: rb row blocks, B: 8 column blocks
// The epilogue's stage: z [rb][3][1 KiB], B [8][1 KiB], then sx [32 rb], src_row [32 rb], sw [256].  Of rb = 8 the last three
// do not fit it and lie behind the ring; a tile needs three k steps then, so that a barrier stands between
// one tile's epilogue and the next one's loads.
constexpr int grouped_lds_bytes(int rb) { return grouped_stages(rb) * grouped_stage_bytes(rb) + (rb == 8 ? 3 * kBlockBytes : 0); }
constexpr uint32_t kGroupedTallMinK = 256;

struct EpilogueFromLds {
  static constexpr bool kLaneAnew = true;  // 28 bytes of scratch -> none in the tall SwiGLU tile, 2048 x 1536, 128 rows a group 92.7 -> 89.2 us (another card 93.4 -> 91.4)
  const unsigned char* zs;  // z of the row block
  const unsigned char* bs;  // B of the wave's first column block
  const float* sxs;
  const int32_t* srcs;
  float s;
  __device__ float sx(int c) const { return sxs[c]; }
  __device__ int src_row(int c) const { return srcs[c]; }
  __device__ uint32_t range() const { return 0u; }  // one group
  __device__ int slot_group(int, int first) const { return first; }
  __device__ float scaling(int) const { return s; }
  template <int NKK>
  __device__ const unsigned char* z(int lane) const { return zs + lane * 16; }
  template <int NKK>
  __device__ const unsigned char* b(int, int j, int lane) const { return bs + j * kBlockBytes + lane * 16; }
};

template <int EPI, int NKK, int kRB>
__global__ __launch_bounds__(kGroupedThreads, 2) void w8a8_grouped_kernel(GemmArgs g) {
  static_assert(kRB == 4 || kRB == 8, "one or two row blocks per wave");
  constexpr int kWR = kRB / 4;                       // row blocks of a wave
  constexpr int kStages = grouped_stages(kRB);
  constexpr uint32_t kStageBytes = grouped_stage_bytes(kRB);
  constexpr uint32_t kRingBytes = kStages * kStageBytes;
  constexpr uint32_t kABytes = kRB * 2u * kBlockBytes;
  constexpr int kLoads = 2 + kRB / 4;                // direct-to-LDS loads per wave and stage (the epilogue's: that many or more)
  constexpr bool kStaged = NKK == 1 && EPI != kEpiAcc;  // the epilogue's operands travel through the ring
  constexpr uint32_t kZBytes = kRB * 3u * kBlockBytes;
  // places of the epilogue's scales and rows, from the start of its stage or, kRB = 8, of the LDS
  constexpr uint32_t kTail = kRB == 8 ? kRingBytes : kZBytes + 8u * kBlockBytes;

  extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // (waves w and w + 4 share a SIMD: wave rows 0 and 2, 1 and 3, so that a tile of few blocks spreads over all)
  const uint32_t wrow = wave >> 1, wcol = wave & 1u;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(lptr_t)lds;
  const uint32_t KT = g.K_pad / 64u;
  const uint32_t ncb_total = n_padded(g.N) / 32u;
  const uint32_t n_out = (EPI == kEpiSwiglu) ? g.N / 2u : g.N;

  // scalar loads: a vector load would wait for the stages in flight in front of it
  uint64_t row_tiles;
  asm volatile("s_load_dwordx2 %0, %1, 0x0\n\ts_waitcnt lgkmcnt(0)" : "=s"(row_tiles) : "s"(g.tile_tab) : "memory");
  const uint32_t ntile = (uint32_t)row_tiles * g.tiles_n;
  const uint32_t per_xcd = (ntile + 7u) / 8u, wgs_per_xcd = gridDim.x >> 3;
  const uint32_t t_begin = (blockIdx.x & 7u) * per_xcd;
  const uint32_t t_end = t_begin + per_xcd < ntile ? t_begin + per_xcd : ntile;

  struct Tile {
    const unsigned char* Ag;
    const unsigned char* Bg;
    uint32_t blk0, nblk, tn, grp, widx;
  };
  auto tile_at = [&](uint32_t t) -> Tile {
    Tile T;
    const uint32_t tm = t / g.tiles_n;
    T.tn = t - tm * g.tiles_n;
    uint64_t e;
    asm volatile("s_load_dwordx2 %0, %1, 0x0\n\ts_waitcnt lgkmcnt(0)" : "=s"(e) : "s"(g.tile_tab + 1u + tm) : "memory");
    T.blk0 = (uint32_t)e;
    T.nblk = (uint32_t)(e >> 32) & 0xffffu;
    T.grp = (uint32_t)(e >> 48);
    T.widx = T.grp / g.groups_per_weight;
    T.Ag = g.xq + (size_t)T.blk0 * g.KB * kBlockBytes;
    T.Bg = g.wp + (size_t)T.widx * g.w_group_stride + (size_t)(T.tn * 8u + wave) * g.KB * kBlockBytes;
    return T;
  };

  // ---- the loads' cursor: stages of this workgroup's tiles in order, kStages - 1 ahead of the MFMAs
  uint32_t ld_t = t_begin + (blockIdx.x >> 3), ld_kt = 0, ld_off = 0;
  bool ld_valid = ld_t < t_end;
  Tile L{};
  auto set_a_row = [&]() {  // the row block this wave fetches
    uint32_t rb = kRB == 8 ? wave : wave >> 1;
    rb = rb < L.nblk ? rb : L.nblk - 1u;
    L.Ag += (size_t)rb * g.KB * kBlockBytes + (kRB == 8 ? 0u : (wave & 1u) * kBlockBytes);
  };
  if (ld_valid) { L = tile_at(ld_t); set_a_row(); }
  const uint32_t ld_steps = KT + (kStaged ? 1u : 0u);
  auto issue_epilogue = [&]() {  // of the tile at the cursor
    const uint32_t es = lds0 + ld_off, tail = kRB == 8 ? lds0 + kTail : es + kTail;
    const uint32_t rb0 = kRB == 8 ? wave : wave >> 1;
    const uint32_t rb = rb0 < L.nblk ? rb0 : L.nblk - 1u;
    const unsigned char* zb = g.zp + (size_t)(L.blk0 + rb) * 3u * kBlockBytes;
    if (kRB == 8 || !(wave & 1u)) {
      lds_load_1k(zb, lane * 16u, es + rb0 * 3u * kBlockBytes);
      lds_load_1k(zb, lane * 16u + kBlockBytes, es + (rb0 * 3u + 1u) * kBlockBytes);
    }
    if (kRB == 8 || (wave & 1u)) lds_load_1k(zb, lane * 16u + 2u * kBlockBytes, es + (rb0 * 3u + 2u) * kBlockBytes);
    lds_load_1k(g.bp + ((size_t)L.grp * ncb_total + L.tn * 8u + wave) * kBlockBytes, lane * 16u, es + kZBytes + wave * kBlockBytes);
    // 64 rows or columns per gather; what lies behind the last slot or column repeats it and is not used
    constexpr uint32_t kRowGathers = kRB / 2;
    auto rows = [&](const void* tab, uint32_t piece, uint32_t dst) {
      const uint32_t p = L.blk0 * 32u + piece * 64u + lane;
      lds_gather_dword(tab, (p < g.slots ? p : g.slots - 1u) * 4u, dst + piece * 256u);
    };
    if (wave < kRowGathers) rows(g.sx, wave, tail);
    else if (wave < 2u * kRowGathers) rows(g.src_row, wave - kRowGathers, tail + kRB * 128u);
    if (wave >= 4u) {
      const uint32_t n = L.tn * kGroupedTileN + (wave - 4u) * 64u + lane;
      lds_gather_dword(g.sw + (size_t)L.widx * g.N, (n < g.N ? n : g.N - 1u) * 4u, tail + kRB * 256u + (wave - 4u) * 256u);
    }
  };
  auto issue = [&]() {
    if (!ld_valid) return;
    if (kStaged && ld_kt == KT) {
      issue_epilogue();
    } else {
      const uint32_t voff = ld_kt * 2u * kBlockBytes + lane * 16u;
      const uint32_t a_dst = lds0 + ld_off + (kRB == 8 ? wave * 2u : wave) * kBlockBytes;
      const uint32_t b_dst = lds0 + ld_off + kABytes + wave * 2u * kBlockBytes;
      lds_load_1k_once(L.Bg, voff, b_dst);
      lds_load_1k_once(L.Bg, voff + kBlockBytes, b_dst + kBlockBytes);
      lds_load_1k(L.Ag, voff, a_dst);
      if constexpr (kRB == 8) lds_load_1k(L.Ag, voff + kBlockBytes, a_dst + kBlockBytes);
    }
    ld_off = ld_off + kStageBytes == kRingBytes ? 0u : ld_off + kStageBytes;
    if (++ld_kt == ld_steps) {
      ld_kt = 0;
      ld_t += wgs_per_xcd;
      ld_valid = ld_t < t_end;
      if (ld_valid) { L = tile_at(ld_t); set_a_row(); }
    }
  };
#pragma unroll 1
  for (int st = 0; st < kStages - 1; ++st) issue();

  uint32_t rd_off = 0;  // the stage that is multiplied next
#pragma unroll 1
  for (uint32_t t = t_begin + (blockIdx.x >> 3); t < t_end; t += wgs_per_xcd) {
    const Tile T = tile_at(t);
    const uint32_t own = T.nblk > wrow ? (T.nblk - wrow + 3u) / 4u : 0u;  // row blocks of this wave in the tile
    v16i acc[kWR][4];
#pragma unroll
    for (int i = 0; i < kWR; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[i][j][e] = 0;
    // (One body whose second half stands under a condition: two bodies for one and two row blocks made the
    // allocator copy and spill the accumulators where they meet.)
    auto multiply = [&]() {
      const unsigned char* As = lds + rd_off + wrow * 2u * kBlockBytes + lane * 16u;
      const unsigned char* Bs = lds + rd_off + kABytes + wcol * 8u * kBlockBytes + lane * 16u;
      v4i bf[2][4];
      auto rows = [&](int i) {
        v4i af[2];
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) af[ks] = *reinterpret_cast<const v4i*>(As + (8u * i + ks) * kBlockBytes);
        if (i == 0) {
#pragma unroll
          for (int ks = 0; ks < 2; ++ks)
#pragma unroll
            for (int j = 0; j < 4; ++j) bf[ks][j] = *reinterpret_cast<const v4i*>(Bs + (2u * j + ks) * kBlockBytes);
        }
#pragma unroll
        for (int ks = 0; ks < 2; ++ks)
#pragma unroll
          for (int j = 0; j < 4; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(af[ks], bf[ks][j], acc[i][j], 0, 0, 0);
      };
      rows(0);
      if constexpr (kWR == 2) {
        if (own == 2u) rows(kWR - 1);
      }
    };
    auto next_stage = [&]() {
      if (ld_valid) wait_vmcnt<(kStages - 2) * kLoads>(); else wait_vmcnt<0>();  // (nothing follows the last issued stage)
      lds_barrier();  // it has landed for every wave, and all are done with the stage that the next loads replace
      issue();
    };
    auto passed = [&]() { rd_off = rd_off + kStageBytes == kRingBytes ? 0u : rd_off + kStageBytes; };
#pragma unroll 1
    for (uint32_t kt = 0; kt < KT; ++kt) {
      next_stage();
      if (own) multiply();
      passed();
    }

    // ---- epilogue
    const uint32_t es = rd_off;
    if constexpr (kStaged) {
      next_stage();
      passed();
    }
    const uint32_t tcol0 = T.tn * kGroupedTileN + wcol * 128u;
    if (own == 0u || tcol0 >= g.N) continue;  // (the wave still takes part in the next tile)
    const uint32_t ncol = tcol0 + 4u * (lane & 31u);
    const bool full_n = (tcol0 + 128u <= g.N) && ((g.N & 3u) == 0);  // wave-uniform
    float sw[4] = {0.f, 0.f, 0.f, 0.f};
    if constexpr (kStaged) {
      const unsigned char* tail = lds + (kRB == 8 ? kTail : es + kTail);
      float s;
      asm volatile("s_load_dword %0, %1, 0x0\n\ts_waitcnt lgkmcnt(0)" : "=s"(s) : "s"(g.lora_scaling + T.grp) : "memory");
      const float4 s4 = *reinterpret_cast<const float4*>(tail + kRB * 256u + wcol * 512u + (lane & 31u) * 16u);
      sw[0] = s4.x; sw[1] = s4.y; sw[2] = s4.z; sw[3] = s4.w;
      auto block = [&](int i) {
        const uint32_t rb = wrow + 4u * i;
        const EpilogueFromLds from{lds + es + rb * 3u * kBlockBytes, lds + es + kZBytes + wcol * 4u * kBlockBytes,
                                   reinterpret_cast<const float*>(tail) + rb * 32u,
                                   reinterpret_cast<const int32_t*>(tail + kRB * 128u) + rb * 32u, s};
        gemm_epilogue_block<EPI, NKK>(g, from, acc[i], sw, tcol0, full_n, n_out);
      };
      block(0);
      if constexpr (kWR == 2) {
        if (own == 2u) block(kWR - 1);
      }
    } else {
      const float* swp = g.sw + (size_t)T.widx * g.N;
      if (EPI != kEpiAcc) {
        if (full_n) {
          const float4 s4 = *reinterpret_cast<const float4*>(swp + ncol);
          sw[0] = s4.x; sw[1] = s4.y; sw[2] = s4.z; sw[3] = s4.w;
        } else {
#pragma unroll
          for (int j = 0; j < 4; ++j)
            if (ncol + j < g.N) sw[j] = swp[ncol + j];
        }
      }
      auto block = [&](int i) {
        const EpilogueFromMemory from{g, (T.blk0 + wrow + 4u * i) * 32u, tcol0, ncb_total};
        gemm_epilogue_block<EPI, NKK>(g, from, acc[i], sw, tcol0, full_n, n_out);
      };
      block(0);
      if constexpr (kWR == 2) {
        if (own == 2u) block(kWR - 1);
      }
    }
  }
}

}  // namespace w8a8
