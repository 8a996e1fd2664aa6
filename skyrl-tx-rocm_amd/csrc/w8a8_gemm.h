// Tiled int8 MFMA GEMM with the fused float32 epilogue:
//   acc[p, n]  = sum_k xq[p, k] * wq[k, n]                         (v_mfma_i32_32x32x32_i8, exact)
//   base       = (float(acc) * sx[p]) * sw[n]                      (skyrl/tx/kernels/quantized_lora.py:248-252)
//   y          = base + low * s[group(p)] (+ residual)             (quantized_lora.py:300-304)
//   low        = z[p, :] @ B[group(p)]                             (bf16 MFMA, z carried as 3 (or 2) bf16 terms)
//   out        = bf16(y)   or   bf16(silu(bf16(y_gate)) * bf16(y_up))
// Workgroup = 256 threads = 4 waves stacked along M (64 x 128 each), tile 256 x 128, 128
// accumulator registers per lane and 72 KiB of LDS, so two workgroups share a CU: while one is
// in its VALU/store epilogue the other keeps the MFMA pipe busy.  K is consumed in steps of 64
// through a ring of three 24 KiB LDS stages filled by 16-byte direct-to-LDS loads of contiguous
// 1 KiB fragment blocks, two tiles ahead of the MFMAs.
#pragma once
#include <type_traits>

#include "w8a8_device.h"

namespace w8a8 {

enum { kEpiPlain = 0, kEpiSwiglu = 1, kEpiAcc = 2 };

struct GemmArgs {
  const unsigned char* xq;   // packed activation codes [slots, K_pad]
  const unsigned char* wp;   // packed weight [N_pad, K_pad]
  const float* sx;           // f32 [slots]
  const float* sw;           // f32 [N]
  const unsigned char* zp;   // packed z fragments [slots/32][NKK][3][64 lanes][8 bf16] or null
  const float* lora_scaling; // f32 [n_groups]
  const unsigned char* bp;   // LoRA B in MFMA operand order [n_groups][N_pad/32][NKK][64 lanes][8 bf16] or null
  const int32_t* src_row;    // original row of every grouped slot, or null (identity)
  const int32_t* slot_group; // LoRA group (adapter) of every grouped slot, or null (group 0)
  const int32_t* blk_range;  // per 32-row block: first group | last group << 16, or null
  const uint16_t* residual;  // bf16 [M, n_out] or null
  void* out;                 // bf16 [M, n_out] or int32 [M, N]
  uint64_t w_group_stride;   // grouped call: bytes between the packed weights of two experts
  uint32_t M, N, K_pad, KB, slots, total_rows;
  uint32_t tiles_m, tiles_n, rank;
  uint32_t groups_per_weight; // grouped call: weight index = group / groups_per_weight
  const uint64_t* tile_tab;   // grouped call: number of row tiles, then first 32-slot block | blocks << 32 | group << 48 of each
  uint32_t* tile_ctr;         // 8 zeroed counters, 64 bytes apart (one per XCD), or null: static schedule
};

// silu(g) * u with g, u already rounded to bf16 (x * logistic(x), exp and reciprocal in
// hardware precision: 1 ulp each)
__device__ inline float swiglu_f32(float g, float u) {
  const float sig = __builtin_amdgcn_rcpf(1.0f + __expf(-g));
  return (g * sig) * u;
}

constexpr int kGemmTileM = 256;
constexpr int kGemmTileN = 128;
constexpr int kGemmStages = 3;
constexpr int kGemmStageBytes = 24576;  // A: 8 row blocks x 2 k blocks, B: 4 column blocks x 2 k blocks
constexpr int kGemmLdsBytes = kGemmStages * kGemmStageBytes;
// (The 256 x 256 geometry for large problems is a kernel of its own: w8a8_gemm16.h.)
// Dense geometry for calls whose 256 x 128 tiles would leave most CUs idle: 128 x 128 tiles, the four
// waves stacked along M with 32 x 128 each, so a wave carries half the MFMAs and half the epilogue.
constexpr int kGemm128TileM = 128;
constexpr int kGemm128StageBytes = 16384;  // A: 4 row blocks x 2 k blocks, B: 4 column blocks x 2 k blocks
enum { kModeDense = 0, kModeDense128 = 1 };

// Where the epilogue of one 32-row block finds its operands: in memory.  (The grouped kernel has a form that finds them in the LDS.)
struct EpilogueFromMemory {
  // (Formed anew, the grouped kernel's registers fell so that a load of the epilogue shares one with an operand of the k
  // loop, which then drains its ring at every step: rank 32, 128 rows a group 97 -> 122 us.)
  static constexpr bool kLaneAnew = false;
  const GemmArgs& g;
  uint32_t pbase, tcol0, ncb_total;
  __device__ float sx(int c) const { return g.sx[pbase + c]; }
  __device__ int src_row(int c) const { return g.src_row ? g.src_row[pbase + c] : (int)(pbase + c); }
  __device__ uint32_t range() const { return g.blk_range ? (uint32_t)g.blk_range[pbase / 32u] : 0u; }
  __device__ int slot_group(int c, int first) const { return g.slot_group ? g.slot_group[pbase + c] : first; }
  __device__ float scaling(int gi) const { return g.lora_scaling[gi]; }
  // (Bases from which the operands lie at constant distances: an address of its own for each took registers that
  // the accumulators need.)  z: operand (kk, term) at kk * 3 + term blocks
  template <int NKK>
  __device__ const unsigned char* z(int lane) const { return g.zp + (size_t)(pbase / 32u) * NKK * 3u * kBlockBytes + lane * 16; }
  // of the wave's packed column block j, operand kk (rows 16 kk + 8 h + 0..7 of column 4 c + j) at kk blocks, block j + 1 at NKK
  template <int NKK>
  __device__ const unsigned char* b(int gi, int j, int lane) const {
    return g.bp + ((size_t)gi * ncb_total + tcol0 / 32u + j) * NKK * kBlockBytes + lane * 16;
  }
};

// Epilogue of one 32-row block of a wave's 128 columns from tcol0 on: accumulators acc[j] of the packed column
// blocks j.  Lane (c = lane % 32, h = lane / 32) owns the four consecutive original columns ncol .. ncol + 3
// (ncol = tcol0 + 4 c) of the 16 rows 8*(v/4) + 4*h + v%4; sw holds their scales.
template <int EPI, int NKK, class Source>
__device__ inline __attribute__((always_inline)) void gemm_epilogue_block(const GemmArgs& g, const Source& from, const v16i (&acc)[4],
                                                                          const float (&sw)[4], uint32_t tcol0, bool full_n,
                                                                          uint32_t n_out) {
  constexpr bool kLora = (NKK > 0) && (EPI != kEpiAcc);
  int lane = threadIdx.x & 63;
  // (opaque: what the epilogue derives from it is formed here and not held, or spilled, through the k loop)
  if constexpr (Source::kLaneAnew) asm volatile("" : "+v"(lane));
  const int c = lane & 31, h = lane >> 5;
  const uint32_t ncol = tcol0 + 4u * c;
  __builtin_amdgcn_sched_barrier(0);  // keep the blocks' register lifetimes apart

  // Per-row scale and output offset of the block's 32 rows live in one register each (lane l
  // holds row l % 32); a lane's 16 rows 8*(v/4) + 4*h + v%4 are fetched across lanes below.
  const float sx_lane = (EPI != kEpiAcc) ? from.sx(c) : 0.0f;
  const int src_lane = from.src_row(c);
  const bool row_ok = src_lane >= 0 && src_lane < (int)g.M;
  const uint32_t off_lane = row_ok ? (uint32_t)src_lane * ((EPI == kEpiAcc) ? g.N : n_out) : 0xffffffffu;
  const bool fast = full_n && (__builtin_amdgcn_ballot_w64(!row_ok) == 0);  // wave-uniform
  const int row_addr = 16 * h;  // byte address (4 * lane) of the lane holding row 4*h

  if (EPI == kEpiAcc) {
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const uint32_t rowoff =
          (uint32_t)__builtin_amdgcn_ds_bpermute(row_addr + 4 * (8 * (v >> 2) + (v & 3)), (int)off_lane);
      if (!fast && rowoff == 0xffffffffu) continue;
      int32_t* o = reinterpret_cast<int32_t*>(g.out) + rowoff + ncol;
      if (fast) {
        *reinterpret_cast<int4*>(o) = make_int4(acc[0][v], acc[1][v], acc[2][v], acc[3][v]);
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (ncol + j < g.N) o[j] = acc[j][v];
      }
    }
    return;
  }

  // Groups (adapters) present in this 32-row block: one, except at a group boundary.  A
  // boundary block is simply processed once per group; each pass stores only its own rows.
  const uint32_t range = kLora ? from.range() : 0u;
  const int glo = (int)(range & 0xffffu), ghi = (int)(range >> 16);
  const int grp_lane = (kLora && ghi > glo) ? from.slot_group(c, glo) : glo;
  for (int gi = glo; gi <= ghi; ++gi) {  // wave-uniform
  // The lane's four columns are processed as two pairs (jp): LoRA MFMAs of the pair (section A),
  // then dequantize + add + activate per row (section B).  The first pair's packed result waits
  // in `hold` so that every row is written with one 4- or 8-byte store.
  uint32_t hold[16];
#pragma unroll
  for (int jp = 0; jp < 2; ++jp) {
    // ---- section A: lowS[j][v] = s_g * (z @ B_g) for the column pair
    v16f lowS[2];
    if constexpr (kLora) {
      const unsigned char* const zb = from.template z<NKK>(lane);
      const unsigned char* const bb0 = from.template b<NKK>(gi, 2 * jp, lane);
#pragma unroll
      for (int kk = 0; kk < NKK; ++kk) {
        v8us zf[3];
#pragma unroll
        for (int t3 = 0; t3 < 3; ++t3) zf[t3] = *reinterpret_cast<const v8us*>(zb + (kk * 3 + t3) * kBlockBytes);
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const v8bf bb = __builtin_bit_cast(v8bf, *reinterpret_cast<const v8us*>(bb0 + (j * NKK + kk) * kBlockBytes));
          v16f cur;
          if (kk == 0) {
#pragma unroll
            for (int e = 0; e < 16; ++e) cur[e] = 0.0f;
          } else {
            cur = lowS[j];
          }
          cur = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8bf, zf[2]), bb, cur, 0, 0, 0);
          cur = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8bf, zf[1]), bb, cur, 0, 0, 0);
          cur = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8bf, zf[0]), bb, cur, 0, 0, 0);
          lowS[j] = cur;
        }
      }
      const float sgrp = from.scaling(gi);
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) lowS[j][e] = lowS[j][e] * sgrp;
    }

    // ---- section B
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      // row 8*(v/4) + 4*h + v%4 of the block: its data sits in that lane (cross-lane read on
      // the LDS crossbar, which is idle here; no vector-ALU work)
      const int src_lane_addr = row_addr + 4 * (8 * (v >> 2) + (v & 3));
      const uint32_t rowoff = (uint32_t)__builtin_amdgcn_ds_bpermute(src_lane_addr, (int)off_lane);
      const float sxv =
          __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute(src_lane_addr, __builtin_bit_cast(int, sx_lane)));
      const float t0 = (float)acc[2 * jp][v] * sxv;
      const float t1 = (float)acc[2 * jp + 1][v] * sxv;
      // same f32 operations, in the same order, as the reference epilogue: a fused
      // multiply-add here would flip rare bf16 roundings that SwiGLU then amplifies
      float y0 = t0 * sw[2 * jp];
      float y1 = t1 * sw[2 * jp + 1];
      if constexpr (kLora) {
        y0 = y0 + lowS[0][v];
        y1 = y1 + lowS[1][v];
      }
      bool row_valid = fast || rowoff != 0xffffffffu;
      if (kLora && ghi > glo)  // boundary block: this pass owns only the rows of group gi
        row_valid = row_valid && (__builtin_amdgcn_ds_bpermute(src_lane_addr, grp_lane) == gi);
      uint32_t mine_bits;
      if (EPI == kEpiSwiglu) {
        // (y0, y1) = (gate, up) of the product column ncol/2 + jp
        const uint32_t f = pack_bf16x2(y0, y1);
        mine_bits = __float_as_uint(swiglu_f32(__uint_as_float(f << 16), __uint_as_float(f & 0xffff0000u)));
      } else {
        if (g.residual && row_valid) {
          uint32_t rr;
          if (fast) {
            rr = *reinterpret_cast<const uint32_t*>(g.residual + rowoff + ncol + 2u * jp);
          } else {
            rr = 0;
            if (ncol + 2u * jp < g.N) rr |= (uint32_t)g.residual[rowoff + ncol + 2u * jp];
            if (ncol + 2u * jp + 1u < g.N) rr |= (uint32_t)g.residual[rowoff + ncol + 2u * jp + 1u] << 16;
          }
          y0 = y0 + __uint_as_float(rr << 16);
          y1 = y1 + __uint_as_float(rr & 0xffff0000u);
        }
        mine_bits = pack_bf16x2(y0, y1);
      }
      if (jp == 0) {
        hold[v] = mine_bits;
        continue;
      }
      if (!row_valid) continue;
      if (EPI == kEpiSwiglu) {
        const uint32_t pk = pack_bf16x2(__uint_as_float(hold[v]), __uint_as_float(mine_bits));
        uint16_t* o = reinterpret_cast<uint16_t*>(g.out) + rowoff + (ncol >> 1);
        if (fast) {
          *reinterpret_cast<uint32_t*>(o) = pk;
        } else {
          if ((ncol >> 1) < n_out) o[0] = (uint16_t)(pk & 0xffffu);
          if ((ncol >> 1) + 1u < n_out) o[1] = (uint16_t)(pk >> 16);
        }
      } else {
        uint16_t* o = reinterpret_cast<uint16_t*>(g.out) + rowoff + ncol;
        if (fast) {
          *reinterpret_cast<uint2*>(o) = make_uint2(hold[v], mine_bits);
        } else {
          if (ncol + 0u < g.N) o[0] = (uint16_t)(hold[v] & 0xffffu);
          if (ncol + 1u < g.N) o[1] = (uint16_t)(hold[v] >> 16);
          if (ncol + 2u < g.N) o[2] = (uint16_t)(mine_bits & 0xffffu);
          if (ncol + 3u < g.N) o[3] = (uint16_t)(mine_bits >> 16);
        }
      }
    }
  }
  }  // groups of the block
}

// One tile of the persistent loop.
struct GemmTile {
  const unsigned char* Ag;  // packed activation panel of the tile
  const unsigned char* Bg;  // packed weight of the tile's group
  const float* swp;         // per-channel scales of the tile's group
  uint32_t tm, tn;
  bool valid;
};

template <int EPI, int NKK, int MODE = kModeDense>
__global__ __launch_bounds__(256, 2)
void w8a8_gemm_kernel(GemmArgs g) {
  constexpr bool D128 = MODE == kModeDense128;
  constexpr int kWaves = 4;
  constexpr int kWR = D128 ? 1 : 2;                                  // 32-row blocks of a wave's tile
  constexpr uint32_t kRowBlocks = D128 ? 4 : 8;                     // 32-row blocks of the activation panel
  constexpr uint32_t kColBlocks = 4;                                // 32-column blocks of the weight panel
  constexpr int kStages = kGemmStages;
  constexpr int kStageBytes = D128 ? kGemm128StageBytes : kGemmStageBytes;
  constexpr int kAChunks = kRowBlocks * 2;                              // 1 KiB chunks of A per stage
  constexpr int kLoadsPerTile = (kAChunks + kColBlocks * 2) / kWaves;   // direct-to-LDS loads per wave per k-tile

  extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wrow = wave;  // wave position along M (32 * kWR rows each)
  const int c = lane & 31;

  const uint32_t total_rows = g.total_rows;
  const uint32_t ntile = g.tiles_m * g.tiles_n;
  const uint32_t ncb_total = n_padded(g.N) / 32u;  // column blocks of the packed weight
  const uint32_t n_out = (EPI == kEpiSwiglu) ? g.N / 2u : g.N;
  const int KT = (int)(g.K_pad / 64u);

  // ---- persistent tile schedule.  Consecutive workgroup ids land on different XCDs, so each XCD
  // walks a contiguous range of a band-major tile order (GM row tiles x all column tiles) and the
  // workgroups of an XCD work on neighbouring tiles at any time (shared panels hit in its L2).
  const uint32_t per_xcd = (ntile + 7u) / 8u;
  const uint32_t wgs_per_xcd = gridDim.x >> 3;
  // `i` is a position inside the XCD's range of the tile order.
  auto tile_at = [&](uint32_t i) -> GemmTile {
    GemmTile T{};
    const uint32_t t = i < per_xcd ? (blockIdx.x & 7u) * per_xcd + i : ntile;
    if (t >= ntile) return T;
    constexpr uint32_t GM = 4;
    const uint32_t band = t / (GM * g.tiles_n);
    const uint32_t band_rows = (g.tiles_m - band * GM) < GM ? (g.tiles_m - band * GM) : GM;
    const uint32_t in_band = t - band * GM * g.tiles_n;
    T.tm = band * GM + in_band % band_rows;
    T.tn = in_band / band_rows;
    T.Ag = g.xq + (size_t)T.tm * kRowBlocks * g.KB * kBlockBytes;
    T.Bg = g.wp;
    T.swp = g.sw;
    T.valid = true;
    return T;
  };
  // Static schedule: position (workgroup index inside the XCD) + step * (workgroups per XCD).
  // Dynamic schedule (two workgroups per CU): positions come from the XCD's counter, because the
  // hardware favours the older workgroup of a CU and a static split would leave the younger one
  // to finish alone.  The result does not depend on which workgroup computes which tile.
  const bool dyn = g.tile_ctr != nullptr;
  uint32_t* const ctr = g.tile_ctr + (blockIdx.x & 7u) * 16u;
  __shared__ uint32_t dyn_slot[2];
  uint32_t cur_i = blockIdx.x >> 3, nxt_i = 0;
  if (dyn) {
    if (tid == 0) dyn_slot[0] = atomicAdd(ctr, 1u);
    __syncthreads();
    cur_i = dyn_slot[0];
  }

  auto issue = [&](const GemmTile& T, int kt) {
    unsigned char* St = lds + (kt % kStages) * kStageBytes;
#pragma unroll
    for (int q = 0; q < kLoadsPerTile; ++q) {
      const int ch = wave * kLoadsPerTile + q;  // chunks < kAChunks: A (row block ch/2, k block ch%2); then B
      const bool isA = ch < kAChunks;
      uint32_t rb = isA ? (uint32_t)(ch >> 1) : T.tn * kColBlocks + (uint32_t)((ch - kAChunks) >> 1);
      if (!isA && rb >= ncb_total) rb = ncb_total - 1u;  // keep every wave's load count equal
      const unsigned char* base = isA ? T.Ag : T.Bg;
      const size_t goff = ((size_t)rb * g.KB + (size_t)kt * 2 + (ch & 1)) * kBlockBytes + lane * 16;
      load_1k_to_lds(base + goff, St + ch * kBlockBytes);
    }
  };
  auto read_frags = [&](int kt, int ks, v4i (&af)[kWR], v4i (&bf)[4]) {
    const unsigned char* As = lds + (kt % kStages) * kStageBytes;
    const unsigned char* Bs = As + kAChunks * kBlockBytes;
#pragma unroll
    for (int i = 0; i < kWR; ++i)
      af[i] = *reinterpret_cast<const v4i*>(As + ((wrow * kWR + i) * 2 + ks) * kBlockBytes + lane * 16);
#pragma unroll
    for (int j = 0; j < 4; ++j)
      bf[j] = *reinterpret_cast<const v4i*>(Bs + (j * 2 + ks) * kBlockBytes + lane * 16);
  };

  bool prefetched = false;  // the first kStages-1 k-tiles of the current tile are already in flight
  for (uint32_t step = 0; cur_i < per_xcd; ++step, cur_i = nxt_i) {
    const GemmTile T = tile_at(cur_i);
    nxt_i = cur_i + wgs_per_xcd;
    if (!T.valid) { prefetched = false; continue; }  // static schedules only (range end)

    v16i acc[kWR][4];
#pragma unroll
    for (int i = 0; i < kWR; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[i][j][e] = 0;
    auto mfma8 = [&](const v4i (&af)[kWR], const v4i (&bf)[4]) {
#pragma unroll
      for (int i = 0; i < kWR; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(af[i], bf[j], acc[i][j], 0, 0, 0);
    };

    // ---- main loop
    v4i fa0[kWR], fb0[4], fa1[kWR], fb1[4];
    if (!prefetched) {
#pragma unroll
      for (int st = 0; st < kStages - 1; ++st)
        if (st < KT) issue(T, st);
      if (KT > kStages - 2) wait_vmcnt<(kStages - 2) * kLoadsPerTile>(); else wait_vmcnt<0>();
    } else {
      wait_vmcnt<0>();  // prefetch of this tile and the previous tile's stores
    }
    lds_barrier();
    uint32_t grabbed = 0;  // next position of a dynamic schedule; it arrives during the main loop
    if (dyn && tid == 0) grabbed = atomicAdd(ctr, 1u);
    read_frags(0, 0, fa0, fb0);
    const int KT_main = KT - (kStages - 1);  // k-tiles that still have a k-tile to prefetch
    int kt = 0;
    for (; kt < KT_main; ++kt) {
      // ---- k-step 0 of k-tile kt: prefetch the k-step 1 fragments and the k-tile kStages-1 ahead.
      // The MFMAs lead so that the wait for their operands does not cover the new LDS reads.
      read_frags(kt, 1, fa1, fb1);
      issue(T, kt + kStages - 1);
      mfma8(fa0, fb0);
      if constexpr (kWR == 2) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // 1 MFMA
#pragma unroll
        for (int q = 0; q < 6; ++q) {
          __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // 1 DS read
          __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);  // 1 VMEM read
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // 1 MFMA
        }
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      } else {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        }
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
      // ---- k-step 1: k-tile kt+1 must have landed before its first fragments are fetched
      wait_vmcnt<(kStages - 2) * kLoadsPerTile>();
      lds_barrier();
      __builtin_amdgcn_sched_barrier(0);
      read_frags(kt + 1, 0, fa0, fb0);
      mfma8(fa1, fb1);
      if constexpr (kWR == 2) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
#pragma unroll
        for (int q = 0; q < 6; ++q) {
          __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        }
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      } else {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        }
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    for (; kt < KT; ++kt) {  // drain: nothing left to prefetch
      read_frags(kt, 1, fa1, fb1);
      mfma8(fa0, fb0);
      wait_vmcnt<0>();
      lds_barrier();
      if (kt + 1 < KT) read_frags(kt + 1, 0, fa0, fb0);
      mfma8(fa1, fb1);
    }
    if (dyn && tid == 0) dyn_slot[(step + 1u) & 1u] = grabbed;  // the drain loop has waited for it
    lds_barrier();  // every wave is done with the stage buffers
    if (dyn) nxt_i = dyn_slot[(step + 1u) & 1u];

    // ---- the next tile's first k-tiles travel while this tile's epilogue runs (no LDS below)
    prefetched = false;
    if (nxt_i < per_xcd) {
      const GemmTile Tn = tile_at(nxt_i);
      if (Tn.valid) {
#pragma unroll
        for (int st = 0; st < kStages - 1; ++st)
          if (st < KT) issue(Tn, st);
        prefetched = true;
      }
    }

    // ---------------------------------------------------------------- epilogue
    const uint32_t m0 = T.tm * (kRowBlocks * 32u) + wrow * (32u * kWR);
    const uint32_t tcol0 = T.tn * (kColBlocks * 32u);  // first column of the wave
    const uint32_t ncol = tcol0 + 4u * c;
    const bool full_n = (tcol0 + 128u <= g.N) && ((g.N & 3u) == 0);  // wave-uniform
    if (tcol0 >= g.N) continue;  // wave beyond the last column; it still takes part in the next tile
    float sw[4] = {0.f, 0.f, 0.f, 0.f};
    if (EPI != kEpiAcc) {
      if (full_n) {
        const float4 s4 = *reinterpret_cast<const float4*>(T.swp + ncol);
        sw[0] = s4.x; sw[1] = s4.y; sw[2] = s4.z; sw[3] = s4.w;
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (ncol + j < g.N) sw[j] = T.swp[ncol + j];
      }
    }
    const auto epilogue_block = [&](int bi) {
      const uint32_t pbase = m0 + bi * 32u;
      if (pbase >= total_rows) return;  // wave-uniform
      gemm_epilogue_block<EPI, NKK>(g, EpilogueFromMemory{g, pbase, tcol0, ncb_total}, acc[bi], sw, tcol0, full_n, n_out);
    };
    epilogue_block(0);
    if constexpr (kWR == 2) epilogue_block(1);
  }
}

// ---------------------------------------------------------------------------------------
// The same product for calls of few rows: 64 x 128 tiles, the four waves of a workgroup taking every fourth 32-wide k block
// of the whole tile.  No two waves read the same bytes, so the operands go from the caches into registers (kRing k blocks
// ahead) without the LDS and without barriers, which then adds the waves' integer sums: exact, so the result is
// the 128 x 128 geometry's bit for bit.  Behind it wave (i, jp) owns row block i and columns 4 c + 2 jp, + 1: a quarter of the
// tile's epilogue each, whose operands have been on their way since the kernel's start.
// PAIR: two workgroups to a CU, for up to twice the tiles: half the registers, so a shorter ring, the epilogue's operands
// fetched behind the main loop, and the sums exchanged a column block at a time.
// Bound by what a CU takes from the caches (24 KiB for 128 of K, 64 bytes a clock: 5 us at K = 4096 for one workgroup) and by the
// latencies before and behind that.  333 x 4096 -> 2560, rank 64: 30 us on 80 tiles of 128 x 128, whose ring of LDS stages takes
// 12 us at the LDS's rate, now 17; 333 x 12288 -> 4096 64 / 38; 700 x 4096 -> 2560 (480 tiles, PAIR) 32 / 31.
// ---------------------------------------------------------------------------------------
constexpr int kGemm64TileM = 64;
constexpr int kGemm64LdsBytes = 4 * 3 * 8192;  // to each wave from the three others: 2 column blocks x 16 registers (PAIR: one)

// What this kernel alone is handed stands behind the arguments of all.  (Amid them it moved what every GEMM kernel reads, whose scalar
// loads then fell apart: the 128 x 128 geometry took 1 to 2 % longer.)
struct GemmKSplitArgs : GemmArgs {
  const float* zpart;  // f32 [4][z_slots][16 NKK] whose sum is z, instead of zp, or null
  uint32_t z_slots;
  uint32_t nterms;     // bf16 terms that z is split into (3 or 2)
};

// CHUNKS: the call stands in for 32-row chunks (sums_again).
template <int EPI, int NKK, bool PAIR, bool CHUNKS>
__global__ __launch_bounds__(256, PAIR ? 2 : 1) void w8a8_gemm_ksplit_kernel(GemmKSplitArgs g) {
  static_assert(EPI != kEpiAcc, "accumulators are read off the other geometries");
  constexpr int kRing = PAIR ? 3 : 6;
  constexpr int kParts = PAIR ? 2 : 1;  // passes of the sums' exchange
  constexpr int kKK = NKK > 0 ? NKK : 1;
  extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];
  const int lane = threadIdx.x & 63, c = lane & 31, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wr = wave & 1, jp = wave >> 1;
  // an XCD's workgroups take the row tiles of neighbouring column tiles: the weight is fetched into one L2
  const uint32_t ntile = g.tiles_m * g.tiles_n, per_xcd = (ntile + 7u) / 8u;
  const uint32_t t = (blockIdx.x & 7u) * per_xcd + (blockIdx.x >> 3);
  if ((blockIdx.x >> 3) >= per_xcd || t >= ntile) return;
  const uint32_t tn = t / g.tiles_m, tm = t - tn * g.tiles_m;
  const uint32_t tcol0 = tn * 128u, n_out = (EPI == kEpiSwiglu) ? g.N / 2u : g.N;
  if (tcol0 >= g.N) return;  // workgroup-uniform
  const uint32_t lane16 = (uint32_t)lane * 16u;

  // ---- what the epilogue needs of this wave's row block and columns
  const uint32_t pbase = tm * 64u + (uint32_t)wr * 32u;
  const bool has_rows = pbase < g.total_rows;  // (the tile's second block may lie behind the slots that can hold rows)
  const uint32_t pblk = has_rows ? pbase : tm * 64u;
  const float sx_lane = g.sx[pblk + c];
  const int src_lane = g.src_row ? g.src_row[pblk + c] : (int)(pblk + c);
  const uint32_t range = (NKK > 0 && g.blk_range) ? (uint32_t)g.blk_range[pblk / 32u] : 0u;
  const int glo = (int)(range & 0xffffu), ghi = (int)(range >> 16);
  const int grp_lane = (NKK > 0 && ghi > glo && g.slot_group) ? g.slot_group[pblk + c] : glo;
  const uint32_t ncol = tcol0 + 4u * c + 2u * jp;  // the lane's two columns
  const bool full_n = tcol0 + 128u <= g.N && (g.N & 3u) == 0;  // workgroup-uniform
  float sw[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) sw[j] = g.sw[ncol + j < g.N ? ncol + j : g.N - 1u];
  const uint32_t ncb_total = n_padded(g.N) / 32u;
  // LoRA operands of chunk kk: B of group gi for the two column blocks, z as bf16 terms (of the packed form, or its quarters
  // added in order and split as quant_lora_store_z does)
  auto fetch_b = [&](int gi, int kk, v8us (&b)[2]) {
    const unsigned char* bb = g.bp + (((size_t)gi * ncb_total + tcol0 / 32u + 2u * jp) * kKK + kk) * kBlockBytes + lane16;
#pragma unroll
    for (int j = 0; j < 2; ++j) b[j] = *reinterpret_cast<const v8us*>(bb + j * (kKK * kBlockBytes));
  };
  auto fetch_z = [&](int kk, v8us (&zt)[3]) {
    const unsigned char* zb = g.zp + ((size_t)(pblk / 32u) * kKK + kk) * 3u * kBlockBytes + lane16;
#pragma unroll
    for (int t3 = 0; t3 < 3; ++t3) zt[t3] = *reinterpret_cast<const v8us*>(zb + t3 * kBlockBytes);
  };
  auto z_from_quarters = [&](int kk, v8us (&zt)[3]) {
    const float* zq = g.zpart + (size_t)(pblk + c) * (16u * kKK) + 16 * kk + 8u * h;
    const size_t quarter = (size_t)g.z_slots * (16u * kKK);
    v4f q4[4][2];
#pragma unroll
    for (int p = 0; p < 4; ++p)
#pragma unroll
      for (int e = 0; e < 2; ++e) q4[p][e] = *reinterpret_cast<const v4f*>(zq + p * quarter + 4 * e);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float z = ((q4[0][e >> 2][e & 3] + q4[1][e >> 2][e & 3]) + q4[2][e >> 2][e & 3]) + q4[3][e >> 2][e & 3];
      const uint32_t b0 = f32_to_bf16_bits(z);
      const float r1 = z - bf16_bits_to_f32(b0);
      const uint32_t b1 = f32_to_bf16_bits(r1);
      const float r2 = r1 - bf16_bits_to_f32(b1);
      zt[0][e] = (unsigned short)b0;
      zt[1][e] = (unsigned short)b1;
      zt[2][e] = (unsigned short)(g.nterms >= 3u ? f32_to_bf16_bits(r2) : 0u);
    }
  };
  // The low-rank sums of a call in the place of chunks where they are not finite: an infinite z has one term (the rest is inf - inf), and an
  // infinite B meets z's first term alone (terms of both signs would cancel to NaN).  z @ B is then infinite where it is in float32, as
  // in the chunks.  (In every call the look at the sums would cost 0.1 us a pass: 0.6 % over 440 calls, 5 % with 48 adapters among few rows.  An instance
  // of its own: compiled into all it cost them 0.2 %.)
  auto sums_again = [&](int gi, v16f (&low)[2]) {
    auto odd = [](unsigned short v) { return (v & 0x7f80u) == 0x7f80u; };
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) low[j][e] = 0.0f;
#pragma unroll 1
    for (int kk = 0; kk < kKK; ++kk) {
      v8us z[3], b[2];
      fetch_b(gi, kk, b);
      if (g.zpart) z_from_quarters(kk, z);
      else fetch_z(kk, z);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        z[1][e] = odd(z[0][e]) ? (unsigned short)0 : z[1][e];
        z[2][e] = odd(z[0][e]) ? (unsigned short)0 : z[2][e];
      }
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        v8us fin = b[j];
#pragma unroll
        for (int e = 0; e < 8; ++e) fin[e] = odd(fin[e]) ? (unsigned short)0 : fin[e];
#pragma unroll
        for (int t3 = 2; t3 >= 0; --t3)
          low[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8bf, z[t3]), __builtin_bit_cast(v8bf, t3 ? fin : b[j]),
                                                           low[j], 0, 0, 0);
      }
    }
  };
  v8us zf[kKK][3], bf[kKK][2];  // (!PAIR: held from here on)
  if constexpr (NKK > 0 && !PAIR) {
#pragma unroll
    for (int kk = 0; kk < kKK; ++kk) {
      fetch_b(glo, kk, bf[kk]);
      if (!g.zpart) fetch_z(kk, zf[kk]);  // kernel-uniform
    }
  }

  // ---- main loop: stage s is k block 4 s + wave of the tile's two row blocks and four column blocks
  const int n_stages = (int)(g.KB / 4u);  // (K_pad is a multiple of 128)
  const size_t rb_bytes = (size_t)g.KB * kBlockBytes;
  const unsigned char* const Ag = g.xq + (size_t)tm * 2u * rb_bytes + (size_t)wave * kBlockBytes;
  const unsigned char* const Bg = g.wp + (size_t)tn * 4u * rb_bytes + (size_t)wave * kBlockBytes;
  v4i af[kRing][2], wf[kRing][4];
  auto fetch = [&](int u, int s) {
    const size_t off = (size_t)(s < n_stages ? s : n_stages - 1) * (4u * kBlockBytes);
#pragma unroll
    for (int i = 0; i < 2; ++i) af[u][i] = *reinterpret_cast<const v4i*>(Ag + i * rb_bytes + off + lane16);
#pragma unroll
    for (int j = 0; j < 4; ++j) wf[u][j] = *reinterpret_cast<const v4i*>(Bg + j * rb_bytes + off + lane16);
  };
  v16i acc[2][4];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0;
#pragma unroll
  for (int u = 0; u < kRing; ++u) {
    fetch(u, u);
    __builtin_amdgcn_sched_barrier(0);
  }
  auto mul = [&](int u) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(af[u][i], wf[u][j], acc[i][j], 0, 0, 0);
  };
  int s0 = 0;
#pragma unroll 1
  for (; s0 + kRing <= n_stages; s0 += kRing) {
#pragma unroll
    for (int u = 0; u < kRing; ++u) {
      mul(u);
      fetch(u, s0 + u + kRing);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
#pragma unroll
  for (int u = 0; u < kRing - 1; ++u)
    if (s0 + u < n_stages) mul(u);  // wave-uniform

  // ---- the waves' sums: to wave d its row block and column pair from the three others
  v16i own[2];
#pragma unroll
  for (int part = 0; part < kParts; ++part) {
    constexpr int kBlocks = 2 / kParts;  // column blocks of a pass
    if (part) __syncthreads();  // (those of the pass before are read)
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      if (wave == d) {
#pragma unroll
        for (int j = 0; j < kBlocks; ++j) own[part + j] = acc[d & 1][2 * (d >> 1) + part + j];
      } else {
        v4i* dst = reinterpret_cast<v4i*>(lds + (d * 3 + (wave < d ? wave : wave - 1)) * (4096 * kBlocks)) + lane;
#pragma unroll
        for (int j = 0; j < kBlocks; ++j)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const v16i& a = acc[d & 1][2 * (d >> 1) + part + j];
            dst[(j * 4 + e) * 64] = v4i{a[4 * e], a[4 * e + 1], a[4 * e + 2], a[4 * e + 3]};
          }
      }
    }
    __syncthreads();
#pragma unroll
    for (int s = 0; s < 3; ++s) {
      const v4i* src = reinterpret_cast<const v4i*>(lds + (wave * 3 + s) * (4096 * kBlocks)) + lane;
#pragma unroll
      for (int j = 0; j < kBlocks; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const v4i v = src[(j * 4 + e) * 64];
#pragma unroll
          for (int q = 0; q < 4; ++q) own[part + j][4 * e + q] += v[q];
        }
    }
  }
  if (!has_rows) return;  // wave-uniform

  if constexpr (NKK > 0 && !PAIR) {
    if (g.zpart) {
#pragma unroll
      for (int kk = 0; kk < kKK; ++kk) z_from_quarters(kk, zf[kk]);
    }
  }
  // ---- epilogue: gemm_epilogue_block's arithmetic on one column pair
  const bool row_ok = src_lane >= 0 && src_lane < (int)g.M;
  const uint32_t off_lane = row_ok ? (uint32_t)src_lane * n_out : 0xffffffffu;
  const bool fast = full_n && __builtin_amdgcn_ballot_w64(!row_ok) == 0;  // wave-uniform
  for (int gi = glo; gi <= ghi; ++gi) {  // wave-uniform; a boundary block runs once per group that has rows in it
    if (NKK > 0 && ghi > glo && __builtin_amdgcn_ballot_w64(grp_lane == gi) == 0) continue;
    v16f low[2];
    if constexpr (NKK > 0) {
      const float sgrp = g.lora_scaling[gi];
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) low[j][e] = 0.0f;
#pragma unroll
      for (int kk = 0; kk < NKK; ++kk) {
        if (PAIR || gi > glo) fetch_b(gi, kk, bf[kk]);
        if constexpr (PAIR) {
          if (g.zpart) z_from_quarters(kk, zf[kk]);
          else fetch_z(kk, zf[kk]);
        }
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int t3 = 2; t3 >= 0; --t3)
            low[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8bf, zf[kk][t3]), __builtin_bit_cast(v8bf, bf[kk][j]),
                                                             low[j], 0, 0, 0);
      }
      if constexpr (CHUNKS) {
        // of the rows of the group (bit 8 (e / 4) + e % 4: the lane's value e): slots without a row may hold anything
        const uint32_t rows = (uint32_t)__builtin_amdgcn_ballot_w64(row_ok && grp_lane == gi) >> (4 * h);
        bool again = false;
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const float probe = __builtin_fmaf(low[0][e], 0.0f, low[1][e] * 0.0f);  // NaN where one is not finite
          again |= !(probe == 0.0f) && ((rows >> (8 * (e >> 2) + (e & 3))) & 1u) != 0;
        }
        if (__builtin_amdgcn_ballot_w64(again) != 0) sums_again(gi, low);  // wave-uniform
      }
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) low[j][e] = low[j][e] * sgrp;
    }
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const int src_lane_addr = 16 * h + 4 * (8 * (v >> 2) + (v & 3));
      const uint32_t rowoff = (uint32_t)__builtin_amdgcn_ds_bpermute(src_lane_addr, (int)off_lane);
      const float sxv = __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute(src_lane_addr, __builtin_bit_cast(int, sx_lane)));
      const float t0 = (float)own[0][v] * sxv, t1 = (float)own[1][v] * sxv;
      float y0 = t0 * sw[0], y1 = t1 * sw[1];
      if constexpr (NKK > 0) {
        y0 = y0 + low[0][v];
        y1 = y1 + low[1][v];
      }
      bool row_valid = fast || rowoff != 0xffffffffu;
      if (NKK > 0 && ghi > glo) row_valid = row_valid && __builtin_amdgcn_ds_bpermute(src_lane_addr, grp_lane) == gi;
      if constexpr (EPI == kEpiSwiglu) {  // (y0, y1) = (gate, up) of product column ncol / 2
        const uint32_t f = pack_bf16x2(y0, y1);
        const float p = swiglu_f32(__uint_as_float(f << 16), __uint_as_float(f & 0xffff0000u));
        if (row_valid && (ncol >> 1) < n_out) reinterpret_cast<uint16_t*>(g.out)[rowoff + (ncol >> 1)] = (uint16_t)f32_to_bf16_bits(p);
      } else {
        uint16_t* o = reinterpret_cast<uint16_t*>(g.out) + (size_t)rowoff + ncol;
        if (!row_valid) continue;
        const bool in0 = full_n || ncol < g.N, in1 = full_n || ncol + 1u < g.N;
        if (g.residual) {
          const uint16_t* r = g.residual + (size_t)rowoff + ncol;
          const uint32_t rr = full_n ? *reinterpret_cast<const uint32_t*>(r) : (in0 ? r[0] : 0u) | (in1 ? (uint32_t)r[1] << 16 : 0u);
          y0 = y0 + __uint_as_float(rr << 16);
          y1 = y1 + __uint_as_float(rr & 0xffff0000u);
        }
        const uint32_t bits = pack_bf16x2(y0, y1);
        if (full_n) {
          *reinterpret_cast<uint32_t*>(o) = bits;
        } else {
          if (in0) o[0] = (uint16_t)(bits & 0xffffu);
          if (in1) o[1] = (uint16_t)(bits >> 16);
        }
      }
    }
  }
}

}  // namespace w8a8
