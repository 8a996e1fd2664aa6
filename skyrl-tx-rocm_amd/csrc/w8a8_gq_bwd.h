// Backward of the group-scaled linear (W4 or W8 codes, one scale per K group and output):
//   dx = dy @ deq(W).T + rs @ A.T    rs = (dy @ B.T) * s      deq(W)[k, n] = float32(code * scale[g(k), n])
// and the LoRA cotangents of w8a8_backward.h (skyrl/tx/kernels/quantized_lora.py:337-394).  The rule there is
// float32 throughout; on the matrix core a float32 weight value is carried as its exact split into bf16
// terms, so that every product dy * deq(W) is exact and only float32 sums round, as in a float32 GEMM:
//   two terms when the scales are bf16 values (a code of at most 8 bits times 8 bits), three otherwise.
//
//   gq_bwd_pack_dy_kernel  dy in operand order, and the partial sums of r = dy @ B.T
//   gq_bwd_dx_wide_kernel  the pull-back
// The rest (tables, r / z finish, LoRA cotangents) is the per-channel backward's.
#pragma once
#include "w8a8_backward.h"
#include "w8a8_bwd_split.h"
#include "w8a8_gq.h"

namespace w8a8 {

// dy in MFMA A-operand order: dyp[row block][n block][q][64 lanes][8 bf16]: lane (i = l % 32, h = l / 32) element e
// of (n block nb, q) holds column 32 nb + 16 q + 8 (e / 4) + 4 h + e % 4, the n that the transposing MFMA
// leaves in contraction slot 8 h + e of its q-th half.  (bwd_pack_dy_kernel without the packed weight's column
// permutation.)  A lane loads 8 consecutive columns of its row, h of its 16, and the two halves of the wave
// exchange four of them.
template <int RB>  // 32-wide rank blocks (0 = packing only)
__global__ __launch_bounds__(256) void gq_bwd_pack_dy_kernel(BwdPackDyArgs a) {
  constexpr int kRB = RB > 0 ? RB : 1;
  __shared__ float red[4][kRB][16][64];
  const uint32_t lane = threadIdx.x & 63u, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t mb = blockIdx.x / a.n_slices, sl = blockIdx.x % a.n_slices;
  if (mb >= a.n_row_blocks) return;
  const uint32_t i = lane & 31u, h = lane >> 5;
  const uint32_t row = mb * 32u + i;
  v16f acc[kRB];
#pragma unroll
  for (int b = 0; b < kRB; ++b)
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[b][e] = 0.0f;
  const uint32_t per = (a.NB + a.n_slices - 1u) / a.n_slices;
  const uint32_t nb1 = (sl + 1u) * per < a.NB ? (sl + 1u) * per : a.NB;
  const uint16_t* const dyr = a.dy + (size_t)(row < a.M ? row : 0u) * a.N;
  // 16 columns in operand order; loads whatever the condition (a load under one becomes a branch with a wait)
  auto fetch = [&](const uint16_t* r, bool live, uint32_t col) -> v8us {
    const bool in = live && col < a.N;
    const v4i raw = *reinterpret_cast<const v4i*>(r + (col < a.N ? col : 0u));
    const v4i z = in ? raw : v4i{0, 0, 0, 0};
    const auto s0 = __builtin_amdgcn_permlane32_swap(z[0], z[2], false, false);
    const auto s1 = __builtin_amdgcn_permlane32_swap(z[1], z[3], false, false);
    return __builtin_bit_cast(v8us, v4i{(int)s0[0], (int)s1[0], (int)s0[1], (int)s1[1]});
  };
  for (uint32_t nb = sl * per + wave; nb < nb1; nb += 4u) {
    v8us pc[2];
#pragma unroll
    for (int q = 0; q < 2; ++q) pc[q] = fetch(dyr, row < a.M, 32u * nb + 16u * q + 8u * h);
    v8us wb[kRB][2];
    if constexpr (RB > 0) {
#pragma unroll
      for (int b = 0; b < RB; ++b) {
        const uint32_t j = b * 32u + i;
#pragma unroll
        for (int q = 0; q < 2; ++q) wb[b][q] = fetch(a.lora_b + (size_t)(j < a.r ? j : 0u) * a.N, j < a.r, 32u * nb + 16u * q + 8u * h);
      }
    }
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      *reinterpret_cast<v8us*>(a.dyp + ((((size_t)mb * a.NB + nb) * 2u + q) * 64u + lane) * 16u) = pc[q];
      if constexpr (RB > 0) {
#pragma unroll
        for (int b = 0; b < RB; ++b)
          acc[b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8bf, pc[q]), __builtin_bit_cast(v8bf, wb[b][q]), acc[b], 0, 0, 0);
      }
    }
  }
  if constexpr (RB > 0) {
#pragma unroll
    for (int b = 0; b < RB; ++b)
#pragma unroll
      for (int e = 0; e < 16; ++e) red[wave][b][e][lane] = acc[b][e];
    __syncthreads();
    for (uint32_t q = threadIdx.x; q < RB * 1024u; q += 256u) {
      const uint32_t l = q & 63u, e = (q >> 6) & 15u, b = q >> 10;
      const float sum = ((red[0][b][e][l] + red[1][b][e][l]) + red[2][b][e][l]) + red[3][b][e][l];
      const uint32_t r = 8u * (e >> 2) + 4u * (l >> 5) + (e & 3u), col = b * 32u + (l & 31u);
      a.rpart[((size_t)sl * a.slots + mb * 32u + r) * kBwdRankStride + col] = sum;
    }
  }
}

// ---------------------------------------------------------------------------------------
// The pull-back.  Workgroup = 4 waves side by side along k, one to a SIMD, tile 256 rows x 128 k, wave tile 256 x 32
// (16 x 2 accumulator blocks of v_mfma_f32_16x16x32_bf16), contraction in stages of one 32-wide n block.  A stage's
// dy panel (16 KiB), its four weight blocks (4 KiB, half that in 4-bit codes) and their scales (128 bytes a block)
// travel L2 -> LDS with direct-to-LDS loads four stages ahead, six per wave.  While the matrix core works on
// a stage, each wave prepares its weight block of the next: transposed by the identity MFMA, scaled in float32,
// split into TERMS bf16 operands.  The order of things is bwd_dx_wide_kernel's; two row blocks take turns so that the terms'
// MFMAs on one accumulator do not follow each other.
// Bound by the matrix core and the term arithmetic beside it: 1536 rows, K = 12288, N = 4096, 8-bit codes, groups of
// 64, two terms: 276 us, 1.12 PFLOP/s of bf16 products (282 with 32x32x16 and the loads' addresses formed anew for every stage; as eight waves of 128 x 32, every two of which converted the same blocks, 322-337 us; the float32 library
// GEMM took 1096 us and the dequantization and casts before it 250).
// ---------------------------------------------------------------------------------------
constexpr int kGqBwdStages = 6;
constexpr int kGqBwdPanel = 16384, kGqBwdWeight = 4096;
constexpr int kGqBwdStageBytes = kGqBwdPanel + kGqBwdWeight + 1024;
constexpr int kGqBwdLdsBytes = kGqBwdStages * kGqBwdStageBytes;
constexpr int kGqBwdLoads = 6;  // per wave and stage: 4 panel chunks, a weight chunk, scales

struct GqBwdDxArgs {
  BwdDxArgs g;          // wp: packed codes; KB: k blocks (k_pad / 32); NB: n blocks of dyp (even)
  const float* ws;      // f32 [k_pad / group, N]
  uint32_t N, group, weight_nb;  // weight_nb: n blocks of the packed weight
};

template <bool W4, int TERMS, int NKK>
__global__ __launch_bounds__(256, 1) void gq_bwd_dx_wide_kernel(GqBwdDxArgs a) {
  const BwdDxArgs& g = a.g;
  extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t lds_base = (uint32_t)(uintptr_t)(lptr_t)lds;
  constexpr uint32_t kBlk8 = W4 ? 512u : 1024u;  // bytes of a weight block
  // identity operand of the transposing MFMA: lane (column c, k half h) holds byte 1 at k == c
  v4i ident = {0, 0, 0, 0};
  {
    const int c = lane & 31, h = lane >> 5;
    const int word = ((c >> 4) == h) ? (int)(1u << (8 * (c & 3))) : 0;
    const int wi = (c & 15) >> 2;
    ident[0] = wi == 0 ? word : 0; ident[1] = wi == 1 ? word : 0;
    ident[2] = wi == 2 ? word : 0; ident[3] = wi == 3 ? word : 0;
  }

  // stages nb0 .. nb0 + L - 1 (an even number) of a tile: all of them (whole), or partial sums for slot `slot`; ROWS: row blocks
  // multiplied, at least live_blocks
  auto segment = [&](auto rows_tag, uint32_t tm, uint32_t tk, int live_blocks, int nb0, int L, bool whole, uint32_t slot) {
    constexpr int ROWS = decltype(rows_tag)::value;
    int lane_s = lane;
    asm volatile("" : "+v"(lane_s));  // (what is derived from it is formed per segment: see bwd_dx_wide_kernel)
    const uint32_t lane16 = (uint32_t)lane_s * 16u, h = (uint32_t)lane_s >> 5;
    const uint32_t rb0 = 2u * (uint32_t)wave < (uint32_t)live_blocks ? 2u * (uint32_t)wave : 0u;
    const uint32_t rb1 = 2u * (uint32_t)wave + 1u < (uint32_t)live_blocks ? 2u * (uint32_t)wave + 1u : 0u;
    const unsigned char* const Ag0 = g.dyp + ((size_t)(tm * 8u + rb0) * g.NB + (uint32_t)nb0) * 2048u;
    const unsigned char* const Ag1 = g.dyp + ((size_t)(tm * 8u + rb1) * g.NB + (uint32_t)nb0) * 2048u;
    const uint32_t kb0 = tk * 4u;
    auto clamp_kb = [&](uint32_t kb) { return kb < g.KB ? kb : g.KB - 1u; };
    // its chunk of the weight blocks: one of four, or in 4-bit codes two of 512 bytes (waves 2 and 3 repeating 0 and 1)
    const uint32_t w_off = W4 ? clamp_kb(kb0 + 2u * ((uint32_t)wave & 1u) + h) * 512u + ((uint32_t)lane_s & 31u) * 16u
                              : clamp_kb(kb0 + (uint32_t)wave) * 1024u + lane16;
    const uint32_t w_dst = (W4 ? (uint32_t)wave & 1u : (uint32_t)wave) * 1024u;
    // the four blocks' scales, by each wave to the same place
    const uint32_t s_piece = ((uint32_t)lane_s & 7u) * 4u;
    const uint32_t s_row = clamp_kb(kb0 + (((uint32_t)lane_s >> 3) & 3u)) * 32u / a.group * a.N;
    const size_t w_stride = (size_t)g.KB * kBlk8;
    const unsigned char* Wg = g.wp + (size_t)gq_bwd_first_block((uint32_t)nb0, a.weight_nb) * w_stride;
    uint32_t a_off = lane16, s_col = (uint32_t)nb0 * 32u + s_piece;
    int nb_load = nb0;
    // Part j of four of the loads of the next stage to be asked for, into the stage buffer at st (behind the last stage: of that
    // one again).  The addresses go on from stage to stage: see bwd_dx_wide_kernel.
    auto issue = [&](uint32_t st, int j) {
      if (j == 0) lds_load_2k(Ag0, a_off, st + (uint32_t)wave * 4096u);
      else if (j == 1) lds_load_2k(Ag1, a_off, st + (uint32_t)wave * 4096u + 2048u);
      else if (j == 2) lds_load_1k(Wg, w_off, st + kGqBwdPanel + w_dst);
      else {
        lds_load_1k(reinterpret_cast<const unsigned char*>(a.ws), (s_row + (s_col < a.N ? s_col : 0u)) * 4u, st + kGqBwdPanel + kGqBwdWeight);
        const bool more = nb_load + 1 < nb0 + L;
        nb_load += more ? 1 : 0;
        a_off += more ? 2048u : 0u;
        s_col += more ? 32u : 0u;
        Wg += more && gq_bwd_next_block((uint32_t)nb_load, a.weight_nb) ? w_stride : 0;
      }
    };
    constexpr int kRows16 = 2 * ROWS;  // row blocks of 16
    v4f acc[kRows16][2];
#pragma unroll
    for (int i = 0; i < kRows16; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[i][j][e] = 0.0f;

    struct NextRegs { v4i raw; v4f s4[4]; };
    const uint32_t weight_off = W4 ? (uint32_t)wave * 512u + lane16 / 2u : (uint32_t)wave * 1024u + lane16;
    // The weight block and scales of the stage at st, in three parts.  (Reads that the compiler waits for where they are used.)
    auto next_read = [&](uint32_t st, int part, NextRegs& r) {
      if (part == 0) {
        uint32_t wa = st + weight_off;
        asm volatile("" : "+v"(wa));
        if constexpr (W4) {
          typedef int v2i __attribute__((ext_vector_type(2)));
          typedef __attribute__((address_space(3))) const v2i* lds_v2ptr;
          const v2i raw = *reinterpret_cast<lds_v2ptr>((uintptr_t)(wa + kGqBwdPanel));
          r.raw[0] = raw[0]; r.raw[1] = raw[1];
        } else {
          typedef __attribute__((address_space(3))) const v4i* lds_v4ptr;
          r.raw = *reinterpret_cast<lds_v4ptr>((uintptr_t)(wa + kGqBwdPanel));
        }
      } else {
        typedef __attribute__((address_space(3))) const v4i* lds_v4ptr;
        uint32_t sa = st + (uint32_t)wave * 128u + 16u * h;
        asm volatile("" : "+v"(sa));
#pragma unroll
        for (int q = 2 * part - 2; q < 2 * part; ++q)
          r.s4[q] = __builtin_bit_cast(v4f, *reinterpret_cast<lds_v4ptr>((uintptr_t)(sa + kGqBwdPanel + kGqBwdWeight + 32 * q)));
      }
    };
    auto next_expand = [&](NextRegs& r) {  // 4-bit codes to 16 * code; the scale takes the exact 1 / 16 (convert_part)
      if constexpr (W4) {
        GqRawFragment<true> f;
        f.v = make_uint4((uint32_t)r.raw[0], (uint32_t)r.raw[1], 0u, 0u);
        r.raw = gq_expand<true>(f);
        // (the transposing MFMA is assembly: without wait states behind the vector ALU's write it read the last register of the
        // operand before it was written)
        asm volatile("s_nop 3" : "+v"(r.raw));
      }
    };
    // rows 8 (t / 2) + 4 h + 2 (t % 2) + 0, 1 of a transposed block: code * scale in float32, split into TERMS bf16 values
    // (step t in 3 * TERMS parts, which stand between different MFMAs)
    constexpr int kParts = 3 * TERMS;
    auto convert_part = [&](const v16i& tr, const v4f (&s4)[4], int t, int part, float (&f)[2], uint32_t (&pk)[TERMS][8]) {
      const int u = part / 3;
      if (part == 0) {
        f[0] = (float)tr[2 * t]; f[1] = (float)tr[2 * t + 1];
      } else if (part == 1) {
        constexpr float kUnit = W4 ? 0.0625f : 1.0f;
        f[0] = f[0] * (s4[t >> 1][2 * (t & 1)] * kUnit); f[1] = f[1] * (s4[t >> 1][2 * (t & 1) + 1] * kUnit);
      } else if (part % 3 == 0) {
        f[0] = f[0] - __uint_as_float(pk[u - 1][t] << 16);
      } else if (part % 3 == 1) {
        f[1] = f[1] - __uint_as_float(pk[u - 1][t] & 0xffff0000u);
      } else {
        pk[u][t] = pack_bf16x2(f[0], f[1]);
      }
    };
    auto operand_rows = [&](int t, uint32_t (&pk)[TERMS][8]) {  // behind step t >= 4
#pragma unroll
      for (int v = 0; v < TERMS; ++v) bwd_operand_rows(pk[v][t - 4], pk[v][t]);
    };
    auto to_operands = [&](const uint32_t (&pk)[TERMS][8], v8bf (&bq)[2][TERMS]) {
#pragma unroll
      for (int t = 0; t < TERMS; ++t)
#pragma unroll
        for (int j = 0; j < 2; ++j)
          bq[j][t] = __builtin_bit_cast(v8bf, v4i{(int)pk[t][4 * j], (int)pk[t][4 * j + 1], (int)pk[t][4 * j + 2], (int)pk[t][4 * j + 3]});
    };
    const uint32_t frag_off = bwd_frag_offset((uint32_t)lane_s);
    auto panel_at = [&](uint32_t st) -> uint32_t {
      uint32_t at = st + frag_off;
      asm volatile("" : "+v"(at));  // (opaque: the rows' offsets are the instructions', not sixteen registers)
      return at;
    };
    // One stage, at st: its MFMAs from the dy panel in the LDS, two blocks of 16 rows at a time, small terms first; between them
    // the operands of the stage at st_next are prepared and the loads of the one at st_load are issued.  af: the fragments of
    // the first two blocks; leaves the next stage's.
    auto stage = [&](uint32_t st, uint32_t st_next, uint32_t st_load, const v8bf (&bqC)[2][TERMS], v8bf (&bqN)[2][TERMS], v8bf (&af)[4]) {
      constexpr int kSlots = kRows16 * TERMS * 2;  // MFMAs
      // the transposing one stands behind kTurn, where its operand has come from the LDS; from kFirst on, five behind it, the
      // eight conversion steps
      constexpr int kTurn = ROWS == 8 ? 7 : 3, kFirst = kTurn + 5, kGap = (kSlots - kFirst - 1) / 8;
      static_assert(kGap > 0 && kFirst + 8 * kGap < kSlots, "the conversion ends inside the stage");
      NextRegs nx;
      v16i tr;
      uint32_t pk[TERMS][8];
      float cf[2];
      asm volatile("s_nop 3");  // (operands converted at the end of the stage before)
      const uint32_t panel = panel_at(st), panel_next = panel_at(st_next);
      auto slot = [&](auto at_slot) __attribute__((always_inline)) {
        constexpr int sl = decltype(at_slot)::value;
        constexpr int p = sl / (4 * TERMS) * 2, t = TERMS - 1 - sl / 4 % TERMS, u = sl / 2 % 2, j = sl % 2;
        bwd_mfma<true>(acc[p + u][j], af[(p + u) & 3], bqC[j][t]);
        if constexpr (t == TERMS - 1 && j == 0) {  // the next two blocks' fragments
          if constexpr (p + 2 < kRows16) af[(p + 2 + u) & 3] = bwd_panel_frag(panel, p + 2 + u);
          else af[(p + 2 + u) & 3] = bwd_panel_frag(panel_next, u);
        }
        if constexpr (sl == 1 || sl == 2 || sl == 3) next_read(st_next, sl - 1, nx);
        if constexpr (sl == kTurn) {
          next_expand(nx);
          bwd_transpose(tr, nx.raw, ident);
        }
        if constexpr (sl == kFirst) asm volatile("" : "+v"(tr));  // (not read before this place)
        if constexpr (sl >= kFirst && (sl - kFirst) % kGap == 0 && (sl - kFirst) / kGap > 4 && (sl - kFirst) / kGap <= 8) {
          operand_rows((sl - kFirst) / kGap - 1, pk);
          if constexpr ((sl - kFirst) / kGap == 8) to_operands(pk, bqN);
        }
        if constexpr (sl >= kFirst && sl < kFirst + 8 * kGap) {
          constexpr int step = (sl - kFirst) / kGap, at = (sl - kFirst) % kGap;
#pragma unroll
          for (int part = at * kParts / kGap; part < (at + 1) * kParts / kGap; ++part) convert_part(tr, nx.s4, step, part, cf, pk);
        }
        if constexpr (sl % (kSlots / 4) == kSlots / 8 && sl / (kSlots / 4) < 4) issue(st_load, sl / (kSlots / 4));
        __builtin_amdgcn_sched_barrier(0);
      };
      each_of(slot, std::make_integer_sequence<int, kSlots>{});
    };

    v8bf bqA[2][TERMS], bqB[2][TERMS], af[4];
    wait_vmcnt<0>();  // stores of the previous tile
    lds_barrier();
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) issue(lds_base + (uint32_t)i * kGqBwdStageBytes, j);
    wait_vmcnt<0>();
    lds_barrier();
    {  // operands of stage 0
      NextRegs nx;
#pragma unroll
      for (int part = 0; part < 3; ++part) next_read(lds_base, part, nx);
      next_expand(nx);
      uint32_t pk[TERMS][8];
      v16i tr;
      bwd_transpose(tr, nx.raw, ident);
      asm volatile("s_nop 15\n\ts_nop 15" : "+v"(tr));
#pragma unroll
      for (int t = 0; t < 8; ++t) {
        float cf[2];
#pragma unroll
        for (int part = 0; part < kParts; ++part) convert_part(tr, nx.s4, t, part, cf, pk);
        if (t >= 4) operand_rows(t, pk);
      }
      to_operands(pk, bqA);
    }
    // Two stages to a barrier: stages i, i + 1 and i + 2 have landed, i + 4 and i + 5 are asked for (into the buffers of i - 2
    // and i - 1).
#pragma unroll
    for (int p = 0; p < 2; ++p) af[p] = bwd_panel_frag(panel_at(lds_base), p);
    uint32_t st_load = lds_base + 4u * kGqBwdStageBytes, st = lds_base, st_next = lds_base + 2u * kGqBwdStageBytes;
#pragma unroll 1
    for (int i = 0; i < L; i += 2) {
      wait_vmcnt<kGqBwdLoads>();
      // (the reads in flight are of stage i, whose buffer is filled again two barriers on)
      asm volatile("s_barrier" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
      stage(st, st + kGqBwdStageBytes, st_load, bqA, bqB, af);
      stage(st + kGqBwdStageBytes, st_next, st_load + kGqBwdStageBytes, bqB, bqA, af);
      const uint32_t before = st_load;
      st_load = st; st = st_next; st_next = before;
    }
    wait_vmcnt<0>();
    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");  // the last MFMAs, which the compiler does not know, have written their sums
#pragma unroll
    for (int p = 0; p < kRows16; ++p)
#pragma unroll
      for (int j = 0; j < 2; ++j) asm volatile("" : "+a"(acc[p][j]));
    auto sums = [&](int rb, int) -> v16f {
      v4f b[2][2];
#pragma unroll
      for (int rh = 0; rh < 2; ++rh)
#pragma unroll
        for (int ch = 0; ch < 2; ++ch) b[rh][ch] = bwd_sums<true>(acc[2 * rb + rh][ch]);
      return bwd_block32(b);
    };

    const uint32_t kbw = kb0 + (uint32_t)wave;
    if (whole) {
      lds_barrier();  // (every wave has read its last stage, and nothing is on its way into the LDS)
      const uint32_t rs_lds = lds_base + 4u * kBwdTurnBytes;
      bwd_dx_fetch_rs<NKK>(g, tm * 256u, live_blocks, rs_lds, wave, 4);
      bwd_dx_store<NKK, 1, ROWS, true>(g, tm * 256u, kbw, live_blocks, lds_base + (uint32_t)wave * kBwdTurnBytes, rs_lds,
                                       sums);
    } else {
#pragma unroll
      for (int rb = 0; rb < ROWS; ++rb)
        if (rb < live_blocks) {
          float4* dst = bwd_dx_part<1>(g, slot, (uint32_t)rb, (uint32_t)wave);
          const v16f y = sums(rb, 0);
#pragma unroll
          for (int e = 0; e < 4; ++e) dst[e * 64] = make_float4(y[4 * e], y[4 * e + 1], y[4 * e + 2], y[4 * e + 3]);
        }
    }
  };

  // whole tiles (an XCD walks a contiguous range of the band-major order), then the split ones
  bwd_dx_schedule(g, true, [&](uint32_t t, int nb0, int len, uint32_t slot) {
    uint32_t tm, tk;
    bwd_dx_tile_at(g, t, tm, tk);
    const int live0 = ((int)(g.M - tm * 256u) + 31) / 32;
    const int live = __builtin_amdgcn_readfirstlane(live0 < 8 ? live0 : 8);
    if (live > 4) segment(std::integral_constant<int, 8>{}, tm, tk, live, nb0, len, len == (int)g.NB, slot);
    else segment(std::integral_constant<int, 4>{}, tm, tk, live, nb0, len, len == (int)g.NB, slot);
  });
}

// ---------------------------------------------------------------------------------------
// Operands that are not finite.  A sum of bf16 terms does not carry an infinity (inf * 0 and inf - inf are NaN where
// the float32 product is a signed infinity), nor does a transposition on the matrix core keep one to its
// column.  The preparation and the tables of r and z note such values (BwdRFinishArgs::beyond); the last launch
// then forms the LoRA cotangents as plain sums and rewrites the entries of dx that are infinite or NaN, as
// the rule in float32 gives them.  A finite call pays the look at the notes.
// ---------------------------------------------------------------------------------------
constexpr uint32_t kGqPlainDxBlocks = 256;
struct GqBwdPlain {
  static constexpr bool kAny = true;
  const uint32_t* beyond; uint32_t n_beyond;
  const uint16_t* x; const uint16_t* dy;          // bf16 [M, K], [M, N]
  const uint16_t* lora_a; const uint16_t* lora_b; // bf16 [K, r], [r, N]
  const float* rs;                                // f32 [M][64]
  uint16_t* dx;                                   // or null
  const unsigned char* wp; const float* ws;       // packed codes, scales [K_pad / group, N]
  uint32_t M, K, N, r, KB, group, bits;

  __device__ bool wanted() const {
    uint32_t any = 0;
    for (uint32_t i = threadIdx.x & 63u; i < n_beyond; i += 64u) any |= beyond[i];
    return __builtin_amdgcn_ballot_w64(any != 0) != 0;
  }
  __device__ static bool is_nan(double v) { return v != v; }
  __device__ float d_a(uint32_t k, uint32_t j) const {
    double sum = 0.0;
    for (uint32_t m = 0; m < M && !is_nan(sum); ++m)
      sum += (double)bf16_bits_to_f32(x[(size_t)m * K + k]) * (double)rs[(size_t)m * kBwdRankStride + j];
    return (float)sum;
  }
  __device__ float d_b(const float* z, uint32_t n, uint32_t j) const {
    double sum = 0.0;
    for (uint32_t m = 0; m < M && !is_nan(sum); ++m)
      sum += (double)z[(size_t)m * kBwdRankStride + j] * (double)bf16_bits_to_f32(dy[(size_t)m * N + n]);
    return (float)sum;
  }
  // This thread's share of sum(dy * (z @ B)).  By rows: r . z, or the products themselves where either is infinite.
  __device__ double d_s(const float* r_raw, const float* z) const {
    double sum = 0.0;
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    for (uint32_t m = 0; m < M && __builtin_amdgcn_ballot_w64(is_nan(sum)) == 0; ++m) {
      const size_t row = (size_t)m * kBwdRankStride;
      const float rv = lane < r ? r_raw[row + lane] : 0.0f, zv = lane < r ? z[row + lane] : 0.0f;
      if (__builtin_amdgcn_ballot_w64(beyond_bf16_terms(rv) || beyond_bf16_terms(zv)) == 0) {
        if (wave == (m & 3u)) sum += (double)rv * (double)zv;
        continue;
      }
      for (uint32_t n = threadIdx.x; n < N; n += 256u) {
        float zb = 0.0f;
        for (uint32_t j = 0; j < r; ++j) zb += z[row + j] * bf16_bits_to_f32(lora_b[(size_t)j * N + n]);
        sum += (double)(bf16_bits_to_f32(dy[(size_t)m * N + n]) * zb);
      }
    }
    return sum;
  }
  __device__ float weight(uint32_t k, uint32_t n) const {
    const size_t blk = (size_t)(n >> 5) * KB + (k >> 5);
    const uint32_t lane = (n & 31u) + 32u * ((k >> 4) & 1u), j = k & 15u;
    int code;
    if (bits == 8u) {
      code = (int8_t)wp[blk * 1024u + lane * 16u + j];
    } else {
      const uint32_t byte = wp[blk * 512u + lane * 8u + 4u * (j >> 3) + (j & 3u)];
      code = (int8_t)((j & 4u) ? byte & 0xf0u : byte << 4) / 16;
    }
    return (float)code * ws[(size_t)(k / group) * N + n];
  }
  // Entries of dx that are not finite: all of a row whose r is not, and a column's whose row of A is not.  Their finite
  // terms do not matter.
  __device__ void d_x(uint32_t block) const {
    if (!dx) return;
    __shared__ uint16_t list[256];
    __shared__ uint32_t count;
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    for (uint32_t m = block; m < M; m += kGqPlainDxBlocks) {
      const float* const rsm = rs + (size_t)m * kBwdRankStride;
      const bool bad_row = __builtin_amdgcn_ballot_w64(lane < r && beyond_bf16_terms(rsm[lane < r ? lane : 0u])) != 0;
      for (uint32_t k0 = 0; k0 < K; k0 += 256u) {
        const uint32_t k = k0 + tid;
        bool redo = bad_row && k < K;
        float v = 0.0f;
        if (k < K) {
          for (uint32_t j = 0; j < r; ++j) {
            const float av = bf16_bits_to_f32(lora_a[(size_t)k * r + j]);
            redo = redo || beyond_bf16_terms(av);
            v += rsm[j] * av;
          }
        }
        if (__syncthreads_or(redo && v == v)) {  // (what is NaN stays NaN)
          for (uint32_t n0 = 0; n0 < N; n0 += 256u) {
            if (tid == 0) count = 0;
            __syncthreads();
            if (n0 + tid < N && (dy[(size_t)m * N + n0 + tid] & 0x7f80u) == 0x7f80u) list[atomicAdd(&count, 1u)] = (uint16_t)tid;
            __syncthreads();
            if (redo) {
              for (uint32_t i = 0; i < count && v == v; ++i) {
                const uint32_t n = n0 + list[i];
                v += bf16_bits_to_f32(dy[(size_t)m * N + n]) * weight(k, n);
              }
            }
            __syncthreads();
          }
        }
        if (!redo) continue;
        if (!(v != v || __builtin_isinf(v)))  // (r of nearly the largest float: finite, but not a sum of bf16 terms)
          for (uint32_t n = 0; n < N; ++n) v += bf16_bits_to_f32(dy[(size_t)m * N + n]) * weight(k, n);
        dx[(size_t)m * K + k] = (uint16_t)f32_to_bf16_bits(v);
      }
    }
  }
};

}  // namespace w8a8
