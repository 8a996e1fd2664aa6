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
// (8 accumulator blocks of v_mfma_f32_32x32x16_bf16), contraction in stages of one 32-wide n block.  A stage's
// dy panel (16 KiB), its four weight blocks (4 KiB, half that in 4-bit codes) and their scales (128 bytes a block)
// travel L2 -> LDS with direct-to-LDS loads four stages ahead, six per wave.  While the matrix core works on
// a stage, each wave prepares its weight block of the next: transposed by the identity MFMA, scaled in float32,
// split into TERMS bf16 operands.  The order of things is bwd_dx_wide_kernel's; two row blocks take turns so that the terms'
// MFMAs on one accumulator do not follow each other.
// Bound by the matrix core and the term arithmetic beside it: 1536 rows, K = 12288, N = 4096, 8-bit codes, groups of
// 64, two terms: 277 us, 1.12 PFLOP/s of bf16 products (as eight waves of 128 x 32, every two of which converted the same blocks, 322-337 us; the float32 library
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
    const unsigned char* Ag0 = g.dyp + ((size_t)(tm * 8u + rb0) * g.NB) * 2048u;
    const unsigned char* Ag1 = g.dyp + ((size_t)(tm * 8u + rb1) * g.NB) * 2048u;
    const uint32_t kb0 = tk * 4u;
    auto clamp_kb = [&](uint32_t kb) { return kb < g.KB ? kb : g.KB - 1u; };
    // its chunk of the weight blocks: one of four, or in 4-bit codes two of 512 bytes (waves 2 and 3 repeating 0 and 1)
    const uint32_t w_off = W4 ? clamp_kb(kb0 + 2u * ((uint32_t)wave & 1u) + h) * 512u + ((uint32_t)lane_s & 31u) * 16u
                              : clamp_kb(kb0 + (uint32_t)wave) * 1024u + lane16;
    const uint32_t w_dst = (W4 ? (uint32_t)wave & 1u : (uint32_t)wave) * 1024u;
    // the four blocks' scales, by each wave to the same place
    const uint32_t s_piece = ((uint32_t)lane_s & 7u) * 4u;
    const uint32_t s_row = clamp_kb(kb0 + (((uint32_t)lane_s >> 3) & 3u)) * 32u / a.group * a.N;
    auto issue = [&](int i, int j) {  // load j of the six of stage i (behind the last stage: of that one again)
      const uint32_t st = lds_base + (uint32_t)(i % kGqBwdStages) * kGqBwdStageBytes;
      const uint32_t nb = (uint32_t)(nb0 + (i < L ? i : L - 1));
      if (j < 4) {
        lds_load_1k((j < 2 ? Ag0 : Ag1) + (size_t)nb * 2048u + 1024 * (j & 1), lane16, st + (uint32_t)(wave * 4 + j) * kBlockBytes);
      } else if (j == 4) {
        const uint32_t nbw = nb < a.weight_nb ? nb : a.weight_nb - 1u;  // (dy is zero beyond the last column)
        lds_load_1k(g.wp + (size_t)nbw * g.KB * kBlk8, w_off, st + kGqBwdPanel + w_dst);
      } else {
        const uint32_t n = nb * 32u + s_piece;
        lds_load_1k(reinterpret_cast<const unsigned char*>(a.ws), (s_row + (n < a.N ? n : 0u)) * 4u, st + kGqBwdPanel + kGqBwdWeight);
      }
    };
    v16f acc[ROWS];
#pragma unroll
    for (int i = 0; i < ROWS; ++i)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][e] = 0.0f;

    // (the wait stands in the same block, so no register is handed out before it is filled)
    struct NextRegs { v4i raw; v4f s4[4]; };
    auto next_read = [&](int i, NextRegs& r) {
      const uint32_t st = lds_base + (uint32_t)(i % kGqBwdStages) * kGqBwdStageBytes + kGqBwdPanel;
      const uint32_t sa = st + kGqBwdWeight + (uint32_t)wave * 128u + 16u * h;
      if constexpr (W4) {
        const uint32_t wa = st + (uint32_t)wave * 512u + lane16 / 2u;
        uint2 raw;
        asm volatile("ds_read_b64 %0, %5\n\tds_read_b128 %1, %6\n\tds_read_b128 %2, %6 offset:32\n\t"
                     "ds_read_b128 %3, %6 offset:64\n\tds_read_b128 %4, %6 offset:96\n\ts_waitcnt lgkmcnt(0)"
                     : "=&v"(raw), "=&v"(r.s4[0]), "=&v"(r.s4[1]), "=&v"(r.s4[2]), "=&v"(r.s4[3])
                     : "v"(wa), "v"(sa) : "memory");
        GqRawFragment<true> f;
        f.v = make_uint4(raw.x, raw.y, 0u, 0u);
        r.raw = gq_expand<true>(f);  // 16 * code; the scale takes the exact 1 / 16
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
          for (int e = 0; e < 4; ++e) r.s4[q][e] = r.s4[q][e] * 0.0625f;
        // (the transposing MFMA is assembly: without wait states behind the vector ALU's write it read the last register of the
        // operand before it was written)
        asm volatile("s_nop 3" : "+v"(r.raw));
      } else {
        const uint32_t wa = st + (uint32_t)wave * 1024u + lane16;
        asm volatile("ds_read_b128 %0, %5\n\tds_read_b128 %1, %6\n\tds_read_b128 %2, %6 offset:32\n\t"
                     "ds_read_b128 %3, %6 offset:64\n\tds_read_b128 %4, %6 offset:96\n\ts_waitcnt lgkmcnt(0)"
                     : "=&v"(r.raw), "=&v"(r.s4[0]), "=&v"(r.s4[1]), "=&v"(r.s4[2]), "=&v"(r.s4[3])
                     : "v"(wa), "v"(sa) : "memory");
      }
    };
    // rows 8 (t / 2) + 4 h + 2 (t % 2) + 0, 1 of a transposed block: code * scale in float32, split into TERMS bf16 values
    auto convert2 = [&](const v16i& tr, const v4f (&s4)[4], int t, uint32_t (&pk)[TERMS][8]) {
      float f0 = (float)tr[2 * t] * s4[t >> 1][2 * (t & 1)], f1 = (float)tr[2 * t + 1] * s4[t >> 1][2 * (t & 1) + 1];
#pragma unroll
      for (int u = 0; u < TERMS; ++u) {
        const uint32_t w = pack_bf16x2(f0, f1);
        pk[u][t] = w;
        if (u + 1 < TERMS) {
          f0 = f0 - __uint_as_float(w << 16);
          f1 = f1 - __uint_as_float(w & 0xffff0000u);
        }
      }
    };
    auto to_operands = [&](const uint32_t (&pk)[TERMS][8], v8bf (&bq)[2][TERMS]) {
#pragma unroll
      for (int t = 0; t < TERMS; ++t)
#pragma unroll
        for (int q = 0; q < 2; ++q)
          bq[q][t] = __builtin_bit_cast(v8bf, v4i{(int)pk[t][4 * q], (int)pk[t][4 * q + 1], (int)pk[t][4 * q + 2], (int)pk[t][4 * q + 3]});
    };
    constexpr int kPairs = 2 * ROWS;  // (half q, row block) of a stage
    auto panel_frag = [&](int i, int pair) -> v8bf {
      typedef __attribute__((address_space(3))) const v4i* lds_v4ptr;
      const uint32_t at = lds_base + (uint32_t)(i % kGqBwdStages) * kGqBwdStageBytes + lane16;
      return __builtin_bit_cast(v8bf, *reinterpret_cast<lds_v4ptr>((uintptr_t)(at + (uint32_t)((pair % ROWS) * 2 + pair / ROWS) * kBlockBytes)));
    };
    // One stage: its MFMAs from the dy panel in the LDS, two row blocks at a time, small terms first; between them the operands
    // of stage i + 1 are prepared.  af: the fragments of the first two pairs; leaves those of stage i + 1 there where that one
    // has landed (ahead).
    auto stage = [&](int i, const v8bf (&bqC)[2][TERMS], v8bf (&bqN)[2][TERMS], bool ahead, v8bf (&af)[4]) {
      constexpr int kSlots = kPairs * TERMS;  // MFMAs
      constexpr int kFirst = 5, kGap = (kSlots - 6) / 8;  // where the eight conversion steps stand: four MFMAs behind the transposing one
      static_assert(kFirst + 7 * kGap < kSlots, "the conversion ends inside the stage");
      NextRegs nx;
      v16i tr;
      uint32_t pk[TERMS][8];
      asm volatile("s_nop 3");  // (operands converted at the end of the stage before)
      next_read(i + 1, nx);
#pragma unroll
      for (int p = 0; p < kPairs; p += 2) {
        const int q = p / ROWS, rb = p % ROWS;
#pragma unroll
        for (int t = TERMS - 1; t >= 0; --t)
#pragma unroll
          for (int u = 0; u < 2; ++u) {
            const int sl = p * TERMS + (TERMS - 1 - t) * 2 + u;
            bwd_mfma<true>(acc[rb + u], af[(p + u) & 3], bqC[q][t]);
            if (t == TERMS - 1) {  // the next two pairs' fragments
              if (p + 2 < kPairs) af[(p + 2 + u) & 3] = panel_frag(i, p + 2 + u);
              else if (ahead) af[(p + 2 + u) & 3] = panel_frag(i + 1, u);
            }
            if (sl == 0) bwd_transpose(tr, nx.raw, ident);
            if (sl == kFirst) asm volatile("" : "+v"(tr));  // (not read before this place)
            if (sl >= kFirst && (sl - kFirst) % kGap == 0 && (sl - kFirst) / kGap < 8) {
              convert2(tr, nx.s4, (sl - kFirst) / kGap, pk);
              if ((sl - kFirst) / kGap == 7) to_operands(pk, bqN);
            }
            if (sl % (kSlots / 8) == 1 && sl / (kSlots / 8) < kGqBwdLoads) issue(i + 4, sl / (kSlots / 8));
            __builtin_amdgcn_sched_barrier(0);
          }
      }
    };

    v8bf bqA[2][TERMS], bqB[2][TERMS], af[4];
    wait_vmcnt<0>();  // stores of the previous tile
    lds_barrier();
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < kGqBwdLoads; ++j) issue(i, j);
    wait_vmcnt<0>();
    lds_barrier();
    {  // operands of stage 0
      NextRegs nx;
      next_read(0, nx);
      uint32_t pk[TERMS][8];
      v16i tr;
      bwd_transpose(tr, nx.raw, ident);
      asm volatile("s_nop 15\n\ts_nop 15" : "+v"(tr));
#pragma unroll
      for (int t = 0; t < 8; ++t) convert2(tr, nx.s4, t, pk);
      to_operands(pk, bqA);
    }
    // Two stages to a barrier: stages i and i + 1 and the weight of i + 2 have landed, i + 4 and i + 5 are asked for
    // (into the slots of i - 2 and i - 1).
#pragma unroll 1
    for (int i = 0; i < L; i += 2) {
      wait_vmcnt<kGqBwdLoads>();
      lds_barrier();
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int p = 0; p < 2; ++p) af[p] = panel_frag(i, p);
      __builtin_amdgcn_sched_barrier(0);
      stage(i, bqA, bqB, true, af);
      stage(i + 1, bqB, bqA, false, af);
    }
    wait_vmcnt<0>();
    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");  // the last MFMAs, which the compiler does not know, have written their sums
#pragma unroll
    for (int rb = 0; rb < ROWS; ++rb) asm volatile("" : "+a"(acc[rb]));

    const uint32_t kbw = kb0 + (uint32_t)wave;
    if (whole) {
      lds_barrier();  // (every wave has read its last stage, and nothing is on its way into the LDS)
      const uint32_t rs_lds = lds_base + 4u * kBwdTurnBytes;
      bwd_dx_fetch_rs<NKK>(g, tm * 256u, live_blocks, rs_lds, wave, 4);
      bwd_dx_store<NKK, 1, ROWS, true>(g, tm * 256u, kbw, live_blocks, lds_base + (uint32_t)wave * kBwdTurnBytes, rs_lds,
                                       [&](int rb, int) -> v16f { return bwd_sums<true>(acc[rb]); });
    } else {
#pragma unroll
      for (int rb = 0; rb < ROWS; ++rb)
        if (rb < live_blocks) {
          float4* dst = bwd_dx_part<1>(g, slot, (uint32_t)rb, (uint32_t)wave);
          const v16f y = bwd_sums<true>(acc[rb]);
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
