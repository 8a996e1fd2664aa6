// Backward of the W8A8 LoRA linear: the W8A16 input pull-back and the LoRA cotangents.
//   dx  = dy @ bf16(codes * sw).T  +  rs @ A[g].T          rs = (dy @ B[g].T) * s[g]
//   dA[g] = x_g.T @ rs_g      dB[g] = ((x_g @ A[g]).T @ dy_g) * s[g]      ds[g] = sum(dy_g * ((x_g @ A[g]) @ B[g]))
// Equations: skyrl/tx/kernels/quantized_lora.py:337-394.  The frozen weight enters the pull-back
// as bf16(codes * scales) per element with float32 accumulation of bf16 products, the policy of
// the reference's ROCm kernel (skyrl/tx/kernels/rocm/w8a8_lora.py:298-339); the LoRA terms stay in
// float32 and every cotangent is cast once.
//
// The packed weight keeps 16 consecutive k of one output column n in a lane; the pull-back
// contracts over n, so every 32 x 32 byte block is transposed on the matrix core itself:
// v_mfma_i32_32x32x32_i8 of the block against an identity operand returns W[n][k] with lane = k and
// sixteen n per lane, exactly the B operand of v_mfma_f32_32x32x16_bf16 once the integers are
// scaled and rounded to bf16.  No transposed ("shadow") copy of the weight exists.
#pragma once
#include <type_traits>

#include "w8a8_device.h"
#include "w8a8_prologue.h"

namespace w8a8 {

// ---------------------------------------------------------------------------------------
// dy in MFMA A-operand order: dyp[row block][n block][q][64 lanes][8 bf16] (1 KiB per (block, q)).
// Lane (i = l % 32, h = l / 32) element e of (n block nb, q) holds packed weight column
//   32 nb + 16 q + 8 (e / 4) + 4 h + e % 4,
// the n that the transposing MFMA leaves in contraction slot 8 h + e of its q-th half.  Rows are
// in grouped (adapter-sorted) slot order; slots without a row and columns beyond N are zero.
// A wave takes a row block and a 128-column group at a time: a lane owns 4 x 16 consecutive
// original columns of its row, the pieces of the eight packed blocks (q, j = column % 4)
// that interleave them.
// The same pass computes r = dy @ B[group].T on bf16 MFMAs (the 8-value pieces a lane has loaded
// are A operands as they are; the matching pieces of B are 16-byte loads), so dy is read once:
// a workgroup of four waves owns one 32-row block and one slice of the 128-column groups, and
// leaves its partial sum in rpart[slice][slot][64]; bwd_r_finish_kernel adds the slices.
// ---------------------------------------------------------------------------------------
constexpr uint32_t kBwdRankStride = 64;  // floats per slot in the z / r tables
constexpr uint32_t kBwdChunkRows = 512;  // rows of a chunk of the LoRA cotangents
constexpr uint32_t kBwdStageRows = 256;  // rows whose skinny operand sits in LDS at a time

struct BwdPackDyArgs {
  const uint16_t* dy;        // bf16 [M, N]
  const int32_t* src_row;    // original row of a slot or null (identity)
  const int32_t* slot_group; // or null (group 0)
  const int32_t* blk_range;  // or null
  unsigned char* dyp;
  const uint16_t* lora_b;    // bf16 [n_groups, r, N] or null (no LoRA: packing only)
  float* rpart;              // f32 [n_slices][slots][64]
  uint32_t M, N, NB, n_row_blocks, n_col_groups, n_slices, groups_per_slice, r, slots;
};

// dy arrives in whole lines, 4 rows x 256 bytes a load and the next group's under this one's work, and changes hands through the
// LDS, piece p of row r in place p ^ (r % 16), so that neither side has bank conflicts.  Asked for as it is consumed (32 rows x two
// pieces of 16 bytes a load, each under a condition and so with a wait of its own) it took, us before -> now: 3003 x 24576, rank 32
// 84.5 -> 67.2 (298 MB); 2048 x 10240, rank 64 24.8 -> 22.2; 333 x 6144, rank 64 12.5 -> 8.2; 8168 x 2048, rank 16 15.0 -> 13.9.
template <int RB>  // 32-wide rank blocks (0 = packing only)
__global__ __launch_bounds__(256, 3) void bwd_pack_dy_kernel(BwdPackDyArgs a) {
  constexpr int kRB = RB > 0 ? RB : 1;
  __shared__ __attribute__((aligned(1024))) unsigned char lds[4][8192];  // a tile of 32 rows x 128 columns per wave; later the waves' sums of r
  static_assert(sizeof(lds) >= 4u * kRB * 16u * 64u * 4u, "");
  const uint32_t lane = threadIdx.x & 63u, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t mb = blockIdx.x / a.n_slices, sl = blockIdx.x % a.n_slices;
  if (mb >= a.n_row_blocks) return;
  if (a.blk_range && a.blk_range[mb] < 0) return;  // block without rows (grouped calls): never consumed
  const uint32_t i = lane & 31u, h = lane >> 5;
  const uint32_t p = mb * 32u + i;
  int src = -1;
  if (a.src_row) src = a.src_row[p]; else if (p < a.M) src = (int)p;
  if (src >= (int)a.M) src = -1;
  const uint32_t range = (RB > 0 && a.blk_range) ? (uint32_t)a.blk_range[mb] : 0u;
  const uint32_t glo = range & 0xffffu, ghi = range >> 16;
  const uint32_t rowgrp = (RB > 0 && a.slot_group && ghi > glo) ? (uint32_t)a.slot_group[p] : glo;
  v16f acc[kRB];
#pragma unroll
  for (int b = 0; b < kRB; ++b)
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[b][e] = 0.0f;
  // load u of a group: piece lane % 16 (8 columns) of row 4 u + lane / 16
  const uint32_t lp = lane & 15u, lr = lane >> 4;
  uint32_t row_off[8];
  uint32_t rows_on = 0u;
#pragma unroll
  for (uint32_t u = 0; u < 8; ++u) {
    const int r = __shfl(src, (int)(4u * u + lr), 64);
    row_off[u] = r < 0 ? 0u : (uint32_t)r * a.N;
    rows_on |= r < 0 ? 0u : 1u << u;
  }
  auto fetch = [&](uint32_t G, v4i (&d)[8]) {  // (a row or column that is not there: the tensor's first bytes, cleared where they are used)
    const uint32_t col = 128u * G + 8u * lp < a.N ? 128u * G + 8u * lp : 0u;
#pragma unroll
    for (uint32_t u = 0; u < 8; ++u) {
      uint32_t off = row_off[u];
      asm volatile("" : "+v"(off));  // (eight 64-bit addresses kept across the loop would spill)
      d[u] = *reinterpret_cast<const v4i*>(a.dy + ((size_t)off + col));
    }
  };
  // B of a group: rows of ranks beyond r lie behind the resource and read as zeros.  The whole offset is the lane's: the check takes a
  // scalar offset off the resource's size, and the columns behind the matrix would take more than there is.
  const uint32_t b_off = (i * a.N + 16u * h) * 2u;
  typedef __attribute__((address_space(3))) v4i* lds_v4ptr;
  const uint32_t tile = (uint32_t)(uintptr_t)(lptr_t)lds + wave * 8192u;
  const uint32_t g_end = (sl + 1u) * a.groups_per_slice < a.n_col_groups ? (sl + 1u) * a.groups_per_slice : a.n_col_groups;
  v4i d[8];
  uint32_t G = sl * a.groups_per_slice + wave;
  if (G < g_end) fetch(G, d);
#pragma unroll 1
  for (; G < g_end; G += 4u) {
    const bool cols_on = 128u * G + 8u * lp < a.N;
#pragma unroll
    for (uint32_t u = 0; u < 8; ++u) {
      const v4i zero = {0, 0, 0, 0};
      *reinterpret_cast<lds_v4ptr>((uintptr_t)(tile + (4u * u + lr) * 256u + (lp ^ ((4u * u + lr) & 15u)) * 16u)) =
          (rows_on >> u) & 1u && cols_on ? d[u] : zero;
    }
    // piece 4 q + t, t = 2 ch + part: the 8 columns 128 G + 64 q + 32 ch + 16 h + 8 part .. + 7 of the lane's row
    auto piece_of = [&](int q, int t) { return 8u * q + 4u * (t >> 1) + 2u * h + (t & 1); };
    v8us wb[kRB][4];
    auto fetch_b = [&](uint32_t grp, int q) {
      const __amdgpu_buffer_rsrc_t brsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(a.lora_b) + (size_t)grp * a.r * a.N, 0,
                                                                             (int)(a.r * a.N * 2u), 0x00020000);
      const uint32_t off = b_off + (128u * G + 64u * q) * 2u;
#pragma unroll
      for (int b = 0; b < RB; ++b)
#pragma unroll
        for (int t = 0; t < 4; ++t)
          wb[b][t] = __builtin_bit_cast(v8us, __builtin_amdgcn_raw_buffer_load_b128(brsrc, off + 64u * b * a.N + (t >> 1) * 64u + (t & 1) * 16u, 0, 0));
      if (128u * G + 128u > a.N) {  // (columns beyond N are another rank's)
#pragma unroll
        for (int b = 0; b < RB; ++b)
#pragma unroll
          for (int t = 0; t < 4; ++t)
            if (128u * G + 8u * piece_of(q, t) >= a.N) wb[b][t] = v8us{0, 0, 0, 0, 0, 0, 0, 0};
      }
    };
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      if constexpr (RB > 0) fetch_b(glo, q);
      v8us pc[4];
#pragma unroll
      for (int t = 0; t < 4; ++t)
        pc[t] = __builtin_bit_cast(v8us, *reinterpret_cast<lds_v4ptr>((uintptr_t)(tile + i * 256u + (piece_of(q, t) ^ (i & 15u)) * 16u)));
      __builtin_amdgcn_wave_barrier();
      if (q == 1 && G + 4u < g_end) fetch(G + 4u, d);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        // element e < 4 of packed block j: column 4 e + j of the first 16, e >= 4: of the second 16
        v8us o;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          o[e] = pc[(4 * e + j) >> 3][(4 * e + j) & 7];
          o[4 + e] = pc[2 + ((4 * e + j) >> 3)][(4 * e + j) & 7];
        }
        const size_t off = ((((size_t)mb * a.NB + 4u * G + j) * 2u + q) * 64u + lane) * 16u;
        *reinterpret_cast<v8us*>(a.dyp + off) = o;
      }
      if constexpr (RB > 0) {
        // a block at a group boundary runs once per group with the other groups' rows zeroed
#pragma unroll 1
        for (uint32_t grp = glo;;) {
          const bool mine = src >= 0 && rowgrp == grp;
#pragma unroll
          for (int t = 0; t < 4; ++t) {
            const v8us zero = {0, 0, 0, 0, 0, 0, 0, 0};
            const v8bf xa = __builtin_bit_cast(v8bf, mine ? pc[t] : zero);
#pragma unroll
            for (int b = 0; b < RB; ++b)
              acc[b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xa, __builtin_bit_cast(v8bf, wb[b][t]), acc[b], 0, 0, 0);
          }
          if (++grp > ghi) break;
          fetch_b(grp, q);
        }
      }
    }
  }
  if constexpr (RB > 0) {
    float (*const red)[kRB][16][64] = reinterpret_cast<float (*)[kRB][16][64]>(&lds[0][0]);
    __syncthreads();  // everybody's tiles are spent
#pragma unroll
    for (int b = 0; b < RB; ++b)
#pragma unroll
      for (int e = 0; e < 16; ++e) red[wave][b][e][lane] = acc[b][e];
    __syncthreads();
    for (uint32_t q = threadIdx.x; q < RB * 1024u; q += 256u) {
      const uint32_t l = q & 63u, e = (q >> 6) & 15u, b = q >> 10;
      const float sum = ((red[0][b][e][l] + red[1][b][e][l]) + red[2][b][e][l]) + red[3][b][e][l];
      const uint32_t row = 8u * (e >> 2) + 4u * (l >> 5) + (e & 3u), col = b * 32u + (l & 31u);
      a.rpart[((size_t)sl * a.slots + mb * 32u + row) * kBwdRankStride + col] = sum;
    }
  }
}

// r and z of a 32-row block: the slices' partial sums added in slice order.  r is written raw, scaled by the row's group (for
// dA), and the scaled value split exactly into three bf16 terms in the operand order of the pull-back epilogue,
// rp[block][kk][term][lane][8]; z is the plain sum, and row_dot the row's r . z in double (for dscaling).
// Bound by the latency of the loads: a workgroup reads 32 rows x n_slices slices, and adding as the slices arrive, a value
// at a time, waited once per slice and value (2048 rows, rank 64, 8 slices: 21.3 us for r and 7.1 us for the 2 slices of z,
// 64 workgroups each).  With four columns a thread and all slices' loads in flight together, both in one launch: 5.6 us
// (3003 rows, rank 32: 11.9 + 10.4 against 4.9).
constexpr uint32_t kBwdMaxSlices = 8;
struct BwdRFinishArgs {
  const float* rpart; const float* zpart;  // [slices][slots][64]
  const int32_t* slot_group; const int32_t* blk_range; const float* lora_scaling;
  float* r_raw; float* rs; unsigned char* rp; float* z;
  double* row_dot;  // [slots]
  uint32_t n_slices, z_slices, slots, nkk, cols, r;  // cols = 16 * nkk rounded up to 32; z_slices 0: no z
  uint32_t* beyond;  // set where a value is beyond what bf16 terms can carry, or null
  // z of every row as the forward left it, f32 [M, r], in the place of zpart, and the row of a slot (null: its own); or null
  const float* z_rows; const int32_t* src_row;
  uint32_t M;
};

// A float32 value that is no sum of bf16 terms: not finite, or rounded to infinity by the first of them.
__device__ inline bool beyond_bf16_terms(float v) { return (__float_as_uint(v) & 0x7fffffffu) >= 0x7f7f8000u; }

__global__ __launch_bounds__(256) void bwd_r_finish_kernel(BwdRFinishArgs a) {
  __shared__ float zs[32][kBwdRankStride + 1];
  const uint32_t pb = blockIdx.x;
  if (a.blk_range && a.blk_range[pb] < 0) return;  // block without rows (grouped calls): never consumed
  const uint32_t quads = a.cols / 4u;  // 8 or 16 lanes to a row
  const size_t slice = (size_t)a.slots * kBwdRankStride;
  for (uint32_t q = threadIdx.x; q < 32u * quads; q += 256u) {
    const uint32_t row = q / quads, col = q % quads * 4u, slot = pb * 32u + row;
    const size_t at = (size_t)slot * kBwdRankStride + col;
    float4 v[kBwdMaxSlices], u[kBwdMaxSlices];
#pragma unroll
    for (uint32_t sl = 0; sl < kBwdMaxSlices; ++sl) v[sl] = *reinterpret_cast<const float4*>(a.rpart + at + (sl < a.n_slices ? sl : 0u) * slice);
    if (a.z_slices) {
#pragma unroll
      for (uint32_t sl = 0; sl < kBwdMaxSlices; ++sl) u[sl] = *reinterpret_cast<const float4*>(a.zpart + at + (sl < a.z_slices ? sl : 0u) * slice);
    }
    const float sc = a.lora_scaling[a.slot_group ? (uint32_t)a.slot_group[slot] : 0u];
    float raw[4] = {0.0f, 0.0f, 0.0f, 0.0f}, scaled[4], z[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (uint32_t sl = 0; sl < kBwdMaxSlices; ++sl)
      if (sl < a.n_slices) { raw[0] += v[sl].x; raw[1] += v[sl].y; raw[2] += v[sl].z; raw[3] += v[sl].w; }
    bool bad = false;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      scaled[e] = raw[e] * sc;
      bad |= beyond_bf16_terms(raw[e]) || beyond_bf16_terms(scaled[e]);
      zs[row][col + e] = scaled[e];
    }
    *reinterpret_cast<float4*>(a.r_raw + at) = make_float4(raw[0], raw[1], raw[2], raw[3]);
    *reinterpret_cast<float4*>(a.rs + at) = make_float4(scaled[0], scaled[1], scaled[2], scaled[3]);
    if (a.z_slices || a.z_rows) {
      if (a.z_rows) {  // kernel-uniform
        const int src = a.src_row ? a.src_row[slot] : (int)slot;
        const bool row_ok = src >= 0 && src < (int)a.M;
        const float* zr = a.z_rows + (row_ok && col < a.r ? (size_t)src * a.r + col : 0u);
        if ((a.r & 3u) == 0) {  // kernel-uniform
          const float4 v4 = *reinterpret_cast<const float4*>(zr);
          if (row_ok && col < a.r) { z[0] = v4.x; z[1] = v4.y; z[2] = v4.z; z[3] = v4.w; }
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (row_ok && col + e < a.r) z[e] = zr[e];
        }
      }
#pragma unroll
      for (uint32_t sl = 0; sl < kBwdMaxSlices; ++sl)
        if (sl < a.z_slices) { z[0] += u[sl].x; z[1] += u[sl].y; z[2] += u[sl].z; z[3] += u[sl].w; }
      *reinterpret_cast<float4*>(a.z + at) = make_float4(z[0], z[1], z[2], z[3]);
      double dot = 0.0;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        bad |= beyond_bf16_terms(z[e]);
        if (col + e < a.r) dot += (double)raw[e] * (double)z[e];  // (beyond the rank: x times a zero of A, no number that counts)
      }
      for (uint32_t o = 1; o < quads; o <<= 1) dot += __shfl_xor(dot, (int)o, 64);
      if (col == 0) a.row_dot[slot] = dot;
    }
    if (a.beyond && bad) *a.beyond = 1u;
  }
  __syncthreads();
  for (uint32_t q = threadIdx.x; q < a.nkk * 3u * 64u; q += 256u) {
    const uint32_t l = q & 63u, term = (q >> 6) % 3u, kk = q / 192u;
    const uint32_t row = l & 31u, hh = l >> 5;
    v8us o;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float z = zs[row][16u * kk + 8u * hh + e];
      const uint32_t b0 = f32_to_bf16_bits(z);
      const float r1 = z - bf16_bits_to_f32(b0);
      const uint32_t b1 = f32_to_bf16_bits(r1);
      const float r2 = r1 - bf16_bits_to_f32(b1);
      const uint32_t b2 = f32_to_bf16_bits(r2);
      o[e] = (unsigned short)(term == 0 ? b0 : (term == 1 ? b1 : b2));
    }
    *reinterpret_cast<v8us*>(a.rp + (((size_t)pb * a.nkk + kk) * 3u + term) * kBlockBytes + l * 16u) = o;
  }
}

// ---------------------------------------------------------------------------------------
// Small per-call tables: LoRA A in B-operand order for the pull-back epilogue,
//   ap[group][k block][kk][64 lanes][8]: lane (c, h) holds A[group][32 kb + c][16 kk + 8 h + 0..7],
// and the per-channel scales in packed column order, swp[p] = sw[packed_to_orig_col(p)].
// ---------------------------------------------------------------------------------------
__device__ inline v8us lora_a_operand_item(const uint16_t* __restrict__ a, unsigned char* __restrict__ ap,
                                           uint32_t n_groups, uint32_t K, uint32_t r, uint32_t kb32, uint32_t nkk,
                                           uint64_t idx) {
  const uint64_t total = (uint64_t)n_groups * kb32 * nkk * 64u;
  if (idx >= total) return v8us{0, 0, 0, 0, 0, 0, 0, 0};
  const uint32_t l = (uint32_t)(idx & 63u);
  const uint64_t rest = idx >> 6;
  const uint32_t kk = (uint32_t)(rest % nkk);
  const uint64_t gc = rest / nkk;
  const uint32_t kb = (uint32_t)(gc % kb32), grp = (uint32_t)(gc / kb32);
  const uint32_t k = kb * 32u + (l & 31u);
  v8us o;
  const uint32_t row0 = 16u * kk + 8u * (l >> 5);
  if ((r & 7u) == 0) {  // kernel-uniform: one 16-byte load (unconditional, like the ones below: a load under a lane
    const bool in = k < K && row0 < r;  // condition becomes a branch with a wait of its own)
    const v8us zero = {0, 0, 0, 0, 0, 0, 0, 0};
    const v8us v = *reinterpret_cast<const v8us*>(a + (in ? ((size_t)grp * K + k) * r + row0 : 0u));
    o = in ? v : zero;
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const bool in = k < K && row0 + e < r;
      const uint16_t v = a[in ? ((size_t)grp * K + k) * r + row0 + e : 0u];
      o[e] = in ? v : (uint16_t)0;
    }
  }
  *reinterpret_cast<v8us*>(ap + idx * 16u) = o;
  return o;
}

struct BwdPrepArgs {
  const int32_t* idx;        // adapter per row, or null
  int32_t* src_row; int32_t* slot_group; int32_t* blk_range; int32_t* group_off;
  const uint16_t* lora_a;    // bf16 [n_groups, K, r]
  uint16_t* at;              // bf16 [n_groups, r, K]
  unsigned char* ap;
  const float* sw; float* swp;
  uint32_t M, K, N, N_pad, n_groups, r, nkk, kb32, slots, route_blocks, a_blocks, ap_blocks;
  uint32_t* beyond;          // word 0 cleared, words 1 .. ap_blocks: A not finite somewhere in that block; or null
};

__global__ __launch_bounds__(1024) void bwd_prep_kernel(BwdPrepArgs p) {
  uint32_t b = blockIdx.x;
  if (b < p.route_blocks) {
    if (p.beyond && threadIdx.x == 0) p.beyond[0] = 0u;
    if (p.idx) {
      route_rows_block(p.idx, p.M, p.n_groups, p.slots, p.src_row, nullptr, p.slot_group, p.blk_range, p.group_off);
    } else {  // one adapter for every row: identity order, everything in group 0
      for (uint32_t g = threadIdx.x; g <= p.n_groups; g += 1024u) p.group_off[g] = g == 0 ? 0 : (int)p.M;
    }
    return;
  }
  b -= p.route_blocks;
  if (b < p.a_blocks) {
    lora_a_transpose_item(p.lora_a, p.at, p.n_groups, p.K, p.r, (uint64_t)b * 1024u + threadIdx.x);
    return;
  }
  b -= p.a_blocks;
  if (b < p.ap_blocks) {
    const v8us o = lora_a_operand_item(p.lora_a, p.ap, p.n_groups, p.K, p.r, p.kb32, p.nkk, (uint64_t)b * 1024u + threadIdx.x);
    if (p.beyond) {  // kernel-uniform
      int bad = 0;
#pragma unroll
      for (int e = 0; e < 8; ++e) bad |= (o[e] & 0x7f80u) == 0x7f80u;
      bad = __syncthreads_or(bad);
      if (threadIdx.x == 0) p.beyond[1u + b] = bad ? 1u : 0u;
    }
    return;
  }
  b -= p.ap_blocks;
  const uint32_t c = b * 1024u + threadIdx.x;
  if (c < p.N_pad) {
    const uint32_t n = packed_to_orig_col(c);
    p.swp[c] = n < p.N ? p.sw[n] : 0.0f;
  }
}

// ---------------------------------------------------------------------------------------
// Tables of a grouped (per-expert) backward: the rows arrive sorted by group, group g owning
// group_sizes[g] consecutive rows, and groups_per_weight consecutive groups share a frozen weight
// (skyrl/tx/layers/lora.py:394-444).  Every weight's rows start at a multiple of the pull-back's tile rows
// (256 slots, or 128 when the weights average few rows), so that
// a pull-back tile never mixes two weights; inside a weight the groups follow each other without
// gaps, exactly as the adapters of a dense call over that weight's rows would.
//   src_row / slot_group / blk_range             as in the dense call; blk_range -1 for 32-slot blocks without a
//                                                row: no kernel prepares or consumes their operands
//   group_beg[g], group_end[g]                   slots of group g
//   tile_weight[t]                               weight of tile t | its rows << 16, -1 beyond the slots in use
//   chunk_tab[c] = (group, first slot, rows)     the 512-row chunks of the LoRA cotangents; rows 0 beyond
//   chunk0[g]                                    first chunk of group g (n_groups + 1 entries)
// Part `part` of `n_parts` workgroups of 1024 threads: every part forms the prefix sums for itself (at most 1024 groups, one
// per thread) and fills its share of the tables, slot by slot.  Rows beyond sum(group_sizes) get no slot; their dx
// rows are cleared.  (As one workgroup whose first thread walked the groups this took 24 us of the launch's 26 for 128
// groups of 8168 rows.)
// ---------------------------------------------------------------------------------------
struct BwdGroupTables {
  int32_t* src_row; int32_t* slot_group; int32_t* blk_range;
  int32_t* group_beg; int32_t* group_end; int32_t* tile_weight; int32_t* chunk_tab; int32_t* chunk0;
  // rows of x gathered through a map: x_row[slot] is the row of x that src_row[slot] stands for
  int32_t* x_row; const int32_t* x_map; uint32_t x_div, x_rows;
};

__device__ inline void route_weight_groups_block(const int32_t* __restrict__ group_sizes, uint32_t M, uint32_t n_groups,
                                                 uint32_t gpw, uint32_t slots, uint32_t max_chunks, BwdGroupTables t,
                                                 uint16_t* __restrict__ dx, uint32_t K, uint32_t tile_rows, uint32_t part,
                                                 uint32_t n_parts) {
  __shared__ uint32_t row_start[kMaxGroups + 1];
  __shared__ uint32_t weight_slot[kMaxGroups];  // of a weight's first group: first slot of the weight
  __shared__ int last_group[kMaxGroups];        // of a weight's first group: the weight's last group that has rows, or its first
  __shared__ uint32_t slot_beg[kMaxGroups];
  const uint32_t tid = threadIdx.x;
  int32_t sz = tid < n_groups ? group_sizes[tid] : 0;
  if (sz < 0) sz = 0;
  uint32_t row[1] = {(uint32_t)sz}, rows_of_all[1];
  block_prefix_capped(row, M, rows_of_all);
  const uint32_t r0 = row[0], rows_total = rows_of_all[0];
  const uint32_t r1 = (uint64_t)r0 + (uint32_t)sz > M ? M : r0 + (uint32_t)sz;
  const uint32_t rows = r1 - r0;
  if (tid < n_groups) { row_start[tid] = r0; last_group[tid] = (int)tid; }
  if (tid == 0) row_start[n_groups] = rows_total;
  __syncthreads();
  const uint32_t g0 = tid / gpw * gpw;  // first group of this one's weight
  const bool heads = tid < n_groups && g0 == tid;
  const uint32_t weight_rows = heads ? row_start[tid + gpw] - r0 : 0u;
  const uint32_t n_chunks = (rows + kBwdChunkRows - 1u) / kBwdChunkRows;
  uint32_t place[2] = {(weight_rows + tile_rows - 1u) / tile_rows * tile_rows, n_chunks}, all[2];
  block_prefix_capped(place, 0xffffffffu, all);
  const uint32_t slots_total = all[0], c0 = place[1], chunks_total = all[1];
  if (heads) weight_slot[tid] = place[0];
  if (tid < n_groups && rows) atomicMax(&last_group[g0], (int)tid);
  __syncthreads();
  const uint32_t p0 = tid < n_groups ? weight_slot[g0] + (r0 - row_start[g0]) : 0u;
  if (tid < n_groups) slot_beg[tid] = p0;
  __syncthreads();
  if (part == 0u && tid < n_groups) {
    t.group_beg[tid] = (int)p0;
    t.group_end[tid] = (int)(p0 + rows);
    t.chunk0[tid] = (int)c0;
  }
  if (part == 0u && tid == 0) t.chunk0[n_groups] = (int)chunks_total;
  for (uint32_t c = part; c < n_chunks; c += n_parts) {
    const uint32_t left = rows - c * kBwdChunkRows;
    int32_t* e = t.chunk_tab + 3u * (c0 + c);
    e[0] = (int)tid; e[1] = (int)(p0 + c * kBwdChunkRows); e[2] = (int)(left < kBwdChunkRows ? left : kBwdChunkRows);
  }
  const uint32_t first = part * 1024u + tid, stride = n_parts * 1024u;
  for (uint32_t c = chunks_total + first; c < max_chunks; c += stride) {
    t.chunk_tab[3u * c] = 0; t.chunk_tab[3u * c + 1u] = 0; t.chunk_tab[3u * c + 2u] = 0;
  }
  // The last group whose first slot is not behind p: the one that holds p if p has a row (the groups behind it
  // start behind p), a group of the same weight otherwise.
  auto group_at = [&](uint32_t p) {
    uint32_t lo = 0, hi = n_groups;
    while (hi - lo > 1u) {
      const uint32_t mid = (lo + hi) >> 1;
      if (slot_beg[mid] <= p) lo = mid; else hi = mid;
    }
    return lo;
  };
  for (uint32_t p = first; p < slots; p += stride) {
    int src = -1, grp = 0, range = -1, tile = -1;
    if (p < slots_total) {
      const uint32_t g = group_at(p), w0 = g / gpw * gpw;
      const uint32_t end = weight_slot[w0] + (row_start[w0 + gpw] - row_start[w0]);  // of the weight's rows
      grp = last_group[w0];  // (padding slots name the weight's last group that has rows)
      if (p < end) {
        src = (int)(row_start[g] + (p - slot_beg[g]));
        grp = (int)g;
        // blocks behind the weight's rows stay at -1
        if ((p & 31u) == 0) range = (int)(g | group_at(p + 31u < end ? p + 31u : end - 1u) << 16);
        const uint32_t left = end - p;
        tile = (int)(w0 / gpw | (left < tile_rows ? left : tile_rows) << 16);
      }
    }
    t.src_row[p] = src;
    if (t.x_row) t.x_row[p] = src < 0 ? -1 : (int)mapped_row(t.x_map[src], t.x_div, t.x_rows);
    t.slot_group[p] = grp;
    if ((p & 31u) == 0) t.blk_range[p >> 5] = range;
    if (p % tile_rows == 0) t.tile_weight[p / tile_rows] = tile;  // (a weight's tiles start at its first slot)
  }
  if (dx) {
    const size_t begin = (size_t)rows_total * K, end = (size_t)M * K;
    for (size_t i = begin + first; i < end; i += stride) dx[i] = 0;
  }
}

struct BwdGroupedPrepArgs {
  const int32_t* group_sizes;
  BwdGroupTables tab;
  const uint16_t* lora_a;    // bf16 [n_groups, K, r]
  uint16_t* at;              // bf16 [n_groups, r, K]
  unsigned char* ap;
  const float* sw;           // f32 [n_weights, N]
  float* swp;                // f32 [n_weights][sw_stride] in packed column order
  uint16_t* dx;              // rows beyond the groups are cleared
  uint32_t M, K, N, N_pad, n_groups, gpw, n_weights, r, nkk, kb32, slots, max_chunks, sw_stride;
  uint32_t a_blocks, ap_blocks, sw_blocks_per_weight;
  uint32_t tile_rows;        // slots every weight's rows are padded to: 256 or 128
  uint32_t route_blocks;
};

__global__ __launch_bounds__(1024) void bwd_grouped_prep_kernel(BwdGroupedPrepArgs p) {
  uint32_t b = blockIdx.x;
  if (b < p.route_blocks) {
    route_weight_groups_block(p.group_sizes, p.M, p.n_groups, p.gpw, p.slots, p.max_chunks, p.tab, p.dx, p.K, p.tile_rows,
                              b, p.route_blocks);
    return;
  }
  b -= p.route_blocks;
  if (b < p.a_blocks) {
    lora_a_transpose_item(p.lora_a, p.at, p.n_groups, p.K, p.r, (uint64_t)b * 1024u + threadIdx.x);
    return;
  }
  b -= p.a_blocks;
  if (b < p.ap_blocks) {
    lora_a_operand_item(p.lora_a, p.ap, p.n_groups, p.K, p.r, p.kb32, p.nkk, (uint64_t)b * 1024u + threadIdx.x);
    return;
  }
  b -= p.ap_blocks;
  const uint32_t w = b / p.sw_blocks_per_weight, c = (b % p.sw_blocks_per_weight) * 1024u + threadIdx.x;
  if (w < p.n_weights && c < p.N_pad) {
    const uint32_t n = packed_to_orig_col(c);
    p.swp[(size_t)w * p.sw_stride + c] = n < p.N ? p.sw[(size_t)w * p.N + n] : 0.0f;
  }
}

// ---------------------------------------------------------------------------------------
// dx = dyp @ bf16(W * sw).T (+ rs @ A.T), one bf16 cast, on tiles of 256 rows x 256 k (bwd_dx_wide_kernel: dense calls, and grouped ones whose weights
// own many rows) or of 128 rows x 512 k (bwd_dx_kernel: grouped calls whose weights own few).
// The contraction runs over n in stages of one 32-wide n block.  A stage's dy panel, weight blocks (24 KiB together) and scales travel
// HBM/L2 -> LDS with direct-to-LDS loads four or five stages ahead.  While the matrix core works on stage
// nb, the vector ALU prepares the weight operands of stage nb + 1: each wave transposes its two
// blocks with the identity MFMA, scales, rounds to bf16 and keeps them in registers.
// ---------------------------------------------------------------------------------------
constexpr int kBwdStages = 6;
constexpr int kBwdStagePanel = 16384;      // dy: 8 row blocks x 2 halves
constexpr int kBwdStageWeight = 8192;      // 8 k blocks of the n block
constexpr int kBwdStageBytes = kBwdStagePanel + kBwdStageWeight + 1024;  // + a 1 KiB chunk of scales (the stage's 32 lead it)
constexpr int kBwdLdsBytes = kBwdStages * kBwdStageBytes;
constexpr int kBwdScalePad = 256;     // floats readable past the last stage's scales

struct BwdDxArgs {
  const unsigned char* dyp;   // packed dy
  const unsigned char* wp;    // packed weight
  const float* swp;           // scales in packed column order [N_pad + 32]
  const unsigned char* rp;    // packed rs fragments [slots/32][NKK][3][64][8] or null
  const unsigned char* ap;    // packed A operands or null
  const int32_t* src_row; const int32_t* slot_group; const int32_t* blk_range;
  uint16_t* dx;               // bf16 [M, K]
  uint32_t M, K, KB, NB, tiles_m, tiles_k;
  // grouped calls: weight | rows << 16 of every 256-slot tile (-1: tile without rows; the rows fill the
  // tile from its first slot), the bytes between two packed weights and the floats between two scale
  // tables; null / 0 for one weight
  const int32_t* tile_weight;
  size_t w_stride;
  uint32_t sw_stride;
  // dense calls: the tiles from direct_tiles on are split (bwd_dx_split): sk_wgs workgroups take sk_q
  // consecutive stages each of their joint stage sequence and leave float32 partial tiles in part
  uint32_t direct_tiles, sk_q, sk_wgs;
  // [slot w + u of workgroup w's stages of split tile u][part_blocks row blocks][4 wave columns][k blocks of a wave][4][64 lanes][4]
  float* part;
  uint32_t part_blocks;  // 8, or the blocks that hold rows when there is one row tile
};
constexpr uint32_t kBwdPartBlockFloats = 4096;  // of a row block of a slot, per k block of a wave

// Where a wave keeps its block of a partial tile (CBN k blocks); row_block: of the tile's eight.
template <int CBN>
__device__ inline float4* bwd_dx_part(const BwdDxArgs& g, uint32_t slot, uint32_t row_block, uint32_t wcol) {
  return reinterpret_cast<float4*>(g.part) + ((size_t)(slot * g.part_blocks + row_block) * 4u + wcol) * (256u * CBN) + (threadIdx.x & 63u);
}

// (row tile, k tile) of position t in the band-major tile order: 4 row tiles x all k tiles to a band
__device__ inline void bwd_dx_tile_at(const BwdDxArgs& g, uint32_t t, uint32_t& tm, uint32_t& tk) {
  const uint32_t band_tiles = 4u * g.tiles_k, band = t / band_tiles, in_band = t - band * band_tiles;
  const uint32_t band_rows = (g.tiles_m - band * 4u) < 4u ? (g.tiles_m - band * 4u) : 4u;
  tm = band * 4u + in_band % band_rows;
  tk = in_band / band_rows;
}

// A wave's ROWS row blocks of dx, of CBN k blocks each: + rs @ A.T, one cast, rows back to their original positions.
// pbase: first slot; kbw: first k block; live: row blocks that hold rows; sums(rb, cb): the sums of a block; turn: 32 rows of
// kBwdTurnStride bytes of the LDS that are the wave's own.
// A block's values are turned in the LDS so that eight lanes store a row's 128 bytes: from the accumulator layout a row went
// out two bytes a lane, 32 stores a block instead of 4.  rs_lds: where in the LDS the operands of rs of the row blocks lie, one
// behind the other (bwd_dx_fetch_rs, whose loads all waves of a tile share and wait for once), or 0: in memory.
// With 2-byte stores and every block waiting for its own operands a whole 256 x 256 tile's epilogue took 39 us (rank 32), now 15.
constexpr uint32_t kBwdTurnStride = 144;  // bytes of a row: 64 values and 16 more, so that rows start on different banks
constexpr uint32_t kBwdTurnBytes = 32u * kBwdTurnStride;
template <int NKK, int CBN, int ROWS, bool RS_LDS, class Sums>
__device__ inline __attribute__((always_inline)) void bwd_dx_store(const BwdDxArgs& g, uint32_t pbase, uint32_t kbw, int live, uint32_t turn, uint32_t rs_lds, Sums&& sums) {
  typedef __attribute__((address_space(3))) uint16_t* lds_u16;
  typedef __attribute__((address_space(3))) const v4i* lds_cv4;
  constexpr int kKK = NKK > 0 ? NKK : 1;
  int lane = threadIdx.x & 63;
  // (opaque: what the epilogue derives from it is formed here and not held in registers through the stages)
  asm volatile("" : "+v"(lane));
  const int c = lane & 31, h = lane >> 5;
  int src[ROWS];  // original row of slot c of every block
#pragma unroll
  for (int rb = 0; rb < ROWS; ++rb) {
    const uint32_t p = pbase + 32u * (uint32_t)(rb < live ? rb : 0) + (uint32_t)c;
    src[rb] = g.src_row ? g.src_row[p] : (int)p;
  }
  v8us ab[CBN][kKK];
  auto operand_r = [&](int rb, int chunk) -> v8bf {
    if constexpr (RS_LDS) return __builtin_bit_cast(v8bf, *reinterpret_cast<lds_cv4>((uintptr_t)(rs_lds + (uint32_t)(rb * kKK * 3 + chunk) * kBlockBytes + (uint32_t)lane * 16u)));
    return __builtin_bit_cast(v8bf, *reinterpret_cast<const v8us*>(g.rp + ((size_t)(pbase / 32u + (uint32_t)rb) * (uint32_t)(kKK * 3) + (uint32_t)chunk) * kBlockBytes + lane * 16));
  };
  int held = -1;  // group whose A operands are in ab
  auto fetch_a = [&](int gi) {
#pragma unroll
    for (int cb = 0; cb < CBN; ++cb) {
      const uint32_t kb = kbw + (uint32_t)cb < g.KB ? kbw + (uint32_t)cb : g.KB - 1u;
      const unsigned char* a0 = g.ap + ((size_t)gi * g.KB + kb) * (uint32_t)kKK * kBlockBytes + lane * 16;
#pragma unroll
      for (int kk = 0; kk < kKK; ++kk) ab[cb][kk] = *reinterpret_cast<const v8us*>(a0 + kk * kBlockBytes);
    }
    held = gi;
  };
#pragma unroll
  for (int rb = 0; rb < ROWS; ++rb) {
    if (rb >= live) break;  // wave-uniform
    const uint32_t blk = pbase / 32u + (uint32_t)rb;
    const bool row_ok = src[rb] >= 0 && src[rb] < (int)g.M;
    if (__builtin_amdgcn_ballot_w64(row_ok) == 0) continue;  // wave-uniform: no row of this block exists
    const uint32_t range = (NKK > 0 && g.blk_range) ? (uint32_t)g.blk_range[blk] : 0u;
    const int glo = (int)(range & 0xffffu), ghi = (int)(range >> 16);
    const int grp = (NKK > 0 && g.slot_group && ghi > glo) ? g.slot_group[blk * 32u + (uint32_t)c] : glo;
    for (int gi = glo; gi <= ghi; ++gi) {  // a block at a group boundary runs once per group
      if (NKK > 0 && gi != held) fetch_a(gi);  // wave-uniform
#pragma unroll
      for (int cb = 0; cb < CBN; ++cb) {
        v16f y = sums(rb, cb);
        if constexpr (NKK > 0) {
          v16f low;
#pragma unroll
          for (int e = 0; e < 16; ++e) low[e] = 0.0f;
#pragma unroll
          for (int kk = 0; kk < NKK; ++kk)
#pragma unroll
            for (int t3 = 2; t3 >= 0; --t3)
              low = __builtin_amdgcn_mfma_f32_32x32x16_bf16(operand_r(rb, kk * 3 + t3), __builtin_bit_cast(v8bf, ab[cb][kk]), low, 0, 0, 0);
          asm volatile("" : "+v"(low));
#pragma unroll
          for (int e = 0; e < 16; ++e) y[e] = y[e] + low[e];
        }
#pragma unroll
        for (int v = 0; v < 16; ++v)
          *reinterpret_cast<lds_u16>((uintptr_t)(turn + (uint32_t)(8 * (v >> 2) + 4 * h + (v & 3)) * kBwdTurnStride + (uint32_t)(cb * 64 + 2 * c))) =
              (uint16_t)f32_to_bf16_bits(y[v]);
      }
      // (a wave's LDS operations are in order, so the reads find the writes and the next block's writes come behind them)
      constexpr int kPieces = 4 * CBN;  // of 16 bytes of a row
#pragma unroll
      for (int t = 0; t < kPieces / 2; ++t) {
        const int row = lane / kPieces + (64 / kPieces) * t, piece = lane % kPieces;
        const v4i v = *reinterpret_cast<lds_cv4>((uintptr_t)(turn + (uint32_t)row * kBwdTurnStride + (uint32_t)piece * 16u));
        const int m = __builtin_amdgcn_ds_bpermute(4 * row, src[rb]);
        int row_grp = gi;
        if (NKK > 0 && ghi > glo) row_grp = __builtin_amdgcn_ds_bpermute(4 * row, grp);
        const uint32_t k = kbw * 32u + 8u * (uint32_t)piece;  // (K is a multiple of 8)
        if (m >= 0 && m < (int)g.M && k < g.K && row_grp == gi) *reinterpret_cast<v4i*>(g.dx + (uint32_t)m * g.K + k) = v;
      }
    }
  }
}

// The operands of rs of a tile's row blocks into the LDS, by all its waves; waits for them.  Everybody is done with what lay there.
template <int NKK>
__device__ inline void bwd_dx_fetch_rs(const BwdDxArgs& g, uint32_t pbase, int blocks, uint32_t rs_lds, int wave, int waves) {
  if constexpr (NKK > 0) {
    const unsigned char* src = g.rp + (size_t)(pbase / 32u) * (uint32_t)(NKK * 3) * kBlockBytes;
    for (int ch = wave; ch < blocks * NKK * 3; ch += waves)
      lds_load_1k(src + (size_t)ch * kBlockBytes, (threadIdx.x & 63u) * 16u, rs_lds + (uint32_t)ch * kBlockBytes);
    wait_vmcnt<0>();
    lds_barrier();
  }
}

// The tiles and split stages of this workgroup in order: work(tile, first stage, stages, slot).
template <class Work>
__device__ inline __attribute__((always_inline)) void bwd_dx_schedule(const BwdDxArgs& g, bool may_split, Work&& work) {
  const uint32_t ntile = g.direct_tiles;
  const uint32_t wgs_per_xcd = gridDim.x >> 3, xcd = blockIdx.x & 7u;
  // band-major tile order, so an XCD's workgroups share panels.  One weight:
  // every XCD walks a contiguous range of bands.  Grouped calls: the bands are dealt round-robin to the
  // XCDs, because the slots in use end before the last bands and a contiguous split would leave the
  // last XCDs without work.
  const uint32_t band_tiles = 4u * g.tiles_k, n_bands = (g.tiles_m + 3u) / 4u;
  const uint32_t per_xcd = g.tile_weight ? ((n_bands + 7u) / 8u) * band_tiles : (ntile + 7u) / 8u;
  uint32_t ti = blockIdx.x >> 3;
  // behind the whole tiles: this workgroup's stages of the split tiles' joint sequence (an XCD's workgroups are
  // neighbours)
  const uint32_t sw8 = g.sk_wgs >> 3, sk_w = xcd * sw8 + (blockIdx.x >> 3);
  uint32_t s0 = 0, s1 = 0;
  if (may_split && (blockIdx.x >> 3) < sw8) {
    const uint32_t total = (g.tiles_m * g.tiles_k - ntile) * g.NB;
    s0 = sk_w * g.sk_q < total ? sk_w * g.sk_q : total;
    s1 = s0 + g.sk_q < total ? s0 + g.sk_q : total;
  }
#pragma unroll 1
  for (;;) {
    uint32_t t, nb0 = 0, len = g.NB, slot = 0;
    if (ti < per_xcd) {
      const uint32_t pos = ti;
      ti += wgs_per_xcd;
      if (g.tile_weight) {
        const uint32_t band = xcd + 8u * (pos / band_tiles), in_band = pos % band_tiles;
        if (band >= n_bands) { ti = per_xcd; continue; }
        const uint32_t band_rows = (g.tiles_m - band * 4u) < 4u ? (g.tiles_m - band * 4u) : 4u;
        if (in_band >= band_rows * g.tiles_k) continue;  // a last band with fewer than 4 row tiles
        t = band * band_tiles + in_band;
      } else {
        t = xcd * per_xcd + pos;
        if (t >= ntile) { ti = per_xcd; continue; }
      }
    } else if (s0 < s1) {
      const uint32_t u = s0 / g.NB;
      nb0 = s0 - u * g.NB;
      len = s1 - s0 < g.NB - nb0 ? s1 - s0 : g.NB - nb0;
      t = ntile + u;
      slot = sk_w + u;
      s0 += len;
    } else {
      break;
    }
    work(t, (int)nb0, (int)len, slot);
  }
}

// The operands of v_mfma_f32_16x16x32_bf16 from blocks packed for 32x32x16.  Lane (column c, half h) of a transposed weight
// block holds the chunks q = 0 (lo) and 1 (hi) of its column; the operand of 16 columns wants the chunks of a column in its four
// rows of lanes, (q, h) = (row % 2, row / 2): one swap leaves that of columns 0..15 in lo and of 16..31 in hi.
__device__ inline void bwd_operand_rows(uint32_t& lo, uint32_t& hi) {
  const auto s = __builtin_amdgcn_permlane16_swap(lo, hi, false, false);
  lo = s[0]; hi = s[1];
}
// ... and where the lane finds its part of dy's rows 0..15 in the two 1 KiB chunks of a row block (rows 16..31: 256 bytes on)
__device__ inline uint32_t bwd_frag_offset(uint32_t lane) {
  return ((lane >> 4) & 1u) * (uint32_t)kBlockBytes + (lane >> 5) * 512u + (lane & 15u) * 16u;
}
// row block p of 16 of the panel
__device__ inline v8bf bwd_panel_frag(uint32_t panel, int p) {
  typedef __attribute__((address_space(3))) const v4i* lds_v4ptr;
  return __builtin_bit_cast(v8bf, *reinterpret_cast<lds_v4ptr>((uintptr_t)(panel + (uint32_t)((p >> 1) * 2048 + (p & 1) * 256))));
}
// Four 16 x 16 blocks, [row half][column half], as the 32 x 32 block that the epilogue and the partial tiles know: a lane's
// rows 4 (lane / 16) + i of a half become rows 8 j + 4 (lane / 32) + i, the column's bit 4 the lane's.
__device__ inline v16f bwd_block32(const v4f (&b)[2][2]) {
  v16f y;
#pragma unroll
  for (int rh = 0; rh < 2; ++rh)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const auto s = __builtin_amdgcn_permlane16_swap(__float_as_uint(b[rh][0][i]), __float_as_uint(b[rh][1][i]), false, false);
      const auto t = __builtin_amdgcn_permlane32_swap(s[0], s[1], false, false);
      y[8 * rh + i] = __uint_as_float(t[0]);
      y[8 * rh + 4 + i] = __uint_as_float(t[1]);
    }
  return y;
}

// The 128 x 512 geometry: eight waves side by side along k, a wave tile of 128 rows x 64 k (8 x 4 accumulator blocks of
// v_mfma_f32_16x16x32_bf16).  A stage holds half the dy panel of the 256 x 256 tile and twice the weight blocks, the same
// bytes.  For grouped calls whose weights own few rows each: half the padding per weight, and every wave has rows.
//
// Bound by HBM (the weights are read once) and by what stands in line behind it in a stage.  The 256 registers that two waves
// per SIMD leave are the kernel's limit: the loads' addresses are a scalar base plus the lane's offset (issue), and the epilogue
// derives its lane constants for itself (bwd_dx_store).  1021 tokens to 8 of 128 experts, 2048 <- 1536 and 768 <- 2048 (600 MB of
// weights): 197 us together with the row blocks skipped by a branch each, behind which the compiler read every fragment at its
// use, and the loads' addresses formed anew for every stage; one loop for each number of row blocks 174.
constexpr int kBwdPanel128 = 8192, kBwdWeight512 = 16384;  // 4 row blocks x 2 halves; 16 k blocks
static_assert(kBwdPanel128 + kBwdWeight512 + 1024 == kBwdStageBytes, "a stage keeps its size in both geometries");
constexpr int kBwdAhead = kBwdStages - 1;  // stages between a load and its use
constexpr int kBwdLoadsPerStage = 4;       // direct-to-LDS loads per wave and stage: a panel chunk, 2 weight blocks, scales
template <int NKK>
__global__ __launch_bounds__(512, 1) void bwd_dx_kernel(BwdDxArgs g) {
  extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 31, h = lane >> 5;
  const uint32_t lane16 = (uint32_t)lane * 16u, lds_base = (uint32_t)(uintptr_t)(lptr_t)lds;

  // identity operand of the transposing MFMA: lane (column c, k half h) holds byte 1 at k == c
  v4i ident = {0, 0, 0, 0};
  {
    const int word = ((c >> 4) == h) ? (int)(1u << (8 * (c & 3))) : 0;
    const int wi = (c & 15) >> 2;
    ident[0] = wi == 0 ? word : 0; ident[1] = wi == 1 ? word : 0;
    ident[2] = wi == 2 ? word : 0; ident[3] = wi == 3 ? word : 0;
  }

  // ROWS: the tile's 32-row blocks that hold rows; the others are not multiplied
  auto tile = [&](auto rows_tag, uint32_t tm, uint32_t tk, int tw) {
    constexpr int ROWS = decltype(rows_tag)::value, kRows16 = 2 * ROWS;
    const int L = (int)g.NB;  // (even)
    // row block of whose dy panel this wave fetches a half.  A block without rows is never multiplied: its slot is filled from block 0
    // of the tile, which is in the caches anyway, instead of streaming unused memory (the load count stays the same)
    const uint32_t load_rb = (wave >> 1) < ROWS ? (uint32_t)wave >> 1 : 0u;
    const unsigned char* const Ag = g.dyp + ((size_t)(tm * 4u + load_rb) * g.NB) * 2048u + (wave & 1) * 1024;
    const uint32_t kbw = tk * 16u + (uint32_t)wave * 2u;  // its two k blocks (blocks past the weight repeat the last)
    const size_t nb_stride = (size_t)g.KB * kBlockBytes;
    const unsigned char* Bg0 = g.wp + (size_t)tw * g.w_stride + (size_t)(kbw < g.KB ? kbw : g.KB - 1u) * kBlockBytes;
    const unsigned char* Bg1 = kbw + 1u < g.KB ? Bg0 : Bg0 - kBlockBytes;  // (lds_load_2k: 1 KiB further)
    const unsigned char* const swp_t = reinterpret_cast<const unsigned char*>(g.swp + (size_t)tw * g.sw_stride);
    uint32_t a_off = lane16, s_off = lane16;
    auto issue = [&](uint32_t st) {  // the next stage's loads, into the stage buffer at st
      lds_load_1k(Ag, a_off, st + (uint32_t)wave * kBlockBytes);
      // (few rows per weight: most of its bytes are read by one workgroup only)
      lds_load_2k<true>(Bg0, Bg1, lane16, st + kBwdPanel128 + (uint32_t)wave * 2048u);
      // every wave fetches the same 1 KiB of scales (the stage's 32 lead it) to the same place
      lds_load_1k(swp_t, s_off, st + kBwdPanel128 + kBwdWeight512);
      a_off += 2048u;
      s_off += 128u;
      Bg0 += nb_stride;
      Bg1 += nb_stride;
    };

    v4f acc[kRows16][4];
#pragma unroll
    for (int i = 0; i < kRows16; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[i][j][e] = 0.0f;

    typedef __attribute__((address_space(3))) const v4i* lds_v4ptr;
    const uint32_t frag_off = bwd_frag_offset((uint32_t)lane), weight_off = (uint32_t)wave * 2048u + lane16, scale_off = 16u * (uint32_t)h;
    struct NextRegs { v4i raw[2]; v4f s4[4]; };
    auto next_read = [&](uint32_t st, NextRegs& r) {  // the wave's weight blocks and the scales of the stage at st
      uint32_t wa = st + weight_off, sa = st + scale_off;
      asm volatile("" : "+v"(wa), "+v"(sa));  // (opaque: constants are the instructions')
#pragma unroll
      for (int b = 0; b < 2; ++b) r.raw[b] = *reinterpret_cast<lds_v4ptr>((uintptr_t)(wa + kBwdPanel128 + b * kBlockBytes));
#pragma unroll
      for (int q = 0; q < 4; ++q)
        r.s4[q] = __builtin_bit_cast(v4f, *reinterpret_cast<lds_v4ptr>((uintptr_t)(sa + kBwdPanel128 + kBwdWeight512 + 32 * q)));
    };
    auto transpose_block = [&](const v4i& rawb) -> v16i {
      v16i z16;
#pragma unroll
      for (int e = 0; e < 16; ++e) z16[e] = 0;
      return __builtin_amdgcn_mfma_i32_32x32x32_i8(rawb, ident, z16, 0, 0, 0);
    };
    // rows 8 (t / 2) + 4 h + 2 (t % 2) + 0, 1 of a transposed block: bf16(float(code) * scale), the per-element
    // weight of the reference's pull-back
    auto convert2 = [&](const v16i& tr, const v4f (&s4)[4], int t, uint32_t (&pk)[8]) {
      const float f0 = (float)tr[2 * t] * s4[t >> 1][2 * (t & 1)], f1 = (float)tr[2 * t + 1] * s4[t >> 1][2 * (t & 1) + 1];
      pk[t] = pack_bf16x2(f0, f1);
    };
    auto to_operands = [&](uint32_t (&pk)[8], v8bf (&bq)[2]) {
#pragma unroll
      for (int t = 0; t < 4; ++t) bwd_operand_rows(pk[t], pk[4 + t]);
      bq[0] = __builtin_bit_cast(v8bf, v4i{(int)pk[0], (int)pk[1], (int)pk[2], (int)pk[3]});
      bq[1] = __builtin_bit_cast(v8bf, v4i{(int)pk[4], (int)pk[5], (int)pk[6], (int)pk[7]});
    };
    auto panel_at = [&](uint32_t st) -> uint32_t {
      uint32_t at = st + frag_off;
      asm volatile("" : "+v"(at));
      return at;
    };

    // One stage, at st: its MFMAs against the dy panel in the LDS; between them the operands of the stage at st_next are
    // prepared, a block of the two in each half of the row blocks.  af: the first row block's fragment; leaves the next stage's.
    auto stage = [&](uint32_t st, uint32_t st_next, const v8bf (&bqC)[2][2], v8bf (&bqN)[2][2], v8bf& af) {
      NextRegs nx;
      v16i tr;
      uint32_t pk[8];
      const uint32_t panel = panel_at(st), panel_next = panel_at(st_next);
      next_read(st_next, nx);
#pragma unroll
      for (int p = 0; p < kRows16; ++p) {
        const v8bf af_next = p + 1 < kRows16 ? bwd_panel_frag(panel, p + 1) : bwd_panel_frag(panel_next, 0);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < 4; ++j)
          acc[p][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af, bqC[j >> 1][j & 1], acc[p][j], 0, 0, 0);
        const int b = p / ROWS, at = p % ROWS;  // weight block, place in its half
        if (at == 0) tr = transpose_block(nx.raw[b]);
        constexpr int kParts = ROWS > 1 ? ROWS - 1 : 1;
        if (ROWS == 1 || at > 0) {
          const int part = ROWS > 1 ? at - 1 : 0;
#pragma unroll
          for (int t = 8 * part / kParts; t < 8 * (part + 1) / kParts; ++t) convert2(tr, nx.s4, t, pk);
          if (part == kParts - 1) to_operands(pk, bqN[b]);
        }
        __builtin_amdgcn_sched_barrier(0);
        af = af_next;
      }
    };

    v8bf bqA[2][2], bqB[2][2], af;
    wait_vmcnt<0>();  // stores of the previous tile
    lds_barrier();
#pragma unroll
    for (int i = 0; i < kBwdAhead; ++i)
      if (i < L) issue(lds_base + (uint32_t)i * kBwdStageBytes);
    if (L >= kBwdAhead) wait_vmcnt<(kBwdAhead - 1) * kBwdLoadsPerStage>();  // stage 0 has landed
    else wait_vmcnt<0>();
    lds_barrier();
    {  // operands of stage 0
      NextRegs nx;
      next_read(lds_base, nx);
      uint32_t pk[8];
#pragma unroll
      for (int cb = 0; cb < 2; ++cb) {
        const v16i tr = transpose_block(nx.raw[cb]);
#pragma unroll
        for (int t = 0; t < 8; ++t) convert2(tr, nx.s4, t, pk);
        to_operands(pk, bqA[cb]);
      }
    }
    af = bwd_panel_frag(panel_at(lds_base), 0);
    uint32_t st = lds_base;  // of stage i; the loads go into the buffer in front of it
    // stages i and i + 1 have landed, i + 2 .. i + 4 are on their way and i + 5 is asked for.  (Behind the last stage nothing reads
    // the operands that are prepared.)
    auto step = [&](int i, const v8bf (&bqC)[2][2], v8bf (&bqN)[2][2]) {
      const uint32_t last = lds_base + (uint32_t)(kBwdStages - 1) * kBwdStageBytes;
      const uint32_t st_next = st == last ? lds_base : st + kBwdStageBytes, st_load = st == lds_base ? last : st - kBwdStageBytes;
      if (i + kBwdAhead < L) {
        wait_vmcnt<(kBwdAhead - 2) * kBwdLoadsPerStage>();
        lds_barrier();
        issue(st_load);
      } else {  // fewer loads in flight than that count assumes
        wait_vmcnt<0>();
        lds_barrier();
      }
      __builtin_amdgcn_sched_barrier(0);
      stage(st, st_next, bqC, bqN, af);
      st = st_next;
    };
#pragma unroll 1
    for (int i = 0; i < L; i += 2) {
      step(i, bqA, bqB);
      step(i + 1, bqB, bqA);
    }

    lds_barrier();  // (every wave has read its last stage)
    const uint32_t rs_lds = lds_base + 8u * kBwdTurnBytes;
    bwd_dx_fetch_rs<NKK>(g, tm * 128u, ROWS, rs_lds, wave, 8);
    bwd_dx_store<NKK, 2, ROWS, true>(g, tm * 128u, kbw, ROWS, lds_base + (uint32_t)wave * kBwdTurnBytes, rs_lds,
                                     [&](int rb, int cb) -> v16f {
      const v4f b[2][2] = {{acc[2 * rb][2 * cb], acc[2 * rb][2 * cb + 1]}, {acc[2 * rb + 1][2 * cb], acc[2 * rb + 1][2 * cb + 1]}};
      return bwd_block32(b);
    });
  };

  bwd_dx_schedule(g, false, [&](uint32_t t, int, int, uint32_t) {
    uint32_t tm, tk;
    bwd_dx_tile_at(g, t, tm, tk);
    const int tv = g.tile_weight[tm];
    if (tv < 0) return;  // workgroup-uniform: no row lives in this tile
    const int tw = tv & 0xffff, blocks = __builtin_amdgcn_readfirstlane(((tv >> 16) + 31) / 32);
    if (blocks <= 1) tile(std::integral_constant<int, 1>{}, tm, tk, tw);
    else if (blocks == 2) tile(std::integral_constant<int, 2>{}, tm, tk, tw);
    else if (blocks == 3) tile(std::integral_constant<int, 3>{}, tm, tk, tw);
    else tile(std::integral_constant<int, 4>{}, tm, tk, tw);
  });
}

// The 256 x 256 geometry: four waves, one to a SIMD, side by side along k: a wave tile of 256 rows x 64 k (16 x 4 accumulator
// blocks, 256 registers, beside 256 others).  No two waves then convert the same weight blocks, which as eight waves of
// 128 x 64 every two did: 2 transposing MFMAs and 88 vector instructions for 64 MFMAs instead of 32.  What a
// second wave per SIMD hid is hidden by order: the conversion of the next stage's blocks stands between single MFMAs, the dy
// fragments are read three row blocks ahead, also across the barrier, which comes every two stages.
// ROWS: row blocks of 32 multiplied (8, or 4 where the tile holds no more: the others' dy is loaded from block 0 and left alone).
// Power bounds it (all-zero dy runs a quarter faster), and the one wave's issue slots: 128 MFMAs hold the matrix core for 2048
// clocks, 512 slots.  v_mfma_f32_16x16x32_bf16 carries half the sums per product of 32x32x16: from registers alone
// 2045 TFLOP/s against 1750 to 1790.  An MLP's two pull-backs, 3003 rows, 4096 <- 24576 and 12288 <- 4096: 837 us with 32x32x16
// and 464 instructions to two stages (the weight's reads waited for where they stood), 789 now (1.15 PFLOP/s; 472).  With
// 16x16x32 but 549 instructions it was 2 % slower than before.  2048 x 2560, N = 10240, rank 64: 110 / 107.
constexpr int kBwdWideLoads = 7;  // direct-to-LDS loads per wave and stage: 4 panel chunks, 2 weight blocks, scales

// The accumulator tied, as one read-write operand, in the half of the register file that is named: left to the compiler, or all
// in one half, up to a half of the sixteen sets was moved between the halves at every pass of the loop (540 moves for 64 MFMAs).
// The compiler does not see that an MFMA writes the sums: they are next touched by the MFMA of the other half block or
// of the next stage, and the epilogue stands behind explicit wait states.
template <bool HIGH>
__device__ inline void bwd_mfma(v4f& acc, const v8bf& a, const v8bf& b) {
  if constexpr (HIGH) asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc) : "v"(a), "v"(b));
  else asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+v"(acc) : "v"(a), "v"(b));
}
// The sums for the vector ALU.  (As plain values their uses behind the loop drew the sums into the other half within it.)
template <bool HIGH>
__device__ inline v4f bwd_sums(v4f& acc) {
  v4f y;
  if constexpr (HIGH) {
#pragma unroll
    for (int e = 0; e < 4; ++e) asm volatile("v_accvgpr_read_b32 %0, %1" : "=v"(y[e]) : "a"(acc[e]));
  } else {
    asm volatile("" : "+v"(acc));  // (behind the wait states, too)
    y = acc;
  }
  return y;
}
// W[n][k] of a 32 x 32 block in vector registers (the builtin's result lands in the half that the sums fill); not to be read for
// 13 wait states (what the compiler leaves behind the builtin; the calls here leave three MFMAs or 32 of s_nop).
__device__ inline void bwd_transpose(v16i& tr, const v4i& raw, const v4i& ident) {
  asm volatile("v_mfma_i32_32x32x32_i8 %0, %1, %2, 0" : "=&v"(tr) : "v"(raw), "v"(ident));
}

template <int NKK>
__global__ __launch_bounds__(256, 1) void bwd_dx_wide_kernel(BwdDxArgs g) {
  extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 31, h = lane >> 5;
  v4i ident = {0, 0, 0, 0};  // identity operand of the transposing MFMA: lane (column c, k half h) holds byte 1 at k == c
  {
    const int word = ((c >> 4) == h) ? (int)(1u << (8 * (c & 3))) : 0;
    const int wi = (c & 15) >> 2;
    ident[0] = wi == 0 ? word : 0; ident[1] = wi == 1 ? word : 0;
    ident[2] = wi == 2 ? word : 0; ident[3] = wi == 3 ? word : 0;
  }
  const uint32_t lds_base = (uint32_t)(uintptr_t)(lptr_t)lds;

  // stages nb0 .. nb0 + L - 1 (an even number) of a tile: all of them (whole), or partial sums for slot `slot`
  auto segment = [&](auto rows_tag, uint32_t tm, uint32_t tk, int live_blocks, int tw, int nb0, int L, bool whole, uint32_t slot) {
    constexpr int ROWS = decltype(rows_tag)::value;
    // (opaque: the addresses derived from it are formed per segment.  Formed once for the kernel they were spilled, and a
    // reload in front of the loop has the compiler drain every load at its first use in it)
    int lane_s = lane;
    asm volatile("" : "+v"(lane_s));
    const uint32_t lane16 = (uint32_t)lane_s * 16u, h16 = (uint32_t)(lane_s >> 5) * 16u;
    // this wave's loads of a stage: dy of two row blocks (both halves), two weight blocks
    const uint32_t rb0 = 2u * (uint32_t)wave < (uint32_t)live_blocks ? 2u * (uint32_t)wave : 0u;
    const uint32_t rb1 = 2u * (uint32_t)wave + 1u < (uint32_t)live_blocks ? 2u * (uint32_t)wave + 1u : 0u;
    const unsigned char* const Ag0 = g.dyp + ((size_t)(tm * 8u + rb0) * g.NB + (uint32_t)nb0) * 2048u;
    const unsigned char* const Ag1 = g.dyp + ((size_t)(tm * 8u + rb1) * g.NB + (uint32_t)nb0) * 2048u;
    const uint32_t kbw = tk * 8u + 2u * (uint32_t)wave;  // its two k blocks (blocks past the weight repeat the last)
    const size_t nb_stride = (size_t)g.KB * kBlockBytes;
    const unsigned char* Bg0 = g.wp + (size_t)tw * g.w_stride + (size_t)nb0 * nb_stride + (size_t)(kbw < g.KB ? kbw : g.KB - 1u) * kBlockBytes;
    const unsigned char* Bg1 = kbw + 1u < g.KB ? Bg0 : Bg0 - kBlockBytes;  // (lds_load_2k: 1 KiB further)
    const unsigned char* const swp_t = reinterpret_cast<const unsigned char*>(g.swp + (size_t)tw * g.sw_stride + 32 * nb0);
    uint32_t a_off = lane16, s_off = lane16;
    int stages_left = L - 1;
    // Part j of four of the loads of the next stage to be asked for, into the stage buffer at st (behind the last stage: of that
    // one again).  Loads the compiler keeps no books on: it would drain them before every read of the LDS.  The addresses go
    // on from stage to stage: a loop of 128 MFMAs leaves 400 issue slots for all else, and formed anew they took 100.
    auto issue = [&](uint32_t st, int j) {
      if (j == 0) lds_load_2k(Ag0, a_off, st + (uint32_t)wave * 4096u);
      else if (j == 1) lds_load_2k(Ag1, a_off, st + (uint32_t)wave * 4096u + 2048u);
      else if (j == 2) lds_load_2k<false>(Bg0, Bg1, lane16, st + kBwdStagePanel + (uint32_t)wave * 2048u);
      else {
        lds_load_1k(swp_t, s_off, st + kBwdStagePanel + kBwdStageWeight);
        const bool more = stages_left > 0;
        --stages_left;
        a_off += more ? 2048u : 0u;
        s_off += more ? 128u : 0u;
        Bg0 += more ? nb_stride : 0;
        Bg1 += more ? nb_stride : 0;
      }
    };
    constexpr int kRows16 = 2 * ROWS;  // row blocks of 16
    v4f acc[kRows16][4];
#pragma unroll
    for (int i = 0; i < kRows16; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[i][j][e] = 0.0f;

    struct NextRegs { v4i raw[2]; v4f s4[4]; };
    const uint32_t weight_off = (uint32_t)wave * 2048u + lane16;
    // The weight blocks and scales of the stage at st, in three parts.  (Reads that the compiler waits for where they are used.)
    auto next_read = [&](uint32_t st, int part, NextRegs& r) {
      typedef __attribute__((address_space(3))) const v4i* lds_v4ptr;
      if (part == 0) {
        uint32_t wa = st + weight_off;
        asm volatile("" : "+v"(wa));
        r.raw[0] = *reinterpret_cast<lds_v4ptr>((uintptr_t)(wa + kBwdStagePanel));
        r.raw[1] = *reinterpret_cast<lds_v4ptr>((uintptr_t)(wa + kBwdStagePanel + kBlockBytes));
      } else {
        uint32_t sa = st + h16;
        asm volatile("" : "+v"(sa));
#pragma unroll
        for (int q = 0; q < 2; ++q)
          r.s4[2 * part - 2 + q] = __builtin_bit_cast(v4f, *reinterpret_cast<lds_v4ptr>((uintptr_t)(sa + kBwdStagePanel + kBwdStageWeight + 32 * (2 * part - 2 + q))));
      }
    };
    // rows 8 (t / 2) + 4 h + 2 (t % 2) + 0, 1 of a transposed block: bf16(float(code) * scale), the per-element
    // weight of the reference's pull-back
    auto convert_first = [&](const v16i& tr, int t, float (&f)[2]) { f[0] = (float)tr[2 * t]; f[1] = (float)tr[2 * t + 1]; };
    auto convert_second = [&](const v4f (&s4)[4], int t, const float (&f)[2], uint32_t (&pk)[8]) {
      pk[t] = pack_bf16x2(f[0] * s4[t >> 1][2 * (t & 1)], f[1] * s4[t >> 1][2 * (t & 1) + 1]);
    };
    auto to_operands = [&](const uint32_t (&pk)[8], v8bf (&bq)[2]) {
      bq[0] = __builtin_bit_cast(v8bf, v4i{(int)pk[0], (int)pk[1], (int)pk[2], (int)pk[3]});
      bq[1] = __builtin_bit_cast(v8bf, v4i{(int)pk[4], (int)pk[5], (int)pk[6], (int)pk[7]});
    };
    const uint32_t frag_off = bwd_frag_offset((uint32_t)lane_s);
    auto panel_at = [&](uint32_t st) -> uint32_t {
      uint32_t at = st + frag_off;
      asm volatile("" : "+v"(at));  // (opaque: the rows' offsets are the instructions', not sixteen registers)
      return at;
    };
    // One stage, at st: its MFMAs from the dy panel in the LDS; between them the operands of the stage at st_next are prepared
    // and the loads of the one at st_load are issued.  af: the fragments of the first three row blocks; leaves the next stage's.
    auto stage = [&](uint32_t st, uint32_t st_next, uint32_t st_load, const v8bf (&bqC)[2][2], v8bf (&bqN)[2][2], v8bf (&af)[4]) {
      NextRegs nx;
      v16i tr;
      uint32_t pk[8];
      float part[2];
      asm volatile("s_nop 3");  // (operands converted at the end of the stage before)
      const uint32_t panel = panel_at(st), panel_next = panel_at(st_next);
      // row blocks behind which the two weight blocks are transposed; their conversion starts behind five more MFMAs, when
      // the result is there
      constexpr int kT0 = ROWS == 8 ? 2 : 0, kT1 = ROWS == 8 ? 8 : 3;
      constexpr int kPer = ROWS == 8 ? 1 : 2;  // conversion steps (of 8 a block) in each half of a row block's MFMAs
      auto convert_part = [&](int p, int quarter) {  // (a step in two quarters; two steps a half: one to a quarter)
#pragma unroll
        for (int b = 0; b < 2; ++b) {
          const int t0 = (b ? kT1 : kT0) + 2;
          if (p == t0 && quarter == 0) asm volatile("" : "+v"(tr));  // (not read before this place)
          const int t = kPer == 1 ? (p - t0) * 2 + (quarter >> 1) : (p - t0) * 4 + quarter;
          const bool opens = kPer == 2 || (quarter & 1) == 0;
          if (p >= t0 && t > 4 && t <= 8 && opens) {  // (of the step before: the swap waits two states for its operands)
            bwd_operand_rows(pk[t - 5], pk[t - 1]);
            if (t == 8) to_operands(pk, bqN[b]);
          }
          if (p >= t0 && t < 8) {
            if (opens) convert_first(tr, t, part);
            if (kPer == 2 || (quarter & 1) == 1) convert_second(nx.s4, t, part, pk);
          }
        }
      };
#pragma unroll
      for (int p = 0; p < kRows16; ++p) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          if (p < 8) bwd_mfma<true>(acc[p][j], af[p & 3], bqC[j >> 1][j & 1]);
          else bwd_mfma<false>(acc[p][j], af[p & 3], bqC[j >> 1][j & 1]);
          if (j == 0) {
            if (p + 3 < kRows16) af[(p + 3) & 3] = bwd_panel_frag(panel, p + 3);
            else af[(p + 3) & 3] = bwd_panel_frag(panel_next, p + 3 - kRows16);
          }
          if (p == 0 && j > 0) next_read(st_next, j - 1, nx);
          if (j == 2 && p % (ROWS / 2) == ROWS / 4 && p / (ROWS / 2) < 4) issue(st_load, p / (ROWS / 2));
          convert_part(p, j);
          if (j == 3 && p == kT0) bwd_transpose(tr, nx.raw[0], ident);
          if (j == 3 && p == kT1) bwd_transpose(tr, nx.raw[1], ident);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    };

    v8bf bqA[2][2], bqB[2][2], af[4];
    wait_vmcnt<0>();  // stores of the previous tile
    lds_barrier();
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) issue(lds_base + (uint32_t)i * kBwdStageBytes, j);
    wait_vmcnt<0>();
    lds_barrier();
    {  // operands of stage 0
      NextRegs nx;
#pragma unroll
      for (int part = 0; part < 3; ++part) next_read(lds_base, part, nx);
      uint32_t pk[8];
#pragma unroll
      for (int cb = 0; cb < 2; ++cb) {
        v16i tr;
        bwd_transpose(tr, nx.raw[cb], ident);
        asm volatile("s_nop 15\n\ts_nop 15" : "+v"(tr));
#pragma unroll
        for (int t = 0; t < 8; ++t) {
          float part[2];
          convert_first(tr, t, part);
          convert_second(nx.s4, t, part, pk);
          if (t >= 4) bwd_operand_rows(pk[t - 4], pk[t]);
        }
        to_operands(pk, bqA[cb]);
      }
    }
    // Two stages to a barrier: stages i, i + 1 and i + 2 have landed, i + 4 and i + 5 are asked for (into the buffers of i - 2
    // and i - 1).
    // (one loop for all stages: those behind the last are loads and a conversion that nothing reads, and a second loop made
    // the allocator move a third of the sums at every pass of this one)
#pragma unroll
    for (int p = 0; p < 3; ++p) af[p] = bwd_panel_frag(panel_at(lds_base), p);
    uint32_t st_load = lds_base + 4u * kBwdStageBytes, st = lds_base, st_next = lds_base + 2u * kBwdStageBytes;
#pragma unroll 1
    for (int i = 0; i < L; i += 2) {
      wait_vmcnt<kBwdWideLoads>();
      // (the reads in flight are of stage i, whose buffer is filled again two barriers on)
      asm volatile("s_barrier" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
      stage(st, st + kBwdStageBytes, st_load, bqA, bqB, af);
      stage(st + kBwdStageBytes, st_next, st_load + kBwdStageBytes, bqB, bqA, af);
      const uint32_t before = st_load;
      st_load = st; st = st_next; st_next = before;
    }
    wait_vmcnt<0>();
    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");  // the last MFMAs, which the compiler does not know, have written their sums
#pragma unroll
    for (int p = 0; p < kRows16; ++p)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if (p < 8) asm volatile("" : "+a"(acc[p][j]));
        else asm volatile("" : "+v"(acc[p][j]));
      }
    auto sums = [&](int rb, int cb) -> v16f {
      v4f b[2][2];
#pragma unroll
      for (int rh = 0; rh < 2; ++rh)
#pragma unroll
        for (int ch = 0; ch < 2; ++ch) {
          v4f& a = acc[2 * rb + rh][2 * cb + ch];
          b[rh][ch] = rb < 4 ? bwd_sums<true>(a) : bwd_sums<false>(a);
        }
      return bwd_block32(b);
    };
    if (whole) {
      lds_barrier();  // (every wave has read its last stage, and nothing is on its way into the LDS)
      const uint32_t rs_lds = lds_base + 4u * kBwdTurnBytes;
      bwd_dx_fetch_rs<NKK>(g, tm * 256u, live_blocks, rs_lds, wave, 4);
      bwd_dx_store<NKK, 2, ROWS, true>(g, tm * 256u, kbw, live_blocks, lds_base + (uint32_t)wave * kBwdTurnBytes, rs_lds,
                                       sums);
    } else {
#pragma unroll
      for (int rb = 0; rb < ROWS; ++rb)
        if (rb < live_blocks) {
          float4* dst = bwd_dx_part<2>(g, slot, (uint32_t)rb, (uint32_t)wave);
#pragma unroll
          for (int cb = 0; cb < 2; ++cb) {
            const v16f y = sums(rb, cb);
#pragma unroll
            for (int e = 0; e < 4; ++e) dst[(cb * 4 + e) * 64] = make_float4(y[4 * e], y[4 * e + 1], y[4 * e + 2], y[4 * e + 3]);
          }
        }
    }
  };

  bwd_dx_schedule(g, true, [&](uint32_t t, int nb0, int len, uint32_t slot) {
    uint32_t tm, tk;
    bwd_dx_tile_at(g, t, tm, tk);
    int tw = 0, live = ((int)(g.M - tm * 256u) + 31) / 32;  // (the rows of a dense call fill the slots from the first)
    if (g.tile_weight) {
      const int tv = g.tile_weight[tm];
      if (tv < 0) return;  // workgroup-uniform: no row lives in this tile
      tw = tv & 0xffff;
      live = ((tv >> 16) + 31) / 32;
    }
    live = __builtin_amdgcn_readfirstlane(live < 8 ? live : 8);
    if (live > 4) segment(std::integral_constant<int, 8>{}, tm, tk, live, tw, nb0, len, len == (int)g.NB, slot);
    else segment(std::integral_constant<int, 4>{}, tm, tk, live, tw, nb0, len, len == (int)g.NB, slot);
  });
}

// The split tiles of a pull-back kernel: the partial sums of a tile added in the order of its stages, then the
// kernel's own epilogue.  A wave per block of 32 rows x CBN k blocks (CBN: k blocks of a wave's tile).
template <int NKK, int CBN>
__global__ __launch_bounds__(256) void bwd_dx_finish_kernel(BwdDxArgs g) {
  __shared__ __attribute__((aligned(16))) unsigned char turn[4 * kBwdTurnBytes];
  const uint32_t item = blockIdx.x * 4u + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t u = item >> 5, wave = (item >> 2) & 7u, rb = item & 3u;
  const uint32_t first = u * g.NB / g.sk_q, last = ((u + 1u) * g.NB - 1u) / g.sk_q;
  if (first == last) return;  // one workgroup had all its stages and has stored it
  uint32_t tm, tk;
  bwd_dx_tile_at(g, g.direct_tiles + u, tm, tk);
  const uint32_t pbase = tm * 256u + (wave >> 2) * 128u + rb * 32u;
  const uint32_t kbw = (tk * 4u + (wave & 3u)) * (uint32_t)CBN;
  if (pbase >= g.M || kbw >= g.KB) return;
  v16f y[CBN];
#pragma unroll
  for (int cb = 0; cb < CBN; ++cb)
#pragma unroll
    for (int e = 0; e < 16; ++e) y[cb][e] = 0.0f;
  for (uint32_t w = first; w <= last; ++w) {
    const float4* src = bwd_dx_part<CBN>(g, w + u, (wave >> 2) * 4u + rb, wave & 3u);
#pragma unroll
    for (int cb = 0; cb < CBN; ++cb)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float4 v = src[(cb * 4 + e) * 64];
        y[cb][4 * e] += v.x; y[cb][4 * e + 1] += v.y; y[cb][4 * e + 2] += v.z; y[cb][4 * e + 3] += v.w;
      }
  }
  bwd_dx_store<NKK, CBN, 1, false>(g, pbase, kbw, 1, (uint32_t)(uintptr_t)(lptr_t)turn + (threadIdx.x >> 6) * kBwdTurnBytes, 0u,
                                   [&](int, int cb) -> v16f { return y[cb]; });
}

// ---------------------------------------------------------------------------------------
// LoRA cotangents.  Rows are in grouped order; group g owns slots group_off[g] .. group_off[g+1].
// Every group is cut into chunks of 512 rows; chunk c of the call computes, for its rows,
//   partA[c][j][k] = sum_m rs[m][j] * x[m][k]        partB[c][j][n] = sum_m z[m][j] * dy[m][n]
// with float32 accumulation (the r rank rows there are), and a second kernel adds a
// group's chunks in chunk order, scales dB, casts and writes dA [g][K][r], dB [g][r][N], plus
// ds[g] = sum_m sum_j r[m][j] * z[m][j] with r the unscaled dy @ B.T.  Fixed orders: results are
// deterministic.
// ---------------------------------------------------------------------------------------

struct BwdDloraArgs {
  const uint16_t* x;        // bf16 [M, K]
  const uint16_t* dy;       // bf16 [M, N]
  const float* rs;          // f32 [slots][64]  (dy @ B.T) * s
  const float* z;           // f32 [slots][64]  x @ A
  const int32_t* src_row;   // or null
  const int32_t* x_row;     // src_row for x
  const int32_t* group_off; // [n_groups + 1]
  const int32_t* chunk_tab; // grouped calls: (group, first slot, rows) per chunk instead of group_off
  const int32_t* chunk0_tab; // grouped calls: first chunk of every group
  float* partA;             // [max_chunks][R][K]
  float* partB;             // [max_chunks][R][N]
  // a group of one chunk has its cotangents written here, and the second kernel leaves it alone
  uint16_t* d_a;            // bf16 [n_groups, K, r]
  uint16_t* d_b;            // bf16 [n_groups, r, N]
  const float* lora_scaling;
  uint32_t M, K, N, r, n_groups, max_chunks, col_tiles_a, col_tiles_b;
};

// chunk id -> (first slot, rows, group and whether it is the group's only chunk); rows = 0 beyond the last chunk.  The same in every
// lane of the wave: 64 groups are looked at together (one after the other they were a chain of loads).
__device__ inline void bwd_find_chunk(const int32_t* group_off, uint32_t n_groups, uint32_t cid, uint32_t lane,
                                      uint32_t& slot0, uint32_t& rows, uint32_t& group, bool& only) {
  slot0 = rows = group = 0;
  only = false;
  uint32_t run = 0;  // chunks of the groups before
  for (uint32_t g0 = 0; g0 < n_groups; g0 += 64u) {
    const uint32_t g = g0 + lane < n_groups ? g0 + lane : n_groups;
    const uint32_t o0 = (uint32_t)group_off[g], o1 = (uint32_t)group_off[g < n_groups ? g + 1u : g];
    const uint32_t nch = (o1 - o0 + kBwdChunkRows - 1u) / kBwdChunkRows;
    const uint32_t upto = wave_scan(nch);  // of this and the lanes below
    const uint64_t reached = __builtin_amdgcn_ballot_w64(cid < run + upto);
    if (reached) {
      const int own = __builtin_ctzll(reached);
      const uint32_t before = run + (uint32_t)__builtin_amdgcn_readlane((int)(upto - nch), own);
      const uint32_t end = (uint32_t)__builtin_amdgcn_readlane((int)o1, own);
      slot0 = (uint32_t)__builtin_amdgcn_readlane((int)o0, own) + (cid - before) * kBwdChunkRows;
      rows = end - slot0 < kBwdChunkRows ? end - slot0 : kBwdChunkRows;
      group = g0 + (uint32_t)own;
      only = __builtin_amdgcn_readlane((int)nch, own) == 1;
      return;
    }
    run += (uint32_t)__builtin_amdgcn_readlane((int)upto, 63);
  }
}

// Matrix-core version.  out[j][c] = sum_m P[m][j] * Q[m][c] contracts over rows, so both operands
// need the row index inside a lane.  P (float32, 32 or 64 rank columns) is split exactly into three
// bf16 terms and staged in LDS in A-operand order.  Q (bf16 rows of x or dy) is read as ordinary
// row fragments and transposed by the matrix core: two v_mfma_f32_32x32x16_bf16 against identity
// halves return Q[m][c] with lane = c and sixteen rows per lane (exact: the values are bf16), which
// packs into the B operands of the contraction over m.  A wave owns 64 columns (two 32-column
// strips) and walks the chunk's 32-row blocks, eight per staging pass of P; a workgroup of four
// waves owns 256 columns.
// Bound by latencies: a call has few chunks, so a SIMD holds one to three waves.  Hence the ring of Q in flight beside
// the block at work, through the staging passes too (one rank block: two blocks, so that three workgroups fit a
// CU; with four blocks and two workgroups experts of 64 rows took 30.2 us instead of 22.5); all of a pass's P
// requested together, with two rank blocks the second pass's while the first is multiplied; P's operands read ahead of
// the transposition; loads without conditions (a row or column that is not there reads the tensor's first bytes and
// is cleared where it is used), so that the waits count.  One block of Q ahead, P's pieces one after the other
// and operands read at their MFMAs, before, us -> now: 2048 rows of rank 64, 2560 + 10240 columns 37.9 -> 29.7; 3003 rows of
// rank 32, 12288 + 4096 40.9 -> 34.3, 4096 + 24576 60-62 both (200 MB, 3.3 TB/s); 1536 rows of one
// adapter 27.7 -> 19.6; 128 experts of 64 rows 22 and 27 both.
template <int RB>  // 32-wide rank blocks
__global__ __launch_bounds__(256, RB == 1 ? 3 : 1) void bwd_dlora_kernel(BwdDloraArgs a) {
  constexpr uint32_t kRing = RB == 1 ? 2 : 4;  // blocks of Q in flight
  constexpr uint32_t kItems = 4 * RB;  // operand pieces of P that a thread stages in a pass
  // P operands: [row block 8][rank block RB][q 2][term 3][64 lanes][8 bf16]
  extern __shared__ __attribute__((aligned(1024))) unsigned char pop[];
  __shared__ int rowsrc[kBwdChunkRows];
  const uint32_t tid = threadIdx.x, lane = tid & 63u;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t per_chunk = a.col_tiles_a + a.col_tiles_b;
  const uint32_t cid = blockIdx.x / per_chunk, ct = blockIdx.x % per_chunk;
  uint32_t slot0, rows, group;
  bool only;
  if (a.chunk_tab) {
    group = (uint32_t)a.chunk_tab[3u * cid];
    slot0 = (uint32_t)a.chunk_tab[3u * cid + 1u];
    rows = (uint32_t)a.chunk_tab[3u * cid + 2u];
    only = a.chunk0_tab[group + 1u] - a.chunk0_tab[group] == 1;
  } else {
    bwd_find_chunk(a.group_off, a.n_groups, cid, lane, slot0, rows, group, only);
  }
  if (rows == 0) return;  // workgroup-uniform
  const bool job_a = ct < a.col_tiles_a;
  const float* psrc = job_a ? a.rs : a.z;
  const uint16_t* Q = job_a ? a.x : a.dy;
  const uint32_t C = job_a ? a.K : a.N;
  float* part = job_a ? a.partA : a.partB;
  const uint32_t c = lane & 31u, h = lane >> 5;
  const uint32_t col0 = ((job_a ? ct : ct - a.col_tiles_a) * 4u + wave) * 64u;  // first column of the wave
  const bool active = col0 < C;
  const uint32_t n_blocks = (rows + 31u) / 32u;

  // item i of a thread = (row block, rank block, q, lane); element e is row 16 q + 8 (e / 4) + 4 h + e % 4
  const uint32_t pq = wave & 1u;
  auto item_block = [&](uint32_t i) { return (4u * i + wave) / (2u * RB); };
  auto item_rank = [&](uint32_t i) { return (4u * i + wave) / 2u % RB; };
  auto load_p = [&](uint32_t base, float (&praw)[kItems][8]) {
#pragma unroll
    for (uint32_t i = 0; i < kItems; ++i)
      if (base + item_block(i) * 32u < rows) {  // wave-uniform
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          uint32_t m = base + item_block(i) * 32u + 16u * pq + 8u * (e >> 2) + 4u * h + (e & 3);
          m = m < rows ? m : rows - 1u;
          praw[i][e] = psrc[(size_t)(slot0 + m) * kBwdRankStride + item_rank(i) * 32u + c];
        }
      }
  };
  auto stage_p = [&](uint32_t base, const float (&praw)[kItems][8]) {
#pragma unroll
    for (uint32_t i = 0; i < kItems; ++i)
      if (base + item_block(i) * 32u < rows) {
        v8us t0, t1, t2;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const uint32_t m = base + item_block(i) * 32u + 16u * pq + 8u * (e >> 2) + 4u * h + (e & 3);
          const float v = m < rows ? praw[i][e] : 0.0f;
          const uint32_t b0 = f32_to_bf16_bits(v);
          const float r1 = v - bf16_bits_to_f32(b0);
          const uint32_t b1 = f32_to_bf16_bits(r1);
          const float r2 = r1 - bf16_bits_to_f32(b1);
          t0[e] = (unsigned short)b0; t1[e] = (unsigned short)b1; t2[e] = (unsigned short)f32_to_bf16_bits(r2);
        }
        unsigned char* dst = pop + (((size_t)item_block(i) * RB + item_rank(i)) * 2u + pq) * 3u * kBlockBytes + lane * 16u;
        *reinterpret_cast<v8us*>(dst) = t0;
        *reinterpret_cast<v8us*>(dst + kBlockBytes) = t1;
        *reinterpret_cast<v8us*>(dst + 2 * kBlockBytes) = t2;
      }
  };
  // (the rows' sources first: Q waits for them)
  int src[kBwdChunkRows / 256u];
#pragma unroll
  for (uint32_t i = 0; i < kBwdChunkRows / 256u; ++i) {
    const uint32_t m = i * 256u + tid < rows ? i * 256u + tid : rows - 1u;
    const int32_t* const rows_of = job_a ? a.x_row : a.src_row;
    src[i] = rows_of ? rows_of[slot0 + m] : (int)(slot0 + m);
  }
  float praw[kItems][8];
  load_p(0, praw);
#pragma unroll
  for (uint32_t i = 0; i < kBwdChunkRows / 256u; ++i) rowsrc[i * 256u + tid] = i * 256u + tid < rows ? src[i] : -1;
  lds_barrier();

  // identity halves: lane (column c, half h) element e is 1 where the contraction slot 8 h + e is column c
  v8us id0 = {0, 0, 0, 0, 0, 0, 0, 0}, id1 = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    id0[e] = (c == 8u * h + e) ? (unsigned short)0x3f80 : (unsigned short)0;
    id1[e] = (c == 16u + 8u * h + e) ? (unsigned short)0x3f80 : (unsigned short)0;
  }
  v16f acc[2][RB];
#pragma unroll
  for (int st = 0; st < 2; ++st)
#pragma unroll
    for (int b = 0; b < RB; ++b)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[st][b][e] = 0.0f;
  v4i qf[kRing][2][2];  // [strip][column half]: row c of the block, 8 columns
  bool row_ok[kRing];
  auto load_q = [&](uint32_t bi, uint32_t u) {
    const int srow = rowsrc[(bi < n_blocks ? bi : n_blocks - 1u) * 32u + c];
    row_ok[u] = srow >= 0;
#pragma unroll
    for (int st = 0; st < 2; ++st)
#pragma unroll
      for (int hc = 0; hc < 2; ++hc) {
        const uint32_t col = col0 + 32u * st + 16u * hc + 8u * h;
        qf[u][st][hc] = *reinterpret_cast<const v4i*>(Q + (row_ok[u] && col + 8u <= C ? (size_t)srow * C + col : 0));
      }
  };
  auto multiply = [&](uint32_t bi, uint32_t u) {  // bi: the block in the staging pass
    v8us pf[RB][2][3];
#pragma unroll
    for (int b = 0; b < RB; ++b)
#pragma unroll
      for (int q = 0; q < 2; ++q)
#pragma unroll
        for (int t3 = 0; t3 < 3; ++t3)
          pf[b][q][t3] = *reinterpret_cast<const v8us*>(pop + ((((size_t)bi * RB + b) * 2u + q) * 3u + t3) * kBlockBytes + lane * 16u);
    // (they arrive behind the transposition; read one by one each makes its MFMAs wait)
    if constexpr (RB == 2) __builtin_amdgcn_sched_barrier(0);
    v4i bq[2][2];
#pragma unroll
    for (int st = 0; st < 2; ++st) {
      v16f tr;
#pragma unroll
      for (int e = 0; e < 16; ++e) tr[e] = 0.0f;
#pragma unroll
      for (int hc = 0; hc < 2; ++hc) {
        const bool ok = row_ok[u] && col0 + 32u * st + 16u * hc + 8u * h + 8u <= C;
        v4i f;
#pragma unroll
        for (int d = 0; d < 4; ++d) f[d] = ok ? qf[u][st][hc][d] : 0;
        tr = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8bf, f), __builtin_bit_cast(v8bf, hc ? id1 : id0), tr, 0, 0, 0);
      }
#pragma unroll
      for (int q = 0; q < 2; ++q)
#pragma unroll
        for (int e = 0; e < 4; ++e) bq[st][q][e] = (int)pack_bf16x2(tr[8 * q + 2 * e], tr[8 * q + 2 * e + 1]);
    }
#pragma unroll
    for (int b = 0; b < RB; ++b)
#pragma unroll
      for (int q = 0; q < 2; ++q)
#pragma unroll
        for (int t3 = 2; t3 >= 0; --t3)
#pragma unroll
          for (int st = 0; st < 2; ++st)
            acc[st][b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8bf, pf[b][q][t3]),
                                                                 __builtin_bit_cast(v8bf, bq[st][q]), acc[st][b], 0, 0, 0);
  };
  constexpr uint32_t kPassBlocks = kBwdStageRows / 32u;
  static_assert(kBwdChunkRows == 2u * kBwdStageRows, "a chunk is two passes");
  static_assert(kPassBlocks % kRing == 0, "a pass holds whole turns of the ring");
  if (active) {
#pragma unroll
    for (uint32_t u = 0; u < kRing; ++u) load_q(u, u);
  }
  stage_p(0, praw);
  lds_barrier();
  if constexpr (RB == 2) load_p(kBwdStageRows, praw);
  for (uint32_t b0 = 0; b0 < n_blocks; b0 += kRing) {
    if (b0 && b0 % kPassBlocks == 0) {
      lds_barrier();  // the pass before is no longer read
      if constexpr (RB == 1) {
        float pn[kItems][8];
        load_p(b0 * 32u, pn);
        stage_p(b0 * 32u, pn);
      } else {
        stage_p(b0 * 32u, praw);
      }
      lds_barrier();
    }
    if (!active) continue;
    // (one body: with a second one for the last blocks the allocator copied and spilled the accumulators where they meet)
#pragma unroll
    for (uint32_t u = 0; u < kRing; ++u) {
      if (u == 0 || b0 + u < n_blocks) multiply(b0 % kPassBlocks + u, u);
      load_q(b0 + u + kRing, u);  // behind the last block: its lines again
    }
  }
  // lane (c, h) holds column col0 + 32 st + c, rank rows 32 b + 8 (v / 4) + 4 h + v % 4
  if (!only) {  // workgroup-uniform
    if (!active) return;
#pragma unroll
    for (int st = 0; st < 2; ++st) {
      const uint32_t col = col0 + 32u * st + c;
      if (col >= C) continue;
#pragma unroll
      for (int b = 0; b < RB; ++b)
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          if (b * 32u + 8u * (v >> 2) >= a.r) continue;  // (uniform; rank rows beyond r are not read)
          const uint32_t j = b * 32u + 8u * (v >> 2) + 4u * h + (v & 3);
          part[((size_t)cid * (RB * 32u) + j) * C + col] = acc[st][b][v];
        }
    }
    return;
  }
  // A group of one chunk is done here, its sums with the second kernel's operations (added to zero, dB scaled, cast).  The values change
  // hands in the LDS (P is spent): dA's lie r to a column there, so that a wave's 64 columns are one piece of memory, dB's 64
  // columns to a rank row.  Both kernels, us, before -> now: 128 experts of 64 rows, rank 16, 2048 -> 1536 and 768 -> 2048 68.8 -> 53.7; 2048 rows of
  // rank 64, 512 to an adapter, 2560 + 10240 columns 35.1 -> 33.0 (straight from the registers 38.6).
  lds_barrier();
  if (!active) return;
  typedef __attribute__((address_space(3))) unsigned char* lds_ptr;
  typedef __attribute__((address_space(3))) const v4i* lds_v4ptr;
  typedef uint32_t v2u __attribute__((ext_vector_type(2)));
  const uint32_t cols = C - col0 < 64u ? C - col0 : 64u;
  if (job_a) {
    constexpr uint32_t kStride = RB * 64u + 16u;  // bytes of a column
    static_assert(4u * 64u * kStride <= (kBwdStageRows / 32u) * RB * 6u * (uint32_t)kBlockBytes, "P's place");
    const lds_ptr turn = (lds_ptr)(lptr_t)pop + wave * (64u * kStride);
#pragma unroll
    for (int st = 0; st < 2; ++st)
#pragma unroll
      for (int b = 0; b < RB; ++b)
#pragma unroll
        for (int v = 0; v < 16; v += 4)
          *reinterpret_cast<__attribute__((address_space(3))) v2u*>(turn + (32u * st + c) * kStride + (b * 32u + 2u * v + 4u * h) * 2u) =
              v2u{pack_bf16x2(0.0f + acc[st][b][v], 0.0f + acc[st][b][v + 1]), pack_bf16x2(0.0f + acc[st][b][v + 2], 0.0f + acc[st][b][v + 3])};
    __builtin_amdgcn_wave_barrier();  // (a wave reads what it has written itself)
    uint16_t* const o = a.d_a + ((size_t)group * a.K + col0) * a.r;
    if ((a.r & 7u) == 0) {
      const uint32_t pieces = a.r / 8u;
      for (uint32_t e = lane; e < cols * pieces; e += 64u)
        *reinterpret_cast<v4i*>(o + e * 8u) = *reinterpret_cast<lds_v4ptr>(turn + (e / pieces) * kStride + (e % pieces) * 16u);
    } else {
      for (uint32_t e = lane; e < cols * a.r; e += 64u)
        o[e] = *reinterpret_cast<__attribute__((address_space(3))) const uint16_t*>(turn + (e / a.r) * kStride + (e % a.r) * 2u);
    }
  } else {
    constexpr uint32_t kStride = 144u;  // bytes of a rank row
    static_assert(4u * RB * 32u * kStride <= (kBwdStageRows / 32u) * RB * 6u * (uint32_t)kBlockBytes, "P's place");
    const lds_ptr turn = (lds_ptr)(lptr_t)pop + wave * (RB * 32u * kStride);
    const float sc = a.lora_scaling[group];
#pragma unroll
    for (int st = 0; st < 2; ++st)
#pragma unroll
      for (int b = 0; b < RB; ++b)
#pragma unroll
        for (int v = 0; v < 16; ++v)
          *reinterpret_cast<__attribute__((address_space(3))) uint16_t*>(turn + (b * 32u + 8u * (v >> 2) + 4u * h + (v & 3)) * kStride + (32u * st + c) * 2u) =
              (uint16_t)f32_to_bf16_bits((0.0f + acc[st][b][v]) * sc);
    __builtin_amdgcn_wave_barrier();
    uint16_t* const o = a.d_b + (size_t)group * a.r * a.N + col0;
    const uint32_t cl = (lane & 7u) * 8u;  // (N is a multiple of 8)
    if (cl < cols)
      for (uint32_t j = lane >> 3; j < a.r; j += 8u)
        *reinterpret_cast<v4i*>(o + (size_t)j * a.N + cl) = *reinterpret_cast<lds_v4ptr>(turn + j * kStride + cl * 2u);
  }
}

struct BwdReduceArgs {
  const float* partA; const float* partB;
  const float* r_raw;       // f32 [slots][64] unscaled dy @ B.T
  const float* z;           // f32 [slots][64]
  const double* row_dot;    // f64 [slots] r . z
  const float* lora_scaling;
  const int32_t* group_off;
  // grouped calls: first chunk of every group (n_groups + 1) and the groups' slot ranges, in memory
  const int32_t* chunk0_tab; const int32_t* group_beg; const int32_t* group_end;
  uint16_t* d_a;            // bf16 [n_groups, K, r] or null
  uint16_t* d_b;            // bf16 [n_groups, r, N] or null
  float* d_s;               // f32 [n_groups] or null
  uint32_t K, N, r, R, n_groups, blocks_a, blocks_b;
};

constexpr uint32_t kBwdReduceCols = 64;  // columns of dA of a workgroup

struct BwdNoPlain { static constexpr bool kAny = false; };

// Adds the chunks.  Bound by memory (2048 rows, rank 64: 26 MB of partials) and by the one workgroup per group that forms ds.
// 2048 rows of rank 64 15-18 -> 7.4 us, 3003 of rank 32 34 -> 6.8 and 8.3, 1536 of one adapter 29 -> 5.6, 128 experts
// 13 and 19 -> 9.1 and 10.6: with ds formed from bwd_r_finish_kernel's row_dot, and dA read along k and turned in the LDS.
// Plain: what replaces the sums of the partials where an operand is not finite (group-scaled calls), or BwdNoPlain.
template <class Plain>
__global__ __launch_bounds__(256) void bwd_dlora_reduce_kernel(BwdReduceArgs a, Plain plain) {
  __shared__ uint32_t chunk0_lds[kMaxAdapters + 1];
  __shared__ double red[256];
  __shared__ __attribute__((aligned(16))) uint16_t turn[kBwdReduceCols][kBwdRankStride + 8];
  const uint32_t tid = threadIdx.x;
  bool use_plain = false;  // kernel-uniform
  if constexpr (Plain::kAny) use_plain = plain.wanted();
  if (!a.chunk0_tab && tid < 64u) {
    // first chunk of every group: the dense tables hold at most 64 groups, so one wave loads all the
    // offsets at once and scans the chunk counts (a serial loop over dependent loads in front of every
    // workgroup of this short kernel cost more than the reduction itself)
    static_assert(kMaxAdapters <= 64, "one wave scans the groups");
    uint32_t cnt = 0;
    if (tid < a.n_groups)
      cnt = ((uint32_t)(a.group_off[tid + 1] - a.group_off[tid]) + kBwdChunkRows - 1u) / kBwdChunkRows;
    cnt = wave_scan(cnt);
    if (tid < a.n_groups) chunk0_lds[tid + 1u] = cnt;  // inclusive sums
    if (tid == 0) chunk0_lds[0] = 0u;
  }
  __syncthreads();
  auto chunk0 = [&](uint32_t gq) -> uint32_t { return a.chunk0_tab ? (uint32_t)a.chunk0_tab[gq] : chunk0_lds[gq]; };
  auto reduce_ds = [&](uint32_t b) {  // one block per group
    const uint32_t o0 = (uint32_t)(a.group_beg ? a.group_beg[b] : a.group_off[b]);
    const uint32_t o1 = (uint32_t)(a.group_end ? a.group_end[b] : a.group_off[b + 1]);
    double sum = 0.0;
    if (use_plain) {
      if constexpr (Plain::kAny) sum = plain.d_s(a.r_raw, a.z);
    } else {
      for (uint32_t slot = o0 + tid; slot < o1; slot += 1024u) {
        double v[4];
#pragma unroll
        for (uint32_t u = 0; u < 4; ++u) v[u] = a.row_dot[slot + 256u * u < o1 ? slot + 256u * u : slot];
#pragma unroll
        for (uint32_t u = 0; u < 4; ++u) sum += slot + 256u * u < o1 ? v[u] : 0.0;
      }
    }
    red[tid] = sum;
    __syncthreads();
    for (uint32_t o = 128; o > 0; o >>= 1) {
      if (tid < o) red[tid] += red[tid + o];
      __syncthreads();
    }
    if (tid == 0) a.d_s[b] = (float)red[0];
  };
  // four adjacent columns of rank row j, the chunks of a group added in order, four of them in flight
  auto sum_chunks = [&](const float* part, uint32_t grp, uint32_t j, uint32_t col, uint32_t C) -> float4 {
    float4 sum = make_float4(0.f, 0.f, 0.f, 0.f);
    const uint32_t ce = chunk0(grp + 1u);
    for (uint32_t ch = chunk0(grp); ch < ce; ch += 4u) {
      float4 v[4];
#pragma unroll
      for (uint32_t u = 0; u < 4; ++u)
        v[u] = *reinterpret_cast<const float4*>(part + ((size_t)(ch + u < ce ? ch + u : ch) * a.R + j) * C + col);
#pragma unroll
      for (uint32_t u = 0; u < 4; ++u)
        if (ch + u < ce) { sum.x += v[u].x; sum.y += v[u].y; sum.z += v[u].z; sum.w += v[u].w; }
    }
    return sum;
  };
  // (groups of one chunk are written by bwd_dlora_kernel)
  auto done = [&](uint32_t grp) { return !use_plain && chunk0(grp + 1u) - chunk0(grp) == 1u; };
  // The blocks of ds come first in the grid: each walks all rows of its group (one number a row, see bwd_r_finish_kernel:
  // over the r and z tables themselves one workgroup a group took longer than the rest of the launch), so it starts at once
  // and runs beside the short dA / dB blocks instead of after them.
  const uint32_t blocks_s = a.d_s ? a.n_groups : 0u;
  if (blockIdx.x < blocks_s) {
    reduce_ds(blockIdx.x);
    return;
  }
  uint32_t b = blockIdx.x - blocks_s;
  if (b < a.blocks_a) {
    // dA [group][k][j]: a block turns 64 columns k of a group, read along k, into rows of j (their outputs are one
    // piece of memory).  (A thread per output, j fastest, read four bytes of every line it touched, once per rank.)
    const uint32_t strips = (a.K + kBwdReduceCols - 1u) / kBwdReduceCols, grp = b / strips, c0 = b % strips * kBwdReduceCols;
    if (done(grp)) return;
    const uint32_t cl = (tid & 15u) * 4u, col = c0 + cl;  // (K is a multiple of 8)
    for (uint32_t j = tid >> 4; j < a.r; j += 16u) {
      float4 sum = make_float4(0.f, 0.f, 0.f, 0.f);
      if (col < a.K) {
        if (use_plain) {
          if constexpr (Plain::kAny)
            sum = make_float4(plain.d_a(col, j), plain.d_a(col + 1u, j), plain.d_a(col + 2u, j), plain.d_a(col + 3u, j));
        } else {
          sum = sum_chunks(a.partA, grp, j, col, a.K);
        }
      }
      turn[cl][j] = (uint16_t)f32_to_bf16_bits(sum.x);
      turn[cl + 1u][j] = (uint16_t)f32_to_bf16_bits(sum.y);
      turn[cl + 2u][j] = (uint16_t)f32_to_bf16_bits(sum.z);
      turn[cl + 3u][j] = (uint16_t)f32_to_bf16_bits(sum.w);
    }
    __syncthreads();
    const uint32_t cols = a.K - c0 < kBwdReduceCols ? a.K - c0 : kBwdReduceCols;
    uint16_t* dst = a.d_a + ((size_t)grp * a.K + c0) * a.r;
    if ((a.r & 7u) == 0) {
      for (uint32_t e = tid * 8u; e < cols * a.r; e += 2048u)
        *reinterpret_cast<v8us*>(dst + e) = *reinterpret_cast<const v8us*>(&turn[e / a.r][e % a.r]);
    } else {
      for (uint32_t e = tid; e < cols * a.r; e += 256u) dst[e] = turn[e / a.r][e % a.r];
    }
    return;
  }
  if (b < a.blocks_a + a.blocks_b) {
    // dB [group][j][n]: a thread per four adjacent columns (N is a multiple of 8)
    const uint64_t e = ((uint64_t)(b - a.blocks_a) * 256u + tid) * 4u;
    if (e >= (uint64_t)a.n_groups * a.r * a.N) return;
    const uint32_t col = (uint32_t)(e % a.N), j = (uint32_t)((e / a.N) % a.r), grp = (uint32_t)(e / ((uint64_t)a.N * a.r));
    if (done(grp)) return;
    float4 sum = make_float4(0.f, 0.f, 0.f, 0.f);
    if (use_plain) {
      if constexpr (Plain::kAny)
        sum = make_float4(plain.d_b(a.z, col, j), plain.d_b(a.z, col + 1u, j), plain.d_b(a.z, col + 2u, j), plain.d_b(a.z, col + 3u, j));
    } else {
      sum = sum_chunks(a.partB, grp, j, col, a.N);
    }
    const float sc = a.lora_scaling[grp];
    *reinterpret_cast<uint2*>(a.d_b + e) = make_uint2(pack_bf16x2(sum.x * sc, sum.y * sc), pack_bf16x2(sum.z * sc, sum.w * sc));
    return;
  }
  if constexpr (Plain::kAny) {
    if (use_plain) plain.d_x(b - a.blocks_a - a.blocks_b);
  }
}

}  // namespace w8a8
