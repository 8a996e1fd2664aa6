// Prologue kernels: weight (un)packing, adapter routing, per-token quantization with the
// optional fused RMSNorm, and the LoRA-A projection z = n @ A[adapter].
#pragma once
#include <type_traits>

#include "w8a8_device.h"

namespace w8a8 {

// ---------------------------------------------------------------------------------------
// Weight pack / unpack (one time per weight)
// ---------------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void pack_weight_kernel(const int8_t* __restrict__ codes,
                                                          unsigned char* __restrict__ packed, uint32_t K,
                                                          uint32_t N, uint32_t KB, uint64_t n_chunks) {
  uint64_t idx = (uint64_t)blockIdx.x * 256 + threadIdx.x;  // one 16-byte chunk per thread
  if (idx >= n_chunks) return;
  uint32_t lane = idx & 63u;
  uint64_t blk = idx >> 6;
  uint32_t kb = (uint32_t)(blk % KB);
  uint32_t nb = (uint32_t)(blk / KB);
  uint32_t c = nb * 32u + (lane & 31u);
  uint32_t n = packed_to_orig_col(c);
  uint32_t k0 = kb * 32u + 16u * (lane >> 5);
  uint32_t w[4] = {0, 0, 0, 0};
  if (n < N) {
#pragma unroll
    for (int b = 0; b < 16; ++b) {
      uint32_t k = k0 + b;
      uint32_t v = (k < K) ? (uint32_t)(uint8_t)codes[(size_t)k * N + n] : 0u;
      w[b >> 2] |= v << (8 * (b & 3));
    }
  }
  uint4 o = make_uint4(w[0], w[1], w[2], w[3]);
  *reinterpret_cast<uint4*>(packed + idx * 16) = o;
}

__global__ __launch_bounds__(256) void unpack_weight_kernel(const unsigned char* __restrict__ packed,
                                                            int8_t* __restrict__ codes, uint32_t K, uint32_t N,
                                                            uint32_t KB) {
  uint64_t idx = (uint64_t)blockIdx.x * 256 + threadIdx.x;
  if (idx >= (uint64_t)K * N) return;
  uint32_t k = (uint32_t)(idx / N), n = (uint32_t)(idx % N);
  codes[idx] = (int8_t)packed[packed_offset(orig_to_packed_col(n), k, KB)];
}

// ---------------------------------------------------------------------------------------
// Adapter routing: rows are grouped by adapter with no padding between groups (the
// counterpart of prepare_routing, skyrl/tx/layers/util.py:66-87).
//   src_row[p]    = original row of grouped slot p (p < M), -1 for the slots beyond M
//   dst_pos[m]    = grouped slot of original row m (optional)
//   slot_group[p] = adapter of grouped slot p
//   blk_range[b]  = first adapter | last adapter << 16 of the 32-row block b
//   group_off[a]  = first grouped slot of adapter a (optional; entry n_groups = M)
// Out-of-range adapter indices are clamped into range (XLA gather semantics).
// ---------------------------------------------------------------------------------------
// With group_pad = 32 every group starts on a 32-slot boundary, so that no 32-slot block holds rows of two
// groups (neither the quantizer nor the GEMM's epilogue then runs a block once per group): the slots between
// a group's last row and the next group's first stay empty.
// One workgroup of sixteen waves, each with a contiguous range of the rows: a wave counts its rows per group
// (lanes with the same group find each other with one ballot per bit of the index, so a group costs a wave one
// LDS atomic per 64 rows), wave 0 turns the counts into first slots, and the waves place their rows in order.
// rows_per_index > 1: an index serves that many rows that follow each other.  (Written out per row by a launch in front,
// 333 rows of nine sequences, 4096 -> 2560, took 34.3 us a call, now 31.8.)
// Rows so keep their order inside a group: reductions over a group's rows have a fixed order.  Bound by the
// latency of its few steps: 14 us for
// 4096 rows with an atomic per row and a search per slot.
__device__ inline void route_rows_block(const int32_t* __restrict__ idx, uint32_t M, uint32_t n_groups,
                                        uint32_t slots, int32_t* __restrict__ src_row,
                                        int32_t* __restrict__ dst_pos, int32_t* __restrict__ slot_group,
                                        int32_t* __restrict__ blk_range, int32_t* __restrict__ group_off = nullptr,
                                        uint32_t group_pad = 1u, uint32_t rows_per_index = 1u) {
  static_assert(kMaxAdapters == 64, "a lane per group");
  __shared__ int wcnt[16][kMaxAdapters];  // rows of group g in wave w; then the wave's next slot in the group
  __shared__ int cnt[kMaxAdapters];
  __shared__ int start[kMaxAdapters + 1];
  __shared__ int last_group;
  const uint32_t tid = threadIdx.x, lane = tid & 63u;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t per = (M + 1024u - 1u) / (1024u);  // 64-row steps of a wave
  auto group_at = [&](uint32_t it) -> int {
    const uint32_t i = (wave * per + it) * 64u + lane;
    const uint32_t row = i < M ? i : M - 1u;
    const int a = idx[rows_per_index > 1u ? row / rows_per_index : row];
    return i < M ? (a < 0 ? 0 : (a >= (int)n_groups ? (int)n_groups - 1 : a)) : -1;
  };
  auto peers_of = [&](int a) -> unsigned long long {  // lanes with this lane's group
    unsigned long long mask = __builtin_amdgcn_ballot_w64(a >= 0);
#pragma unroll
    for (int bit = 0; bit < 6; ++bit) {
      const unsigned long long set = __builtin_amdgcn_ballot_w64((a >> bit) & 1);
      mask &= ((a >> bit) & 1) ? set : ~set;
    }
    return mask;
  };
  wcnt[wave][lane] = 0;
  auto count = [&](int a) {
    const unsigned long long peers = peers_of(a);
    if (a >= 0 && (int)lane == __builtin_ctzll(peers)) atomicAdd(&wcnt[wave][a], __builtin_popcountll(peers));
  };
#pragma unroll 4
  for (uint32_t it = 0; it < per; ++it) count(group_at(it));
  __syncthreads();
  if (wave == 0) {  // lane g: group g
    int total = 0;
#pragma unroll
    for (uint32_t w = 0; w < 16; ++w) total += wcnt[w][lane];  // (groups that do not exist: zeros)
    const int padded = (int)round_up((uint32_t)total, group_pad);
    const int incl = (int)wave_scan((uint32_t)padded);
    int pos = incl - padded;
    cnt[lane] = total;
    start[lane] = pos;  // (groups that do not exist: empty, behind the last one)
    if (lane == 63u) start[64] = incl;
#pragma unroll
    for (uint32_t w = 0; w < 16; ++w) {
      const int c = wcnt[w][lane];
      wcnt[w][lane] = pos;
      pos += c;
    }
    const unsigned long long nonempty = __builtin_amdgcn_ballot_w64(total > 0);
    if (lane == 0) last_group = nonempty ? 63 - __builtin_clzll(nonempty) : 0;
  }
  __syncthreads();
  const uint32_t E = (uint32_t)start[n_groups];  // first slot behind the last group (M when the groups are packed)
  auto place = [&](int a, uint32_t it) {
    const unsigned long long peers = peers_of(a);
    const int leader = peers ? __builtin_ctzll(peers) : 0;
    int p = 0;
    if (a >= 0 && (int)lane == leader) p = atomicAdd(&wcnt[wave][a], __builtin_popcountll(peers));
    p = __builtin_amdgcn_ds_bpermute(4 * leader, p) + __builtin_popcountll(peers & ((1ull << lane) - 1ull));
    if (a >= 0) {
      const int i = (int)((wave * per + it) * 64u + lane);
      src_row[p] = i;
      if (dst_pos) dst_pos[i] = p;
      slot_group[p] = a;
    }
  };
#pragma unroll 4
  for (uint32_t it = 0; it < per; ++it) place(group_at(it), it);
  if (group_off && tid <= n_groups) group_off[tid] = start[tid];  // first slot of every group, then E
  if (group_pad > 1u) {  // the empty slots between groups (fewer than group_pad <= 32 behind each)
    for (uint32_t t = tid; t < n_groups * 32u; t += 1024u) {
      const uint32_t g = t >> 5, p = (uint32_t)(start[g] + cnt[g]) + (t & 31u);
      if (p < (uint32_t)start[g + 1u] && p < slots) { src_row[p] = -1; slot_group[p] = (int)g; }
    }
  }
  for (uint32_t p = E + tid; p < slots; p += 1024u) {  // padding slots follow the last non-empty group
    src_row[p] = -1;
    slot_group[p] = last_group;
  }
  // group of a slot = the group whose [start, next start) range holds it
  for (uint32_t b = tid; b < slots / 32u; b += 1024u) {
    const int p0 = (int)b * 32, p1 = (p0 + 31 < (int)E) ? p0 + 31 : (int)E - 1;
    int g0 = 0, g1 = 0;
    for (uint32_t a = 0; a < n_groups; ++a) {
      if (p0 >= start[a] && p0 < start[a + 1]) g0 = (int)a;
      if (p1 >= start[a] && p1 < start[a + 1]) g1 = (int)a;
    }
    if (p0 >= (int)E) { g0 = 0; g1 = 0; }
    blk_range[b] = g0 | (g1 << 16);
  }
}

// ---------------------------------------------------------------------------------------
// Tables for rows that arrive already grouped (ragged groups of an expert layer,
// skyrl/tx/layers/util.py:8-59): group g owns group_sizes[g] consecutive rows and is padded
// to a multiple of 32 grouped slots so that a 32-row block never mixes two weights.
//   src_row[p]   = original row of slot p, -1 for padding
//   blk_range[b] = g | g << 16 for the 32-row blocks in use, -1 beyond
//   tile_tab     = number of row tiles, then first block | blocks << 32 | group << 48 of each: a group's blocks
//                  in the fewest tiles of at most tile_blocks, of heights that differ by one at most
// ---------------------------------------------------------------------------------------
constexpr int kMaxGroups = 1024;
// Exclusive prefix sums of N values per thread over a workgroup of 1024 threads, every partial sum capped
// at `limit` (a capped sum of non-negative terms does not depend on the order they are added in).  v becomes
// the thread's prefix; total receives the sum of all.
// A chain in front of everything that waits for the tables: two barriers, the sums of the sixteen waves read by every thread at
// once.  With __shfl_up, one thread adding the waves' sums and a barrier more, the launches of an expert layer's routing
// (16 tokens, 128 experts) took 5.9 and 5.7 us (lora_prep_kernel) and 4.0 (moe_sort_kernel), now 4.7, 4.2 and 3.4.
template <int N>
__device__ inline void block_prefix_capped(uint32_t (&v)[N], uint32_t limit, uint32_t (&total)[N]) {
  __shared__ __attribute__((aligned(16))) uint32_t wave_sums[N][16];
  const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
  auto add = [&](uint32_t x, uint32_t y) {
    const uint32_t t = __builtin_elementwise_add_sat(x, y);
    return t > limit ? limit : t;
  };
  uint32_t incl[N];
#pragma unroll
  for (int i = 0; i < N; ++i) incl[i] = wave_scan(v[i] > limit ? limit : v[i], add);
  __syncthreads();  // (the table may still be read from a call before)
#pragma unroll
  for (int i = 0; i < N; ++i)
    if (lane == 63u) wave_sums[i][wave] = incl[i];
  __syncthreads();
#pragma unroll
  for (int i = 0; i < N; ++i) {
    uint32_t before = 0, all = 0;
#pragma unroll
    for (uint32_t w = 0; w < 16; ++w) {
      const uint32_t t = wave_sums[i][w];
      before = w < wave ? add(before, t) : before;
      all = add(all, t);
    }
    total[i] = all;
    v[i] = add(before, lane_before(incl[i]));  // the waves before, then the lanes before
  }
}

// Part `part` of `n_parts` workgroups of 1024 threads: every part forms the prefix sums for itself (at most
// 1024 groups, one per thread) and fills its share of the tables, slot by slot.  Group g keeps
// min(size, rows left) rows, as a sequential pass over the sizes would give it.  Rows beyond
// sum(group_sizes) get no slot; their output rows (zero_out, bf16 [M, zero_cols], optional) are cleared here.
__device__ inline void route_groups_block(const int32_t* __restrict__ group_sizes, uint32_t M, uint32_t n_groups,
                                          uint32_t slots, int32_t* __restrict__ src_row,
                                          int32_t* __restrict__ blk_range,
                                          uint64_t* __restrict__ tile_tab, uint32_t tile_blocks, uint16_t* __restrict__ zero_out, uint32_t zero_cols,
                                          uint32_t part, uint32_t n_parts) {
  __shared__ uint32_t row_start[kMaxGroups + 1];
  __shared__ uint32_t slot_start[kMaxGroups + 1];
  const uint32_t tid = threadIdx.x;
  int32_t sz = tid < n_groups ? group_sizes[tid] : 0;
  if (sz < 0) sz = 0;
  uint32_t row[1] = {(uint32_t)sz}, rows_of_all[1];
  block_prefix_capped(row, M, rows_of_all);
  const uint32_t r0 = row[0], rows_total = rows_of_all[0];
  // the group's rows after the cap: up to the next group's start
  const uint32_t r1 = (uint64_t)r0 + (uint32_t)sz > M ? M : r0 + (uint32_t)sz;
  const uint32_t nblk = (r1 - r0 + 31u) / 32u;
  const uint32_t n_tiles = (nblk + tile_blocks - 1u) / tile_blocks;
  uint32_t place[2] = {nblk * 32u, n_tiles}, all[2];
  block_prefix_capped(place, 0xffffffffu, all);
  const uint32_t p0 = place[0], slots_total = all[0], t0 = place[1], tiles_total = all[1];
  if (part == 0 && tid == 0) tile_tab[0] = tiles_total;
  for (uint32_t i = part; i < n_tiles; i += n_parts) {
    const uint32_t low = nblk / n_tiles, high = nblk % n_tiles;  // the first `high` tiles have a block more
    const uint32_t first = i * low + (i < high ? i : high), count = low + (i < high ? 1u : 0u);
    tile_tab[1u + t0 + i] = (uint64_t)(p0 / 32u + first) | (uint64_t)count << 32 | (uint64_t)tid << 48;
  }
  if (tid < n_groups) { row_start[tid] = r0; slot_start[tid] = p0; }
  if (tid == 0) { row_start[n_groups] = rows_total; slot_start[n_groups] = slots_total; }
  __syncthreads();
  const uint32_t stride = n_parts * 1024u;
  for (uint32_t p = part * 1024u + tid; p < slots; p += stride) {
    int src = -1, range = -1;
    if (p < slots_total) {
      // the last group whose first slot is not behind p (empty groups share their successor's first slot)
      uint32_t lo = 0, hi = n_groups;  // slot_start[lo] <= p < slot_start[hi]
      while (hi - lo > 1u) {
        const uint32_t mid = (lo + hi) >> 1;
        if (slot_start[mid] <= p) lo = mid; else hi = mid;
      }
      const uint32_t i = p - slot_start[lo];
      if (i < row_start[lo + 1u] - row_start[lo]) src = (int)(row_start[lo] + i);
      range = (int)(lo | (lo << 16));
    }
    src_row[p] = src;
    if ((p & 31u) == 0) blk_range[p >> 5] = range;
  }
  if (zero_out) {
    const size_t begin = (size_t)rows_total * zero_cols, end = (size_t)M * zero_cols;
    for (size_t i = begin + part * 1024u + tid; i < end; i += stride) zero_out[i] = 0;
  }
}

// ---------------------------------------------------------------------------------------
// Per-token dynamic int8 quantization (skyrl/tx/kernels/quantized_lora.py:199-212 with one
// group per row), row-major: the public row quantizer, and the rows of a grouped call that have no slot.  One
// wave per row; the row lives in registers (NCH chunks of 8 bf16 per lane).  Bit-exact rules, of every quantizer here:
//   scale = amax > 0 ? amax / 127 : 1         IEEE float32 division
//   code  = clamp(rint(v / scale), -127, 127) IEEE division, round half to even
//   RMSNorm (skyrl/tx/kernels/rocm/bf16_rms_gate_up_lora_swiglu.py:299-303): mean = float(sum_f64(x*x) / K),
//            inv = 1 / sqrt(mean + eps) (IEEE), and n = bf16((x * inv) * gamma) with two separate float32
//            multiplications.
// ---------------------------------------------------------------------------------------
struct QuantArgs {
  const uint16_t* x;       // bf16 [M, K]
  uint32_t M, K;
  int8_t* codes_rm;        // row-major codes [M, K] or null
  float* scales_rm;        // f32 [M] or null
  // Optional gather on the way in: row m is read from x[row_map[m] / row_div] (the sorted (token,
  // choice) pairs of an expert layer read their token's row; x then has the tokens' row count,
  // row_limit, to which the source row is clamped)
  const int32_t* row_map;
  uint32_t row_div, row_limit;
};

// source row of a gathered read: map value / divisor, clamped into [0, limit)
__device__ inline uint32_t mapped_row(int32_t value, uint32_t div, uint32_t limit) {
  const uint32_t r = value < 0 ? 0u : (uint32_t)value / div;
  return r < limit ? r : limit - 1u;
}

template <int NCH>
__global__ __launch_bounds__(256) void quant_rows_kernel(QuantArgs a) {
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t m = blockIdx.x * 4u + (threadIdx.x >> 6);
  if (m >= a.M) return;
  const uint32_t xrow = a.row_map ? mapped_row(a.row_map[m], a.row_div, a.row_limit) : m;
  const uint16_t* xr = a.x + (size_t)xrow * a.K;
  float v[NCH][8];
#pragma unroll
  for (int j = 0; j < NCH; ++j) {
    uint32_t k0 = (j * 64u + lane) * 8u;
    uint4 raw = make_uint4(0, 0, 0, 0);
    if (k0 < a.K) raw = *reinterpret_cast<const uint4*>(xr + k0);
    uint32_t w[4] = {raw.x, raw.y, raw.z, raw.w};
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      v[j][2 * e] = __uint_as_float(w[e] << 16);
      v[j][2 * e + 1] = __uint_as_float(w[e] & 0xffff0000u);
    }
  }
  float amax = 0.0f;
#pragma unroll
  for (int j = 0; j < NCH; ++j)
#pragma unroll
    for (int e = 0; e < 8; ++e) amax = fmaxf(amax, fabsf(v[j][e]));
  amax = wave_max(amax);
  const float scale = amax > 0.0f ? amax / 127.0f : 1.0f;
  if (lane == 0 && a.scales_rm) a.scales_rm[m] = scale;
  if (!a.codes_rm) return;
  // codes = rint(v / scale) with the correctly rounded quotient, as in quant_lora_kernel: v * (1 / scale)
  // with the hardware reciprocal rounds to the same integer unless the product lies within 1e-4 of a
  // tie; those cases (and scales outside the reciprocal's safe range) are redone with the division.
  const float rscale = __builtin_amdgcn_rcpf(scale);
  const bool scale_safe = scale > 1e-30f && scale < 1e30f;
#pragma unroll
  for (int j = 0; j < NCH; ++j) {
    const uint32_t k0 = (j * 64u + lane) * 8u;
    if (k0 >= a.K) continue;
    uint32_t lo = 0, hi = 0;
    float q[8];
    float off_integer = 0.0f;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float t = v[j][e] * rscale;
      q[e] = rintf(t);
      off_integer = fmaxf(off_integer, fabsf(t - q[e]));
    }
    if (!scale_safe || off_integer > 0.4999f) {
#pragma unroll
      for (int e = 0; e < 8; ++e) q[e] = rintf(v[j][e] / scale);
    }
    // q is an integer in [-127, 127] (|v| <= the row's absmax): q + 128 lands in its byte with one
    // v_cvt_pk_u8_f32, and flipping bit 7 of every byte turns the biased value into two's complement
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      lo = __builtin_amdgcn_cvt_pk_u8_f32(q[e] + 128.0f, (uint32_t)e, lo);
      hi = __builtin_amdgcn_cvt_pk_u8_f32(q[e + 4] + 128.0f, (uint32_t)e, hi);
    }
    lo ^= 0x80808080u;
    hi ^= 0x80808080u;
    *reinterpret_cast<uint2*>(a.codes_rm + (size_t)m * a.K + k0) = make_uint2(lo, hi);
  }
}

// ---------------------------------------------------------------------------------------
// LoRA A re-layout: A [n, K, r] (rank contiguous) -> At [n, r, K] (K contiguous), so that an
// MFMA operand (8 consecutive k of one rank column) is one 16-byte load.  LoRA parameters
// are trainable and may change between calls, so this runs per call; it moves n*K*r*2 bytes.
// ---------------------------------------------------------------------------------------
__device__ inline void lora_a_transpose_item(const uint16_t* __restrict__ a, uint16_t* __restrict__ at,
                                             uint32_t n_groups, uint32_t K, uint32_t r, uint64_t idx) {
  const uint32_t rc = (r + 7u) / 8u;  // 8-wide rank chunks per k
  const uint64_t total = (uint64_t)n_groups * K * rc;
  if (idx >= total) return;
  const uint32_t ch = (uint32_t)(idx % rc);
  const uint64_t gk = idx / rc;  // group * K + k
  const uint32_t k = (uint32_t)(gk % K);
  const uint32_t grp = (uint32_t)(gk / K);
  const uint16_t* src = a + gk * r + ch * 8u;
  uint16_t v[8];
  if ((r & 7u) == 0) {
    const v8us w = *reinterpret_cast<const v8us*>(src);
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = w[e];
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = (ch * 8u + e < r) ? src[e] : (uint16_t)0;
  }
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const uint32_t col = ch * 8u + e;
    if (col < r) at[((size_t)grp * r + col) * K + k] = v[e];
  }
}

// ---------------------------------------------------------------------------------------
// LoRA B re-layout: B [n, r, N] -> MFMA B-operand order bp[n][N_pad/32][nkk][64 lanes][8]:
// lane (c = l % 32, h = l / 32) of packed column block cb holds rows 16 kk + 8 h + 0..7 (zero
// beyond the rank) of the original column packed_to_orig_col(32 cb + c) (zero beyond N).
// Like A^T this runs per call because LoRA parameters are trainable.
// ---------------------------------------------------------------------------------------
__device__ inline void lora_b_pack_item(const uint16_t* __restrict__ b, unsigned char* __restrict__ bp,
                                        uint32_t n_groups, uint32_t r, uint32_t N, uint32_t ncb, uint32_t nkk,
                                        uint64_t idx) {
  const uint64_t total = (uint64_t)n_groups * ncb * nkk * 64u;  // one 16-byte operand per thread
  if (idx >= total) return;
  const uint32_t l = (uint32_t)(idx & 63u);
  const uint64_t rest = idx >> 6;
  const uint32_t kk = (uint32_t)(rest % nkk);
  const uint64_t gc = rest / nkk;
  const uint32_t cb = (uint32_t)(gc % ncb), grp = (uint32_t)(gc / ncb);
  const uint32_t col = packed_to_orig_col(cb * 32u + (l & 31u));
  v8us o;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const uint32_t row = 16u * kk + 8u * (l >> 5) + e;
    const bool in = col < N && row < r;
    const uint16_t v = b[in ? ((size_t)grp * r + row) * N + col : 0u];
    o[e] = in ? v : (uint16_t)0;
  }
  *reinterpret_cast<v8us*>(bp + idx * 16u) = o;
}
// Four operands per thread where a row's columns come in aligned fours (N % 4 == 0): the lane's column of each
// of a group's four column blocks, four adjacent columns of B, so a quarter of the loads.  The packing is
// bound by the loads it issues: 8 adapters of rank 32 at 4096 -> 24576 take 6 us where one two-byte load per
// value takes 20.
__device__ inline void lora_b_pack4_item(const uint16_t* __restrict__ b, unsigned char* __restrict__ bp,
                                         uint32_t n_groups, uint32_t r, uint32_t N, uint32_t ncb, uint32_t nkk,
                                         uint64_t idx) {
  const uint64_t total = (uint64_t)n_groups * (ncb / 4u) * nkk * 64u;
  if (idx >= total) return;
  const uint32_t l = (uint32_t)(idx & 63u);
  const uint64_t rest = idx >> 6;
  const uint32_t kk = (uint32_t)(rest % nkk);
  const uint64_t gc = rest / nkk;
  const uint32_t G = (uint32_t)(gc % (ncb / 4u)), grp = (uint32_t)(gc / (ncb / 4u));
  const uint32_t col = 128u * G + 4u * (l & 31u), row0 = 16u * kk + 8u * (l >> 5);
  v8us o[4];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const bool in = col < N && row0 + e < r;
    // (loaded whatever the condition: a load under a lane condition becomes a branch with a wait of its own)
    const uint2 v = *reinterpret_cast<const uint2*>(b + (in ? ((size_t)grp * r + row0 + e) * N + col : 0u));
    const uint32_t vx = in ? v.x : 0u, vy = in ? v.y : 0u;
    o[0][e] = (uint16_t)vx; o[1][e] = (uint16_t)(vx >> 16);
    o[2][e] = (uint16_t)vy; o[3][e] = (uint16_t)(vy >> 16);
  }
#pragma unroll
  for (uint32_t j = 0; j < 4; ++j)
    *reinterpret_cast<v8us*>(bp + ((((size_t)grp * ncb + 4u * G + j) * nkk + kk) * 64u + l) * 16u) = o[j];
}


// ---------------------------------------------------------------------------------------
// LoRA A re-layout for the dense path's quantizer: A [n, K, r] -> the B-operand order of
// v_mfma_f32_16x16x32_bf16, ap[n][K_pad/32][nkk][64 lanes][8]: lane (i = l % 16, q = l / 16) of
// k-block kb and rank block b holds k = 32 kb + 8 q + 0..7 (zero beyond K) of rank column
// 16 b + i (zero beyond the rank).  A wave's operand load is then 1 KiB of consecutive memory
// (eight cache lines) where the transposed layout gives it sixteen half-used lines, and the
// quantizer's LoRA-A step is bound by the cache lines its loads touch.
// ---------------------------------------------------------------------------------------
__device__ inline void lora_a_pack_item(const uint16_t* __restrict__ a, unsigned char* __restrict__ ap,
                                        uint32_t n_groups, uint32_t K, uint32_t r, uint32_t KB, uint32_t nkk,
                                        uint64_t idx) {
  const uint64_t total = (uint64_t)n_groups * KB * nkk * 64u;  // one 16-byte operand per thread
  if (idx >= total) return;
  const uint32_t l = (uint32_t)(idx & 63u);
  const uint64_t rest = idx >> 6;
  const uint32_t b = (uint32_t)(rest % nkk);
  const uint64_t gk = rest / nkk;
  const uint32_t kb = (uint32_t)(gk % KB), grp = (uint32_t)(gk / KB);
  const uint32_t col = 16u * b + (l & 15u);
  v8us o;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const uint32_t k = 32u * kb + 8u * (l >> 4) + e;
    const bool in = col < r && k < K;
    const uint16_t v = a[in ? ((size_t)grp * K + k) * r + col : 0u];
    o[e] = in ? v : (uint16_t)0;
  }
  *reinterpret_cast<v8us*>(ap + idx * 16u) = o;
}

// Four operands per thread (r % 4 == 0): four adjacent rank columns of the same eight k.
__device__ inline void lora_a_pack4_item(const uint16_t* __restrict__ a, unsigned char* __restrict__ ap,
                                         uint32_t n_groups, uint32_t K, uint32_t r, uint32_t KB, uint32_t nkk,
                                         uint64_t idx) {
  const uint64_t total = (uint64_t)n_groups * KB * nkk * 16u;
  if (idx >= total) return;
  const uint32_t i4 = (uint32_t)(idx & 3u), q = (uint32_t)(idx >> 2) & 3u;
  const uint64_t rest = idx >> 4;
  const uint32_t b = (uint32_t)(rest % nkk);
  const uint64_t gk = rest / nkk;
  const uint32_t kb = (uint32_t)(gk % KB), grp = (uint32_t)(gk / KB);
  const uint32_t col = 16u * b + 4u * i4, k0 = 32u * kb + 8u * q;
  v8us o[4];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const bool in = col < r && k0 + e < K;
    const uint2 v = *reinterpret_cast<const uint2*>(a + (in ? ((size_t)grp * K + k0 + e) * r + col : 0u));
    const uint32_t vx = in ? v.x : 0u, vy = in ? v.y : 0u;
    o[0][e] = (uint16_t)vx; o[1][e] = (uint16_t)(vx >> 16);
    o[2][e] = (uint16_t)vy; o[3][e] = (uint16_t)(vy >> 16);
  }
  v8us* dst = reinterpret_cast<v8us*>(ap) + (rest * 64u + 16u * q + 4u * i4);
#pragma unroll
  for (uint32_t j = 0; j < 4; ++j) dst[j] = o[j];
}

// The same for lora_a_kernel (v_mfma_f32_32x32x16_bf16, 64-wide k steps), whose operand loads of the
// transposed A touch 32 cache lines each:
// ap[n][ceil(K / 64)][RB][4][64 lanes][8]: lane (i = l % 32, h = l / 32) of k step s, rank block b and
// quarter t holds k = 64 s + 32 h + 8 t + 0..7 of rank column 32 b + i.  Pays with few adapters of many
// rows each; with 128 experts of rank 16 (padded to 32 columns, packed per call) it measured slower.
__device__ inline void lora_a_pack32_item(const uint16_t* __restrict__ a, unsigned char* __restrict__ ap,
                                          uint32_t n_groups, uint32_t K, uint32_t r, uint32_t n_steps, uint32_t rb,
                                          uint64_t idx) {
  const uint64_t total = (uint64_t)n_groups * n_steps * rb * 256u;  // one 16-byte operand per thread
  if (idx >= total) return;
  const uint32_t l = (uint32_t)(idx & 63u), t = (uint32_t)(idx >> 6) & 3u;
  const uint64_t rest = idx >> 8;
  const uint32_t b = (uint32_t)(rest % rb);
  const uint64_t gs = rest / rb;
  const uint32_t st = (uint32_t)(gs % n_steps), grp = (uint32_t)(gs / n_steps);
  const uint32_t col = 32u * b + (l & 31u);
  v8us o;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const uint32_t k = 64u * st + 32u * (l >> 5) + 8u * t + e;
    const bool in = col < r && k < K;
    const uint16_t v = a[in ? ((size_t)grp * K + k) * r + col : 0u];
    o[e] = in ? v : (uint16_t)0;
  }
  *reinterpret_cast<v8us*>(ap + idx * 16u) = o;
}

// Clears `count` 32-bit words (one workgroup).
__global__ __launch_bounds__(256) void zero_words_kernel(uint32_t* p, uint32_t count) {
  for (uint32_t i = threadIdx.x; i < count; i += 256u) p[i] = 0u;
}

// ---------------------------------------------------------------------------------------
// One launch for the independent preparation jobs of a call: adapter routing (block 0
// when `idx` is given), the rows' statistics (dense calls), LoRA A and LoRA B in operand order
// (the other blocks).
// ---------------------------------------------------------------------------------------
struct LoraPrepArgs {
  const int32_t* idx;        // adapter per row, or null (no routing block)
  int32_t* src_row; int32_t* dst_pos; int32_t* slot_group; int32_t* blk_range;
  const uint16_t* lora_a;    // bf16 [n_groups, K, r]
  const uint16_t* lora_b;    // bf16 [n_groups, r, N]
  uint16_t* at;              // A in operand order
  unsigned char* bp;         // packed B operands
  uint32_t M, K, N, n_groups, r, nkk, ncb, slots, route_blocks, a_blocks;
  uint32_t rows_per_index;   // rows that an entry of idx serves (0 or 1: one)
  uint32_t route_pad;        // dense routing block: every group's first slot is a multiple of this (0 or 1: packed)
  uint32_t a_operand_kb;     // K_pad / 32: the quantizer's operand order (lora_a_pack_item) ...
  uint32_t a_operand_steps, a_operand_rb;  // ... or ceil(K / 64) and the 32-wide rank blocks of lora_a_kernel's (lora_a_pack32_item)
  // grouped (ragged) call: the routing block lays the groups out from their sizes instead
  const int32_t* group_sizes;  // int32 [n_groups] or null
  uint64_t* tile_tab;          // row tiles of the grouped GEMM ...
  uint32_t tile_blocks;        // ... and the 32-row blocks they hold at most
  uint16_t* zero_out;          // bf16 [M, zero_cols]: rows beyond the groups are cleared, or null
  uint32_t zero_cols;
  // row statistics (STATS != 0): sixteen rows per block, behind the routing block
  uint32_t stat_blocks, stat_rows;
  const int32_t* stat_map;     // statistics of row m are those of source row mapped_row(stat_map[m], ...), or null
  uint32_t stat_div, stat_limit;
  const uint16_t* x;           // bf16 [M, K]
  const float* gamma;          // f32 [K] (STATS == 2)
  float eps;
  float* row_scale;            // f32 [M]: absmax / 127 of the (normalized) row, 1 where that is not positive
  float* row_inv;              // f32 [M]: 1 / sqrt(mean square + eps) (STATS == 2)
  float* scales_rm;            // f32 [M] for the caller, or null
  uint16_t* xn_aux;            // bf16 [M, K] normalized rows for the caller, or null (STATS == 2)
};

// (x * inv) * gamma, one bf16 rounding, of eight values
__device__ inline uint4 rms_normalize8(const uint4& raw, float inv, const float4& g0, const float4& g1) {
  const float g[8] = {g0.x, g0.y, g0.z, g0.w, g1.x, g1.y, g1.z, g1.w};
  uint32_t w[4] = {raw.x, raw.y, raw.z, raw.w};
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    float t0 = __uint_as_float(w[e] << 16) * inv, t1 = __uint_as_float(w[e] & 0xffff0000u) * inv;
    t0 = t0 * g[2 * e];
    t1 = t1 * g[2 * e + 1];
    w[e] = pack_bf16x2(t0, t1);
  }
  return make_uint4(w[0], w[1], w[2], w[3]);
}

// The scale of a row from its wave's running maxima.
__device__ inline float row_scale_of(uint32_t amax_bits) {
  uint32_t top = (amax_bits >> 16) > (amax_bits & 0xffffu) ? (amax_bits >> 16) : (amax_bits & 0xffffu);
  top = wave_fold(top, [](uint32_t a, uint32_t b) { return a > b ? a : b; });
  const float amax = __uint_as_float(top << 16);
  return amax > 0.0f ? amax / 127.0f : 1.0f;
}

// Statistics of row m by one wave: kPieces 1 KiB pieces of the row in flight at a time.  With RMSNorm the row
// is read a second time for the normalized maximum (from the L2: its wave has just read it); holding it took
// registers that cost the launch its second workgroup per CU.
template <bool RMS>
__device__ inline void row_stats(const LoraPrepArgs& p, uint32_t m) {
  constexpr uint32_t kPieces = RMS ? 4 : 8;
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t row_bytes = 2u * p.K;
  const uint32_t xrow = p.stat_map ? mapped_row(p.stat_map[m], p.stat_div, p.stat_limit) : m;
  // (the row and the norm weights through buffer resources that end with them: a load under a lane condition
  // becomes a branch with a wait of its own, and the loads then run one after the other)
  const __amdgpu_buffer_rsrc_t xrsrc =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(p.x) + (size_t)xrow * p.K, 0, (int)row_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t grsrc =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p.gamma), 0, RMS ? (int)(p.K * 4u) : 0, 0x00020000);
  uint32_t amax_bits = 0;
  uint4 r[kPieces];
  auto fetch = [&](uint32_t base) {
#pragma unroll
    for (uint32_t j = 0; j < kPieces; ++j)
      r[j] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(xrsrc, base + j * 1024u + lane * 16u, 0, 0));
  };
  if constexpr (!RMS) {
#pragma unroll 1
    for (uint32_t base = 0; base < row_bytes; base += kPieces * 1024u) {
      fetch(base);
#pragma unroll
      for (uint32_t j = 0; j < kPieces; ++j) amax_bits = bf16_absmax_pairs(amax_bits, r[j]);
    }
  } else {
    double ss = 0.0;
#pragma unroll 1
    for (uint32_t base = 0; base < row_bytes; base += kPieces * 1024u) {
      fetch(base);
#pragma unroll
      for (uint32_t j = 0; j < kPieces; ++j) {
        const uint32_t w[4] = {r[j].x, r[j].y, r[j].z, r[j].w};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          // the square of a bf16 value is exact in double, so the fused form rounds like mul + add
          const double lo = (double)__uint_as_float(w[e] << 16), hi = (double)__uint_as_float(w[e] & 0xffff0000u);
          ss = __builtin_fma(lo, lo, ss);
          ss = __builtin_fma(hi, hi, ss);
        }
      }
    }
    ss = wave_sum(ss);
    const float var = (float)(ss / (double)p.K);
    const float inv = 1.0f / sqrtf(var + p.eps);
    if (lane == 0) p.row_inv[m] = inv;
#pragma unroll 1
    for (uint32_t base = 0; base < row_bytes; base += kPieces * 1024u) {
      fetch(base);
#pragma unroll
      for (uint32_t j = 0; j < kPieces; ++j) {
        const uint32_t off = base + j * 1024u + lane * 16u;
        if ((j & 1u) == 0) __builtin_amdgcn_sched_barrier(0);  // (norm weights of two pieces at a time: registers)
        const float4 g0 = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(grsrc, 2u * off, 0, 0));
        const float4 g1 = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(grsrc, 2u * off + 16u, 0, 0));
        const uint4 n = rms_normalize8(r[j], inv, g0, g1);  // (zeros beyond the row)
        if (p.xn_aux && off < row_bytes) *reinterpret_cast<uint4*>(reinterpret_cast<unsigned char*>(p.xn_aux) + (size_t)m * row_bytes + off) = n;
        amax_bits = bf16_absmax_pairs(amax_bits, n);
      }
    }
  }
  const float scale = row_scale_of(amax_bits);
  if (lane == 0) {
    p.row_scale[m] = scale;
    if (p.scales_rm) p.scales_rm[m] = scale;
  }
}

// (Two workgroups per CU: 4096 rows are 256 blocks of statistics, and the routing block beside them must not
// put one of them into a second round.)
// (Aligned so that its 20 KB of instructions lie within 64 KiB: across such a line the launch took 6.4 us instead of 5.95 at 333 rows, 4096 -> 2560, 4
// adapters of rank 64, in the same code.)
template <int STATS>  // 0: no row statistics, 1: of x, 2: of the normalized rows
__global__ __launch_bounds__(1024, 8) __attribute__((aligned(32768))) void lora_prep_kernel(LoraPrepArgs p) {
  uint32_t b = blockIdx.x;
  if (b < p.route_blocks) {
    __builtin_amdgcn_s_setprio(3);  // a chain of short steps beside waves that wait for memory
    if (p.group_sizes)
      route_groups_block(p.group_sizes, p.M, p.n_groups, p.slots, p.src_row, p.blk_range, p.tile_tab,
                         p.tile_blocks, p.zero_out, p.zero_cols, b, p.route_blocks);
    else
      route_rows_block(p.idx, p.M, p.n_groups, p.slots, p.src_row, p.dst_pos, p.slot_group, p.blk_range, nullptr,
                       p.route_pad > 1u ? p.route_pad : 1u, p.rows_per_index);
    return;
  }
  b -= p.route_blocks;
  if constexpr (STATS != 0) {
    if (b < p.stat_blocks) {
      const uint32_t m = b * 16u + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
      if (m < p.stat_rows) row_stats<STATS == 2>(p, m);
      return;
    }
    b -= p.stat_blocks;
  }
  if (b < p.a_blocks) {
    if (p.a_operand_steps)
      lora_a_pack32_item(p.lora_a, reinterpret_cast<unsigned char*>(p.at), p.n_groups, p.K, p.r, p.a_operand_steps,
                         p.a_operand_rb, (uint64_t)b * 1024u + threadIdx.x);
    else if ((p.r & 3u) == 0)
      lora_a_pack4_item(p.lora_a, reinterpret_cast<unsigned char*>(p.at), p.n_groups, p.K, p.r, p.a_operand_kb, p.nkk,
                        (uint64_t)b * 1024u + threadIdx.x);
    else
      lora_a_pack_item(p.lora_a, reinterpret_cast<unsigned char*>(p.at), p.n_groups, p.K, p.r, p.a_operand_kb, p.nkk,
                       (uint64_t)b * 1024u + threadIdx.x);
    return;
  }
  b -= p.a_blocks;
  if ((p.N & 3u) == 0)
    lora_b_pack4_item(p.lora_b, p.bp, p.n_groups, p.r, p.N, p.ncb, p.nkk, (uint64_t)b * 1024u + threadIdx.x);
  else
    lora_b_pack_item(p.lora_b, p.bp, p.n_groups, p.r, p.N, p.ncb, p.nkk, (uint64_t)b * 1024u + threadIdx.x);
}

// ---------------------------------------------------------------------------------------
// LoRA-A projection on bf16 MFMA: z[p, :] = n[src_row[p], :] @ A[group(p)]  (float32
// accumulation of exact bf16 products; skyrl/tx/kernels/quantized_lora.py:300-301 and
// skyrl/tx/layers/lora.py:150), of the backward and of the group-scaled call.  One workgroup of 16 waves per
// 32-row block and slice of K; the waves take disjoint K ranges and are reduced through LDS in a fixed order.
// ---------------------------------------------------------------------------------------
struct LoraAArgs {
  const uint16_t* xsrc;     // bf16 [M, K] (x, or the normalized rows)
  const uint16_t* at;       // bf16 [n_groups, r, K], or A in operand order (lora_a_pack32_item) when at_operand is set
  uint32_t at_operand;      // 0 or 1
  const int32_t* src_row;   // or null (identity)
  const int32_t* slot_group;// or null (group 0)
  const int32_t* blk_range; // or null
  uint32_t M, K, r, steps_per_wave, n_steps, n_blocks;
  float* zf; uint32_t zf_stride;  // the projection, [slot][zf_stride]
  // K split: with n_ksplit > 1 the grid holds n_ksplit workgroups per row block, each
  // sums its own range of k steps and writes zf + ksplit_index * zf_slice (floats); the caller adds
  // the slices.  0 or 1: one workgroup per row block.
  uint32_t n_ksplit, zf_slice;
};

// STAGED (RB = 1, the transposed A; with or without the K split): the operands of a k step travel through 8 KiB of LDS
// per wave.  A register load of an MFMA operand touches 32 cache lines of 32 used bytes, which the
// vector memory path delivers at a third of the rate of whole lines; a direct-to-LDS load in which
// eight lanes fetch one 128-byte line (of a row of x, of a rank column of A) moves eight whole lines,
// and the operands are then read from LDS (line pieces XOR-swizzled by the row, so that eight lanes
// never share a bank).  Which wave adds which k step, and in which order, does not change.
constexpr uint32_t kLoraAStageBytes = 16u * 8192u;
template <int RB, bool STAGED = false>  // RB: number of 32-wide rank blocks (1 or 2)
__global__ __launch_bounds__(1024) void lora_a_kernel(LoraAArgs a) {
  static_assert(!STAGED || RB == 1, "the staged form holds one rank block");
  __shared__ float red[4][RB][16][64];
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
  const uint32_t nks = a.n_ksplit > 1u ? a.n_ksplit : 1u;
  const uint32_t pb = blockIdx.x / nks, ks = blockIdx.x % nks;
  if (pb >= a.n_blocks) return;
  if (a.blk_range && a.blk_range[pb] < 0) return;  // block beyond the rows in use
  const uint32_t range = a.blk_range ? (uint32_t)a.blk_range[pb] : 0u;
  const uint32_t glo = range & 0xffffu, ghi = range >> 16;
  const uint32_t i = lane & 31u, h = lane >> 5;
  const uint32_t p = pb * 32u + i;
  int src = a.src_row ? a.src_row[p] : (int)p;
  if (src >= (int)a.M) src = -1;
  const uint32_t rowgrp = (a.slot_group && ghi > glo) ? (uint32_t)a.slot_group[p] : glo;
  const uint16_t* xr = a.xsrc + (size_t)(src < 0 ? 0 : src) * a.K;
  v16f acc[RB];
#pragma unroll
  for (int b = 0; b < RB; ++b)
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[b][e] = 0.0f;
  const uint32_t slice_steps = (a.n_steps + nks - 1u) / nks;
  const uint32_t slice_end = (ks + 1u) * slice_steps < a.n_steps ? (ks + 1u) * slice_steps : a.n_steps;
  uint32_t s0 = ks * slice_steps + wave * a.steps_per_wave, s1 = s0 + a.steps_per_wave;
  if (s1 > slice_end) s1 = slice_end;
  if constexpr (STAGED) {
    extern __shared__ __attribute__((aligned(1024))) unsigned char stage_lds[];
    unsigned char* const my = stage_lds + wave * 8192u;  // x lines at 0, A lines at 4096
    // lane l fetches, for j = 0..3, piece (l % 8) ^ (l / 8) of the 128-byte line of row / column 8 j + l / 8
    const uint32_t r8 = lane >> 3, piece = (lane & 7u) ^ r8;
    const uint16_t* xrow[4];
#pragma unroll
    for (uint32_t j = 0; j < 4; ++j) {
      const uint32_t pj = pb * 32u + 8u * j + r8;
      int sj = a.src_row ? a.src_row[pj] : (int)pj;
      if (sj >= (int)a.M) sj = -1;
      xrow[j] = a.xsrc + (size_t)(sj < 0 ? 0 : sj) * a.K;
    }
    // where lane (i, h) finds quarter t of its operand: line i, piece 4 h + t
    const uint32_t rd = (i >> 3) * 1024u + (i & 7u) * 128u;
    for (uint32_t grp = glo; grp <= ghi; ++grp) {
      const bool mine = src >= 0 && rowgrp == grp;
      const uint16_t* atg = a.at + (size_t)grp * a.r * a.K;
      for (uint32_t s = s0; s < s1; ++s) {
        uint32_t kp = s * 64u + piece * 8u;
        if (kp >= a.K) kp = 0;  // a piece beyond K: any address inside the row; it is zeroed where it is used
#pragma unroll
        for (uint32_t j = 0; j < 4; ++j)
          load_1k_to_lds(reinterpret_cast<const unsigned char*>(xrow[j] + kp), my + j * 1024u);
        v8us xa[4], wb[4];
        if (a.at_operand) {  // kernel-uniform: A already lies in operand order (zero beyond K and the rank)
#pragma unroll
          for (uint32_t t = 0; t < 4; ++t)
            wb[t] = *(reinterpret_cast<const v8us*>(a.at) + (((size_t)grp * a.n_steps + s) * 4u + t) * 64u + lane);
        } else {
#pragma unroll
          for (uint32_t j = 0; j < 4; ++j) {
            uint32_t col = 8u * j + r8;
            if (col >= a.r) col = 0;
            load_1k_to_lds(reinterpret_cast<const unsigned char*>(atg + (size_t)col * a.K + kp), my + 4096u + j * 1024u);
          }
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
        for (uint32_t t = 0; t < 4; ++t) {
          const uint32_t off = rd + (((4u * h + t) ^ (i & 7u)) * 16u);
          const v8us zero = {0, 0, 0, 0, 0, 0, 0, 0};
          const bool ok = s * 64u + 32u * h + 8u * t < a.K;
          const v8us xv = *reinterpret_cast<const v8us*>(my + off);
          xa[t] = (mine && ok) ? xv : zero;
          if (!a.at_operand) {
            const v8us wv = *reinterpret_cast<const v8us*>(my + 4096u + off);
            wb[t] = (i < a.r && ok) ? wv : zero;
          }
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the lines are read before the next step's loads land on them
#pragma unroll
        for (int t = 0; t < 4; ++t)
          acc[0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8bf, xa[t]), __builtin_bit_cast(v8bf, wb[t]),
                                                           acc[0], 0, 0, 0);
      }
    }
  } else
  // A block at a group boundary runs once per group with the other groups' rows zeroed.
  for (uint32_t grp = glo; grp <= ghi; ++grp) {
    const bool mine = src >= 0 && rowgrp == grp;
    const uint16_t* atg = a.at + (size_t)grp * a.r * a.K;
    // U 64-wide k steps per iteration: all their operand loads go out before the MFMAs
    constexpr int U = RB == 1 ? 2 : 1;  // 1024 threads leave 128 registers per lane
    for (uint32_t s = s0; s < s1; s += U) {
      v8us xa[U][4], wb[U][RB][4];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const uint32_t kbase = (s + u) * 64u + 32u * h;
        const bool step_ok = (s + u) < s1;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          const uint32_t k0 = kbase + 8u * t;
          const v8us zero = {0, 0, 0, 0, 0, 0, 0, 0};
          const bool ok = step_ok && k0 < a.K;
          xa[u][t] = (mine && ok) ? *reinterpret_cast<const v8us*>(xr + k0) : zero;
#pragma unroll
          for (int b = 0; b < RB; ++b) {
            const uint32_t col = b * 32u + i;
            if (a.at_operand)  // kernel-uniform: 1 KiB of consecutive memory per wave and load (zero beyond K and the rank)
              wb[u][b][t] = step_ok ? *(reinterpret_cast<const v8us*>(a.at) +
                                        ((((size_t)grp * a.n_steps + (s + u)) * RB + b) * 4u + t) * 64u + lane)
                                    : zero;
            else
              wb[u][b][t] = (col < a.r && ok) ? *reinterpret_cast<const v8us*>(atg + (size_t)col * a.K + k0) : zero;
          }
        }
      }
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
          for (int b = 0; b < RB; ++b)
            acc[b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8bf, xa[u][t]),
                                                             __builtin_bit_cast(v8bf, wb[u][b][t]), acc[b], 0, 0, 0);
    }
  }
  // fixed-order reduction over the 16 waves: waves 4..7, 8..11, 12..15 are added, in that order,
  // onto waves 0..3, whose four partial sums are then added in wave order
  for (uint32_t round = 1; round < 4; ++round) {
    if ((wave >> 2) == round) {
#pragma unroll
      for (int b = 0; b < RB; ++b)
#pragma unroll
        for (int e = 0; e < 16; ++e) red[wave & 3u][b][e][lane] = acc[b][e];
    }
    __syncthreads();
    if (wave < 4) {
#pragma unroll
      for (int b = 0; b < RB; ++b)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[b][e] = acc[b][e] + red[wave][b][e][lane];
    }
    __syncthreads();
  }
  if (wave < 4) {
#pragma unroll
    for (int b = 0; b < RB; ++b)
#pragma unroll
      for (int e = 0; e < 16; ++e) red[wave][b][e][lane] = acc[b][e];
  }
  __syncthreads();
  for (uint32_t q = threadIdx.x; q < RB * 1024u; q += 1024u) {
    const uint32_t l = q & 63u, e = (q >> 6) & 15u, b = q >> 10;
    float sum = red[0][b][e][l];
#pragma unroll
    for (int w = 1; w < 4; ++w) sum += red[w][b][e][l];
    const uint32_t row = 8u * (e >> 2) + 4u * (l >> 5) + (e & 3u), col = b * 32u + (l & 31u);
    a.zf[(size_t)ks * a.zf_slice + (size_t)(pb * 32u + row) * a.zf_stride + col] = sum;
  }
}

// ---------------------------------------------------------------------------------------
// Codes and LoRA-A projection of the dense path's prologue, behind the launch that took the rows'
// statistics (row_stats, beside the routing and the LoRA operand layouts).
// One workgroup of 16 waves per half of a 32-slot block: the waves split K in 32-wide blocks; lane
// (i = lane % 16, q = lane / 16) takes the 8 (normalized) values k = 32 kb + 8 q .. +7 of slot row i and
// uses them twice: as int8 codes written into the activation's 1 KiB fragment block, and as the A operand
// of v_mfma_f32_16x16x32_bf16 against the LoRA A of the row's group in that instruction's operand order.
// The waves' z tiles are added in a fixed order, split exactly into three bf16 terms and stored in the
// operand order the GEMM epilogue reads: zp[block][kk][term][lane][8], lane = row % 32 + 32 * h holding the
// rank columns 16 kk + 8 h + 0..7.
// Arithmetic: the rules at quant_rows_kernel, operation for operation.
// Bound by memory for long rows and by latency for few of them.  Splitting the statistics off reads x twice,
// the second time largely from the caches, and in return nothing has to be held: rows that had to wait in the
// LDS for their scale gave a workgroup 16 of them only up to K = 4608 and four at K = 12288, where every
// workgroup fetched the whole LoRA A for four rows.  Measured: 4096 x 12288, 8 adapters of rank 32: 22 us
// (statistics, routing, operand layouts) + 54 us against 14 us (layouts, routing) + 120 us; 333 x 4096, 4 adapters
// of rank 64: 7 + 16 us against 6 + 20 us.  Where the rows fit the LDS and the call has no operands to lay out, or
// sixteen slots hold several groups, quant_lora_rows_kernel below is the faster one (prologue_keeps_rows).
// The grouped (per-expert) call takes the same pass, its rows gathered through a row map and their statistics taken once
// per source row; as a quantizer and a LoRA-A launch over the gathered rows, 16384 of 2048, top 8 of 2048 tokens, it took
// 7 + 26 + 30 us, now 7 + 31.
// ---------------------------------------------------------------------------------------
struct QuantLoraArgs {
  const uint16_t* x;        // bf16 [M, K]: the rows, or (RMS false) rows that are normalized already
  const float* gamma;       // f32 [K] (RMS only)
  const float* row_scale;   // f32 [M] from row_stats
  const float* row_inv;     // f32 [M] from row_stats (RMS only)
  uint32_t M, K, K_pad, KB, n_half_blocks;  // n_half_blocks = ceil(slots that can hold rows / 16)
  const int32_t* src_row;   // original row of a slot, or null (identity)
  const int32_t* slot_group;// or null
  const int32_t* blk_range; // per 32-slot block, or null (group 0)
  unsigned char* xq_packed; // packed codes [slots/32][KB][1 KiB]
  float* sx_slots;          // f32 [slots]
  const uint16_t* at;       // LoRA A in MFMA operand order [n_groups][KB][CB][64 lanes][8 bf16] (lora_a_pack_item) or null (CB == 0)
  unsigned char* zp;        // packed z fragments
  uint32_t r, nkk, nterms;
  uint32_t* tile_ctr;       // 256 words cleared for the GEMM launches' tile counters, or null
  uint32_t group_pad;       // > 1: whole half blocks may be empty
  // Optional gather on the way in (see QuantArgs): source row = row_map[row] / row_div, clamped to row_limit;
  // row_scale then holds a value per source row (scale_by_source) or per row
  const int32_t* row_map;
  uint32_t row_div, row_limit, scale_by_source;
  float* z_rows;            // f32 [M, r]: z of every row for the backward, or null
};
// the form that leaves z in quarters
struct QuantLoraSplitArgs : QuantLoraArgs {
  float* zpart;             // f32 [4][slots][16 CB], the quarters' sums
  uint32_t slots;
};

// Row-major copies of the packed codes and of the slots' scales for a caller that asks for them (one workgroup per slot;
// either may be null).
__global__ __launch_bounds__(256) void codes_row_major_kernel(const unsigned char* __restrict__ xq, const float* __restrict__ sx,
                                                              const int32_t* __restrict__ src_row, int8_t* __restrict__ codes,
                                                              float* __restrict__ scales, uint32_t M, uint32_t K, uint32_t KB) {
  const uint32_t p = blockIdx.x;
  const int src = src_row ? src_row[p] : (int)p;
  if (src < 0 || src >= (int)M) return;
  if (scales && threadIdx.x == 0) scales[src] = sx[p];
  if (!codes) return;
  for (uint32_t k = threadIdx.x * 8u; k < K; k += 2048u)
    *reinterpret_cast<uint2*>(codes + (size_t)src * K + k) = *reinterpret_cast<const uint2*>(xq + packed_offset(p, k, KB));
}

constexpr uint32_t kPaddedRouteMaxRows = 8192;  // groups start on block boundaries up to here (padded_groups_fit)

// How a wave's rows are quantized: 0 by code_quotient; 1 the same, but a scale of one may stand for a row with a NaN, whose
// other values then need the clip; 2 a scale is not an ordinary number.  Wave-uniform.
__device__ inline uint32_t quant_mode(float scale) {
  if (__builtin_amdgcn_ballot_w64(!code_scale_ordinary(scale)) != 0) return 2u;
  return __builtin_amdgcn_ballot_w64(scale == 1.0f) != 0 ? 1u : 0u;
}
// The int8 codes of eight (normalized) bf16 values.  The division stands in a loop over the pairs: written out eight times at each
// of the fifteen places of a pass it made a third of the kernel's instructions, which a launch of few workgroups fetches as it goes
// (93 rows of 7680, rank 16: 9.7 us, 7.9 in the loop).
__device__ inline uint2 quant_codes8(const uint4& raw, float scale, float rscale, uint32_t mode) {
  if (mode != 0u) {
    const uint32_t top = bf16_absmax_pairs(0u, raw);  // 127.5 or more, as no value of a row of scale one without a NaN is
    if (mode == 2u || __builtin_amdgcn_ballot_w64(scale == 1.0f && ((top >> 16) >= 0x42ffu || (top & 0xffffu) >= 0x42ffu)) != 0) {
      // biased by 128 the code lands in its byte, clipped, with one v_cvt_pk_u8_f32; flipping bit 7 makes it two's complement
      uint32_t r[4] = {raw.x, raw.y, raw.z, raw.w}, lo = 0, hi = 0;
#pragma unroll 1
      for (int p = 0; p < 4; ++p) {
        uint32_t c = __builtin_amdgcn_cvt_pk_u8_f32(rintf(__uint_as_float(r[0] << 16) / scale) + 128.0f, 2u, 0u);
        c = __builtin_amdgcn_cvt_pk_u8_f32(rintf(__uint_as_float(r[0] & 0xffff0000u) / scale) + 128.0f, 3u, c);
        r[0] = r[1]; r[1] = r[2]; r[2] = r[3];
        lo = __builtin_amdgcn_alignbit(hi, lo, 16u);  // the earlier pairs move down
        hi = (hi >> 16) | c;
      }
      return make_uint2(lo ^ 0x80808080u, hi ^ 0x80808080u);
    }
  }
  const uint32_t nb[4] = {raw.x, raw.y, raw.z, raw.w};  // the (normalized) values as bf16 pairs
  float q[2][4];
#pragma unroll
  for (int e = 0; e < 8; ++e)
    q[e >> 2][e & 3] = code_quotient((e & 1) ? __uint_as_float(nb[e >> 1] & 0xffff0000u) : __uint_as_float(nb[e >> 1] << 16), scale, rscale);
  return make_uint2(code_bytes4(q[0]), code_bytes4(q[1]));
}

// z of a half block: the waves' tiles added in a fixed order, split into three bf16 terms and stored as the GEMM
// epilogue reads them (its rows first_row .. end_row - 1).  red: a wave tile each for waves 0..7 (of 16) or 0..3; zs: the
// sixteen rows of z.
// src_of(row): the row of x in it, or -1.
template <int kCB, uint32_t WAVES, class SrcOf>
__device__ inline void quant_lora_store_z(const QuantLoraArgs& a, v4f (&acc)[kCB], float (*red)[kCB][4][64], float (*zs)[kCB * 16 + 1],
                                          uint32_t pb, uint32_t half16, SrcOf&& src_of, uint32_t first_row = 0u, uint32_t end_row = 16u) {
  const uint32_t tid = threadIdx.x, lane = tid & 63u;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // of 16 waves, 8..15 onto 0..7, 4..7 onto 0..3; then 0+1+2+3
#pragma unroll 1
  for (uint32_t half = WAVES / 2u; half >= 4u; half >>= 1) {
    if (wave >= half && wave < 2u * half) {
#pragma unroll
      for (int b = 0; b < kCB; ++b)
#pragma unroll
        for (int e = 0; e < 4; ++e) red[wave - half][b][e][lane] = acc[b][e];
    }
    __syncthreads();
    if (wave < half) {
#pragma unroll
      for (int b = 0; b < kCB; ++b)
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[b][e] = acc[b][e] + red[wave][b][e][lane];
    }
    __syncthreads();
  }
  if (wave < 4u) {
#pragma unroll
    for (int b = 0; b < kCB; ++b)
#pragma unroll
      for (int e = 0; e < 4; ++e) red[wave][b][e][lane] = acc[b][e];
  }
  __syncthreads();
  // MFMA result layout: lane l holds column l % 16 and rows 4 * (l / 16) + e
  for (uint32_t t = tid; t < (uint32_t)kCB * 256u; t += WAVES * 64u) {
    const uint32_t l = t & 63u, e = (t >> 6) & 3u, b = t >> 8;
    const float sum = ((red[0][b][e][l] + red[1][b][e][l]) + red[2][b][e][l]) + red[3][b][e][l];
    zs[4u * (l >> 4) + e][b * 16u + (l & 15u)] = sum;
  }
  __syncthreads();
  if (a.z_rows) {  // kernel-uniform
    for (uint32_t t = tid; t < 16u * a.r; t += WAVES * 64u) {
      const uint32_t row = t / a.r, col = t % a.r;
      if (row < first_row || row >= end_row) continue;
      const int src = src_of(row);
      if (src >= 0 && src < (int)a.M) a.z_rows[(size_t)src * a.r + col] = zs[row][col];
    }
  }
  // zp[pb][kk][term][lane64][8]: lane = row % 32 + 32 * hh holds rank columns 16 kk + 8 hh + 0..7
  for (uint32_t t = tid; t < a.nkk * 3u * 32u; t += WAVES * 64u) {
    const uint32_t row = t & 15u, hh = (t >> 4) & 1u, term = (t >> 5) % 3u, kk = t / 96u;
    if (row < first_row || row >= end_row) continue;
    v8us o;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const uint32_t col = 16u * kk + 8u * hh + e;
      const float z = col < (uint32_t)kCB * 16u ? zs[row][col] : 0.0f;
      const uint32_t b0 = f32_to_bf16_bits(z);
      const float r1 = z - bf16_bits_to_f32(b0);
      const uint32_t b1 = f32_to_bf16_bits(r1);
      const float r2 = r1 - bf16_bits_to_f32(b1);
      const uint32_t b2 = f32_to_bf16_bits(r2);
      o[e] = (unsigned short)(term == 0 ? b0 : (term == 1 ? b1 : (a.nterms >= 3u ? b2 : 0u)));
    }
    const uint32_t l64 = 16u * half16 + row + 32u * hh;
    *reinterpret_cast<v8us*>(a.zp + (((size_t)pb * a.nkk + kk) * 3u + term) * kBlockBytes + l64 * 16u) = o;
  }
}

// The sum of a quarter's four tiles (waves w, w + 4, w + 8, w + 12 of the sixteen), in quant_lora_store_z's order.
template <int kCB>
__device__ inline void quant_lora_store_quarter(const QuantLoraSplitArgs& a, const v4f (&acc)[kCB], float (*red)[kCB][4][64], uint32_t hb, uint32_t part) {
  const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
#pragma unroll
  for (int b = 0; b < kCB; ++b)
#pragma unroll
    for (int e = 0; e < 4; ++e) red[wave][b][e][lane] = acc[b][e];
  __syncthreads();
  for (uint32_t t = tid; t < (uint32_t)kCB * 256u; t += 256u) {
    const uint32_t l = t & 63u, e = (t >> 6) & 3u, b = t >> 8;
    const float sum = (red[0][b][e][l] + red[2][b][e][l]) + (red[1][b][e][l] + red[3][b][e][l]);
    a.zpart[((size_t)part * a.slots + hb * 16u + 4u * (l >> 4) + e) * (kCB * 16u) + b * 16u + (l & 15u)] = sum;
  }
}

// At a group boundary: the rows of group grp (rowgrp: a lane's slot row lane % 16) keep this pass's sums, the others what they have (`first`: nothing
// yet).  Zeroing the other groups' rows of x instead leaves them 0 x infinity where the group's A is not finite.
template <int kCB, class Keep>
__device__ inline void keep_group_rows(const v4f (&acc)[kCB], uint32_t rowgrp, uint32_t grp, bool first, Keep&& keep) {
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const bool own = (uint32_t)__shfl((int)rowgrp, (int)(4u * ((threadIdx.x & 63u) >> 4)) + e, 64) == grp;
#pragma unroll
    for (int b = 0; b < kCB; ++b)
      if (own || first) keep(b, e, own ? acc[b][e] : 0.0f);
  }
}

// SPLIT: four workgroups of four waves share the half block, for calls whose half blocks are far fewer than the CUs.  Workgroup
// `part` plays waves part, part + 4, + 8, + 12 of the sixteen, fetches a quarter of A, and leaves the sum of its waves'
// tiles, added as the sixteen add theirs, in zpart: the consumer adds the quarters in order and so has the same z to the last bit
// (w8a8_gemm_ksplit_kernel).  With few rows the sixteen-wave form is a chain of operand fetches in 128 registers a lane
// (512 KiB of A for a workgroup at K = 4096, rank 64); a quarter of it fits in flight at once.
template <int CB, bool RMS, uint32_t WAVES = 16, bool SPLIT = false>  // CB: 16-wide rank blocks (0 = no LoRA, 1, 2, 4)
__global__ __launch_bounds__(WAVES * 64, SPLIT ? 2 : 4) void quant_lora_kernel(std::conditional_t<SPLIT, QuantLoraSplitArgs, QuantLoraArgs> a) {
  static_assert(!SPLIT || (WAVES == 4 && CB > 0), "four workgroups of four waves, for LoRA-A");
  constexpr int kCB = CB > 0 ? CB : 1;
  constexpr uint32_t kStride = SPLIT ? 16 : WAVES;  // k-blocks between two of a wave's
  constexpr uint32_t kRing = SPLIT ? (RMS ? 4 : 8) : (CB == 4 || (CB == 2 && RMS) ? 2 : 4);  // operand sets (what the registers hold)
  constexpr uint32_t kAhead = SPLIT ? 8 : 4;  // k-blocks of x a wave has in flight; a multiple of kRing
  static_assert(WAVES == 4 || WAVES == 16, "the reduction ends in four waves");
  __shared__ float red[CB > 0 ? (WAVES == 16 ? 8 : 4) : 1][kCB][4][64];  // wave tiles on their way to waves 0..7, then 0..3
  __shared__ float zs[16][kCB * 16 + 1];
  const uint32_t tid = threadIdx.x, lane = tid & 63u;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t hb = SPLIT ? blockIdx.x >> 2 : blockIdx.x;  // half block: slots 16 hb .. 16 hb + 15
  const uint32_t vw = SPLIT ? (blockIdx.x & 3u) + 4u * wave : wave;  // the wave of the sixteen
  if (a.tile_ctr && blockIdx.x == 0 && tid < 256u) a.tile_ctr[tid] = 0u;
  if (hb >= a.n_half_blocks) return;
  const uint32_t pb = hb >> 1, half16 = hb & 1u;
  const uint32_t i = lane & 15u, q = lane >> 4;
  int src = a.src_row ? a.src_row[hb * 16u + i] : (int)(hb * 16u + i);
  if (src < 0 || src >= (int)a.M) src = -1;
  if (a.group_pad > 1u && __builtin_amdgcn_ballot_w64(src >= 0) == 0)
    return;  // workgroup-uniform: padded groups leave whole stretches of slots empty: nothing reads their codes, scales or z
  // (a slot without a row works on row 0: nothing reads what it leaves, and no load sits under a lane condition)
  const uint32_t row = src < 0 ? 0u : (uint32_t)src;
  const uint32_t xrow = a.row_map ? mapped_row(a.row_map[row], a.row_div, a.row_limit) : row;
  const float scale = a.row_scale[a.scale_by_source ? xrow : row];
  const float inv = RMS ? a.row_inv[row] : 1.0f;
  if (vw == 0 && lane < 16u) a.sx_slots[hb * 16u + i] = scale;
  const float rscale = __builtin_amdgcn_rcpf(scale);
  const unsigned char* const xr = reinterpret_cast<const unsigned char*>(a.x) + (size_t)xrow * 2u * a.K;
  const uint32_t range = (CB > 0 && a.blk_range) ? (uint32_t)a.blk_range[pb] : 0u;
  const uint32_t glo = range & 0xffffu, ghi = range >> 16;
  const uint32_t rowgrp = (CB > 0 && ghi > glo && a.slot_group) ? (uint32_t)a.slot_group[hb * 16u + i] : glo;
  v4f acc[kCB];
#pragma unroll
  for (int b = 0; b < kCB; ++b) acc[b] = v4f{0.f, 0.f, 0.f, 0.f};
  // this lane's 8 codes of a fragment block: row 16*half16 + i, k half q/2, byte 8*(q%2)
  unsigned char* const xq_dst =
      a.xq_packed + (size_t)pb * a.KB * kBlockBytes + (16u * half16 + i + 32u * (q >> 1)) * 16u + 8u * (q & 1u);

  // The wave's j-th k-block is vw + kStride j.  Everything beyond the last block is read as zeros without a
  // condition: A and the norm weights through buffer resources that end with the data, x from the row's start.
  const __amdgpu_buffer_rsrc_t grsrc =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(a.gamma), 0, RMS ? (int)(a.K * 4u) : 0, 0x00020000);
  const uint32_t at_bytes = a.KB * (uint32_t)kCB * kBlockBytes;  // of one group
  const uint32_t kq = vw * 32u + q * 8u;                         // the lane's k in its wave's first k-block
  auto fetch_x = [&](uint32_t j) -> uint4 {
    const uint32_t k0 = kq + kStride * 32u * j;
    return *reinterpret_cast<const uint4*>(xr + 2u * (k0 < a.K ? k0 : 0u));  // (beyond K: zeroed where it is used)
  };
  struct Operands { v4i w[kCB]; v4f g0, g1; };
  auto fetch_operands = [&](const __amdgpu_buffer_rsrc_t& arsrc, uint32_t j, Operands& o) {
    if constexpr (CB > 0) {  // CB consecutive 1 KiB pieces (zero beyond K and the rank)
      const uint32_t off = (vw + kStride * j) * (uint32_t)(kCB * kBlockBytes) + lane * 16u;
#pragma unroll
      for (int b = 0; b < CB; ++b) o.w[b] = __builtin_amdgcn_raw_buffer_load_b128(arsrc, off + b * kBlockBytes, 0, 0);
    }
    if constexpr (RMS) {
      const uint32_t off = (kq + kStride * 32u * j) * 4u;
      o.g0 = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(grsrc, off, 0, 0));
      o.g1 = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(grsrc, off + 16u, 0, 0));
    }
  };
  const uint32_t mode = quant_mode(scale);
  auto work = [&](auto codes, uint32_t j, const uint4& rawx, const Operands& o) {
    const uint32_t kb = vw + kStride * j;
    uint4 raw = rawx;
    if constexpr (RMS)
      raw = rms_normalize8(rawx, inv, make_float4(o.g0[0], o.g0[1], o.g0[2], o.g0[3]), make_float4(o.g1[0], o.g1[1], o.g1[2], o.g1[3]));
    if (kb * 32u + 32u > a.K) {  // wave-uniform: the last k-block of an odd K, and the padding behind it
      const bool live = kq + kStride * 32u * j < a.K;
      raw.x = live ? raw.x : 0u; raw.y = live ? raw.y : 0u; raw.z = live ? raw.z : 0u; raw.w = live ? raw.w : 0u;
    }
    if constexpr (decltype(codes)::value) {
      *reinterpret_cast<uint2*>(xq_dst + (size_t)kb * kBlockBytes) = quant_codes8(raw, scale, rscale, mode);
    }
    if constexpr (CB > 0) {
      const v4i xa = {(int)raw.x, (int)raw.y, (int)raw.z, (int)raw.w};
#pragma unroll
      for (int b = 0; b < CB; ++b)
        acc[b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, xa), __builtin_bit_cast(v8bf, o.w[b]),
                                                         acc[b], 0, 0, 0);
    }
  };
  // A pass over the k-blocks, kAhead per trip: the x of kAhead k-blocks and the other operands of kRing - 1
  // are in flight beside the one at work.  (With few workgroups on the chip the loop is a chain of those
  // loads' latencies; no load or store in it is conditional, so the compiler's waits can count.)
  const uint32_t n_j = vw < a.KB ? (a.KB - vw + kStride - 1u) / kStride : 0u;
  auto pass = [&](auto codes, uint32_t grp) {
    const __amdgpu_buffer_rsrc_t arsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint16_t*>(a.at) + (size_t)grp * (at_bytes / 2u), 0, CB > 0 ? (int)at_bytes : 0, 0x00020000);
    uint4 xc[kAhead];
    Operands o[kRing];
#pragma unroll
    for (uint32_t u = 0; u < kAhead; ++u) xc[u] = fetch_x(u);
#pragma unroll
    for (uint32_t u = 0; u + 1u < kRing; ++u) fetch_operands(arsrc, u, o[u]);
    uint32_t j = 0;
#pragma unroll 1
    for (; j + kAhead <= n_j; j += kAhead) {
#pragma unroll
      for (uint32_t u = 0; u < kAhead; ++u) {
        fetch_operands(arsrc, j + u + kRing - 1u, o[(u + kRing - 1u) % kRing]);
        work(codes, j + u, xc[u], o[u % kRing]);
        xc[u] = fetch_x(j + u + kAhead);
      }
    }
#pragma unroll
    for (uint32_t u = 0; u + 1u < kAhead; ++u) {  // the rest, fewer than kAhead
      if (j + u >= n_j) break;  // wave-uniform
      fetch_operands(arsrc, j + u + kRing - 1u, o[(u + kRing - 1u) % kRing]);
      work(codes, j + u, xc[u], o[u % kRing]);
    }
  };
  // one pass per group present among the slots (one, except at a group boundary): the first also forms the
  // codes, a later one only z, and every row keeps the sums of its own group's pass
  pass(std::true_type{}, glo);
  if (CB > 0 && ghi > glo) {  // workgroup-uniform
    v4f z[kCB];
    auto keep = [&](int b, int e, float v) {
      if constexpr (SPLIT) red[wave][b][e][lane] = v;  // (its registers are all taken)
      else z[b][e] = v;
    };
    keep_group_rows<kCB>(acc, rowgrp, glo, true, keep);
#pragma unroll 1
    for (uint32_t grp = glo + 1u; grp <= ghi; ++grp) {
      if (__builtin_amdgcn_ballot_w64(rowgrp == grp) == 0) continue;
#pragma unroll
      for (int b = 0; b < kCB; ++b) acc[b] = v4f{0.f, 0.f, 0.f, 0.f};
      pass(std::false_type{}, grp);
      keep_group_rows<kCB>(acc, rowgrp, grp, false, keep);
    }
#pragma unroll
    for (int b = 0; b < kCB; ++b)
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[b][e] = SPLIT ? red[wave][b][e][lane] : z[b][e];
  }
  if constexpr (SPLIT) quant_lora_store_quarter<kCB>(a, acc, red, hb, blockIdx.x & 3u);
  else if constexpr (CB > 0)
    quant_lora_store_z<kCB, WAVES>(a, acc, red, zs, pb, half16, [&](uint32_t r) -> int { return a.src_row ? a.src_row[hb * 16u + r] : (int)(hb * 16u + r); });
}

// ---------------------------------------------------------------------------------------
// The same with the rows in the LDS: a wave brings one row in with direct-to-LDS loads, takes its statistics there
// (RMSNorm: and leaves it normalized), and the pass then reads the workgroup's R rows.  No launch takes statistics
// in front of it, x is read once and normalized once, and a further group among the rows costs a pass over the LDS; in return
// a workgroup has a CU to itself, starts the pass behind its own chain of statistics, and fetches the whole of A
// for as few rows as fit.
// With route_idx the workgroup sorts the adapter indices for its own slots, too, so that a call whose LoRA operands lie
// in the workspace already has this launch alone in front of the GEMM.
// ---------------------------------------------------------------------------------------
// LDS bytes of a row: its 2 K bytes rounded up to the 1 KiB a wave's direct-to-LDS load moves, plus 16 so
// that the sixteen rows a wave reads side by side (16 bytes each) fall on sixteen different bank groups.
__host__ __device__ inline uint32_t quant_lora_row_stride(uint32_t k) { return round_up(2u * k, 1024u) + 16u; }
inline uint32_t quant_lora_rows_per_wg(uint32_t k) {  // 16 up to K = 4608, then 8, from 9728 on 4
  uint32_t r = 16u;
  while (r > 4u && r * quant_lora_row_stride(k) > 150u * 1024u) r >>= 1;
  return r;
}
// dynamic LDS of a launch: the rows, or the reduction tiles that reuse the same bytes once the rows are spent
inline uint32_t quant_lora_rows_lds_bytes(uint32_t k, uint32_t cb) {
  const uint32_t rows = quant_lora_rows_per_wg(k) * quant_lora_row_stride(k), red = 8u * (cb ? cb : 1u) * 4u * 64u * 4u;
  return rows > red ? rows : red;
}

struct QuantLoraRowsArgs {
  QuantLoraArgs q;           // row_scale, row_inv unused
  float eps;
  float* scales_rm;          // f32 [M] for the caller, or null
  uint16_t* xn_aux;          // bf16 [M, K] normalized rows for the caller, or null (RMS only)
  // Routing inside this launch (M <= kInlineRouteMaxRows): every workgroup sorts the indices for itself and writes
  // its slots' entries of the tables, which the GEMM reads.
  const int32_t* route_idx;  // adapter per row, or null: the tables of an earlier launch, or none
  int32_t* src_row; int32_t* slot_group; int32_t* blk_range;
  uint32_t n_groups, slots;
  uint32_t rows_per_wg, row_stride;
};
constexpr uint32_t kInlineRouteMaxRows = 8192;  // eight rows per thread of a 1024-thread workgroup

// The routing tables of route_rows_block for the 16 slots [16 hb, 16 hb + 16), computed by the
// workgroup itself: rows keep their order inside a group (slot start[g] + j holds the j-th row of group
// g), which every workgroup derives alike from the adapter indices alone.  Returns through LDS:
// out_src[16], out_grp[16], out_range (the group range of the 32-slot block that holds the slots).
// With group_pad = 32 every group starts on a block boundary (the slots between a group's last row and
// the next group's first stay empty, src -1), so no 32-slot block holds rows of two groups: neither
// this kernel nor the GEMM's epilogue then runs a block once per group.  The slots in use end at
// sum(round_up(count, group_pad)) <= M + (group_pad - 1) * min(n_groups, M).
// Steps: every wave counts its rows per group (LDS atomics on its own counters: with 16 waves on a CU
// the vector ALU's share per wave makes a ballot per group and row several times dearer); wave 0 turns
// the counts into per-wave prefixes, the groups' first slots and the groups of the sixteen slots; the
// waves that hold the wanted ranks of a group pick their rows.  Three barriers.
__device__ inline void route_rows_inline(const int32_t* __restrict__ idx, uint32_t M, uint32_t n_groups,
                                         uint32_t slots, uint32_t group_pad, uint32_t hb, int* out_src, int* out_grp,
                                         uint32_t* out_range, int* out_last_group) {
  __shared__ int wcnt[kMaxAdapters][17];  // rows of group g in wave w; then the exclusive prefix over the waves
  __shared__ int start[kMaxAdapters + 1];
  __shared__ int cnt[kMaxAdapters];
  __shared__ uint32_t used_end;  // first slot behind the last group
  __shared__ int g_first_s, g_last_s;
  const uint32_t tid = threadIdx.x, lane = tid & 63u;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t per = (M + 1023u) / 1024u;  // consecutive rows per thread (<= 8)
  int mine[8];
#pragma unroll
  for (uint32_t j = 0; j < 8; ++j) {
    const uint32_t i = tid * per + j;
    int a = -1;
    if (j < per && i < M) {
      a = idx[i];
      a = a < 0 ? 0 : (a >= (int)n_groups ? (int)n_groups - 1 : a);
    }
    mine[j] = a;
  }
  if (lane < n_groups) wcnt[lane][wave] = 0;  // (the loads above are still in flight)
  __builtin_amdgcn_wave_barrier();
#pragma unroll
  for (uint32_t j = 0; j < 8; ++j)
    if (j < per && mine[j] >= 0) atomicAdd(&wcnt[mine[j]][wave], 1);  // integer counts of one wave: any order
  __syncthreads();
  const uint32_t p0 = hb * 16u;
  if (wave == 0) {  // lane g: group g (n_groups <= 64)
    int total = 0;
    if (lane < n_groups) {
      int c[16];
#pragma unroll
      for (uint32_t w = 0; w < 16; ++w) c[w] = wcnt[lane][w];  // all reads first: one round trip
#pragma unroll
      for (uint32_t w = 0; w < 16; ++w) {
        wcnt[lane][w] = total;
        total += c[w];
      }
    }
    const int padded = (int)round_up((uint32_t)total, group_pad);
    const int incl = (int)wave_scan((uint32_t)padded);
    const int st = incl - padded;  // first slot of group `lane`
    const uint32_t E = (uint32_t)__builtin_amdgcn_readlane(incl, 63);
    const unsigned long long nonempty = __builtin_amdgcn_ballot_w64(total > 0);
    const int last_ne = nonempty ? 63 - __builtin_clzll(nonempty) : 0;
    if (lane < n_groups) { start[lane] = st; cnt[lane] = total; }
    if (lane == 0) { start[n_groups] = (int)E; used_end = E; *out_last_group = last_ne; }
    // group of a slot: the last group whose first slot is not behind it (empty groups share their
    // successor's first slot, so the last one is the one that holds the slot); slots behind the last
    // group follow the last non-empty one
    auto group_of = [&](uint32_t p) -> int {
      if (p >= E) return last_ne;
      const unsigned long long m = __builtin_amdgcn_ballot_w64(lane < n_groups && (uint32_t)st <= p);
      return m ? 63 - __builtin_clzll(m) : 0;
    };
    const uint32_t p_end = (p0 + 16u < E) ? p0 + 16u : E;
    const int gf = group_of(p0), gl = group_of(p_end ? p_end - 1u : 0u);
    int my_grp = group_of(p0 + 15u);  // (the slots behind the last group follow the last non-empty one)
    if (my_grp != gf) {  // wave-uniform: the sixteen slots hold a group boundary (or the end)
#pragma unroll
      for (uint32_t s16 = 0; s16 < 16; ++s16) {
        const int g = group_of(p0 + s16);
        if (lane == s16) my_grp = g;
      }
    }
    if (lane < 16u) { out_grp[lane] = my_grp; out_src[lane] = -1; }
    const uint32_t b0 = (p0 / 32u) * 32u;
    const uint32_t b1 = (b0 + 31u < E) ? b0 + 31u : (E ? E - 1u : 0u);
    const int gb0 = group_of(b0), gb1 = group_of(b1);
    if (lane == 0) {
      *out_range = b0 >= E ? 0u : ((uint32_t)gb0 | ((uint32_t)gb1 << 16));
      g_first_s = p0 < E ? gf : 1;  // an empty range when the slots lie behind the last group
      g_last_s = p0 < E ? gl : 0;
    }
  }
  __syncthreads();
  // the rows of the slots in use, group by group (a workgroup's 16 slots usually lie in one group)
  const uint32_t E = used_end;
  const uint32_t p_end = (p0 + 16u < E) ? p0 + 16u : E;
  const int g_first = g_first_s, g_last = g_last_s;
  for (int g = g_first; g <= g_last; ++g) {  // workgroup-uniform
    const int cg = cnt[g], sg = start[g];
    if (cg == 0) continue;
    // slots of group g among mine: ranks [lo, hi)
    const int lo = ((int)p0 > sg ? (int)p0 : sg) - sg;
    const int hi = ((int)p_end < sg + cg ? (int)p_end : sg + cg) - sg;
    const int wbefore = wcnt[g][wave];
    const int wafter = wave < 15u ? wcnt[g][wave + 1u] : cg;
    if (hi <= lo || wafter <= lo || wbefore >= hi) continue;  // wave-uniform: none of the wanted ranks is in this wave
    int c = 0;
#pragma unroll
    for (uint32_t j = 0; j < 8; ++j) c += (mine[j] == g) ? 1 : 0;
    int rank = wbefore + (int)wave_scan((uint32_t)c) - c;
#pragma unroll
    for (uint32_t j = 0; j < 8; ++j) {
      if (mine[j] == g) {
        if (rank >= lo && rank < hi) out_src[sg + rank - (int)p0] = (int)(tid * per + j);
        ++rank;
      }
    }
  }
  __syncthreads();
}

template <int CB, bool RMS>  // CB: 16-wide rank blocks (0 = no LoRA, 1, 2, 4)
__global__ __launch_bounds__(1024) void quant_lora_rows_kernel(QuantLoraRowsArgs p) {
  const QuantLoraArgs& a = p.q;
  constexpr int kCB = CB > 0 ? CB : 1;
  extern __shared__ __attribute__((aligned(1024))) unsigned char ql_lds[];  // the rows; later the wave tiles of z
  __shared__ float row_scale[16];
  __shared__ int row_src[16];
  __shared__ float zs[16][kCB * 16 + 1];
  const uint32_t tid = threadIdx.x, lane = tid & 63u;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t R = p.rows_per_wg, per_hb = 16u / R;
  const uint32_t hb = blockIdx.x / per_hb;           // half block: slots 16 hb .. 16 hb + 15
  const uint32_t r0 = (blockIdx.x % per_hb) * R;     // this workgroup's slots inside it: r0 .. r0 + R - 1
  if (a.tile_ctr && blockIdx.x == 0 && tid < 256u) a.tile_ctr[tid] = 0u;
  if (hb >= a.n_half_blocks) return;
  const uint32_t pb = hb >> 1, half16 = hb & 1u;
  __shared__ int route_src[16], route_grp[16], route_last_group;
  __shared__ uint32_t route_range;
  const bool route_here = p.route_idx != nullptr;  // kernel-uniform
  if (route_here) {
    route_rows_inline(p.route_idx, a.M, p.n_groups, p.slots, a.group_pad, hb, route_src, route_grp, &route_range,
                      &route_last_group);
    // the tables the GEMM reads later (every workgroup of a block derives the same range)
    if (tid >= r0 && tid < r0 + R) {
      p.src_row[hb * 16u + tid] = route_src[tid];
      p.slot_group[hb * 16u + tid] = route_grp[tid];
    }
    if (tid == 16u) p.blk_range[pb] = (int32_t)route_range;
    if (blockIdx.x + 1u == gridDim.x) {  // the padding slots behind the last 32-row block, up to the GEMM's tile rows
      for (uint32_t s = a.n_half_blocks * 16u + tid; s < p.slots; s += 1024u) {
        p.src_row[s] = -1;
        p.slot_group[s] = route_last_group;
        if ((s & 31u) == 0) p.blk_range[s / 32u] = 0;
      }
    }
  }
  // ---- 1. the rows into the LDS and their statistics: wave w < R, slot row r0 + w
  const uint32_t slot = hb * 16u + r0 + wave;
  int wsrc = -1;
  if (wave < R) wsrc = route_here ? route_src[r0 + wave] : (a.src_row ? a.src_row[slot] : (int)slot);
  if (wsrc < 0 || wsrc >= (int)a.M) wsrc = -1;
  wsrc = __builtin_amdgcn_readfirstlane(wsrc);
  if (a.group_pad > 1u) {  // padded groups leave whole stretches of slots empty: nothing reads their codes, scales or z
    if (__syncthreads_or(wsrc >= 0) == 0) return;
  }
  const uint32_t lds_addr = (uint32_t)(uintptr_t)(lptr_t)ql_lds;
  const uint32_t row_bytes = 2u * a.K;
  if (wave < R) {
    unsigned char* const rowl = ql_lds + wave * p.row_stride;
    float inv = 1.0f;
    uint32_t amax_bits = 0;  // largest |value| as bf16 bits in both halves
    if (wsrc >= 0) {
      const unsigned char* xr = reinterpret_cast<const unsigned char*>(a.x) + (size_t)wsrc * row_bytes;
      for (uint32_t off = 0; off < row_bytes; off += 1024u) {
        const uint32_t voff = off + lane * 16u;
        if (voff < row_bytes) lds_load_1k(xr, voff, lds_addr + wave * p.row_stride + off);
      }
      // (the first piece's norm weights travel with the row)
      float4 gn0 = make_float4(0.f, 0.f, 0.f, 0.f), gn1 = gn0;
      if (RMS && lane * 16u < row_bytes) {
        gn0 = *reinterpret_cast<const float4*>(a.gamma + lane * 8u);
        gn1 = *reinterpret_cast<const float4*>(a.gamma + lane * 8u + 4);
      }
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      if (RMS) {
        double ss = 0.0;
        for (uint32_t off = lane * 16u; off < row_bytes; off += 1024u) {
          const uint4 raw = *reinterpret_cast<const uint4*>(rowl + off);
          const uint32_t w[4] = {raw.x, raw.y, raw.z, raw.w};
#pragma unroll
          for (int e = 0; e < 4; ++e) {  // (exact squares, as in row_stats)
            const double lo = (double)__uint_as_float(w[e] << 16), hi = (double)__uint_as_float(w[e] & 0xffff0000u);
            ss = __builtin_fma(lo, lo, ss);
            ss = __builtin_fma(hi, hi, ss);
          }
        }
        ss = wave_sum(ss);
        const float var = (float)(ss / (double)a.K);
        inv = 1.0f / sqrtf(var + p.eps);
      }
      for (uint32_t off = lane * 16u; off < row_bytes; off += 1024u) {
        const float4 g0 = gn0, g1 = gn1;
        if (RMS && off + 1024u < row_bytes) {  // the norm weights of the next piece are requested before this one is worked on
          gn0 = *reinterpret_cast<const float4*>(a.gamma + ((off + 1024u) >> 1));
          gn1 = *reinterpret_cast<const float4*>(a.gamma + ((off + 1024u) >> 1) + 4);
        }
        uint4 raw = *reinterpret_cast<const uint4*>(rowl + off);
        if (RMS) {
          raw = rms_normalize8(raw, inv, g0, g1);
          *reinterpret_cast<uint4*>(rowl + off) = raw;  // the normalized row replaces the row
          if (p.xn_aux) *reinterpret_cast<uint4*>(reinterpret_cast<unsigned char*>(p.xn_aux) + (size_t)wsrc * row_bytes + off) = raw;
        }
        amax_bits = bf16_absmax_pairs(amax_bits, raw);
      }
    }
    const float scale = row_scale_of(amax_bits);
    if (lane == 0) {
      row_scale[r0 + wave] = scale;
      row_src[r0 + wave] = wsrc;
      a.sx_slots[slot] = scale;
      if (p.scales_rm && wsrc >= 0) p.scales_rm[wsrc] = scale;
    }
  }
  __syncthreads();

  // ---- 2. codes and z: lane (i, q) takes k = 32 kb + 8 q .. + 7 of slot row i, wave w the k-blocks w + 16 j
  const uint32_t i = lane & 15u, q = lane >> 4;
  const bool mine_row = i >= r0 && i < r0 + R;  // slot row i belongs to this workgroup
  const int src = mine_row ? row_src[i] : -1;
  const float scale = mine_row ? row_scale[i] : 1.0f;
  const float rscale = __builtin_amdgcn_rcpf(scale);
  const uint32_t mode = quant_mode(scale);
  const unsigned char* const rowl = ql_lds + (mine_row ? i - r0 : 0u) * p.row_stride;
  const uint32_t range = CB == 0 ? 0u : (route_here ? route_range : (a.blk_range ? (uint32_t)a.blk_range[pb] : 0u));
  const uint32_t glo = range & 0xffffu, ghi = range >> 16;
  const uint32_t rowgrp = (CB > 0 && ghi > glo)
                              ? (route_here ? (uint32_t)route_grp[i] : (a.slot_group ? (uint32_t)a.slot_group[hb * 16u + i] : glo))
                              : glo;
  v4f acc[kCB];
#pragma unroll
  for (int b = 0; b < kCB; ++b) acc[b] = v4f{0.f, 0.f, 0.f, 0.f};
  unsigned char* const xq_dst =
      a.xq_packed + (size_t)pb * a.KB * kBlockBytes + (16u * half16 + i + 32u * (q >> 1)) * 16u + 8u * (q & 1u);
  // One pass over the k-blocks per group present among the slots (one, except at a group boundary): the
  // first pass also forms the codes; a later pass only z.  The loop is kept rolled, two
  // k-blocks per trip with their operands requested one trip ahead and no load inside the work on a
  // k-block, so that the compiler's waits count loads instead of draining them.
  auto request = [&](uint32_t grp, uint32_t kb, v4i (&w)[kCB], uint4& raw) {
    if constexpr (CB > 0) {
      // operands of group grp, k-block kb: CB consecutive 1 KiB pieces (zero beyond K and the rank)
      const v4i* ap = reinterpret_cast<const v4i*>(a.at) + (((size_t)grp * a.KB + kb) * CB) * 64u + lane;
#pragma unroll
      for (int b = 0; b < CB; ++b) w[b] = kb < a.KB ? ap[b * 64] : v4i{0, 0, 0, 0};
    }
    const uint32_t k0 = kb * 32u + q * 8u;
    raw = (kb < a.KB && k0 < a.K && src >= 0) ? *reinterpret_cast<const uint4*>(rowl + 2u * k0) : make_uint4(0, 0, 0, 0);
  };
  auto work = [&](bool first, uint32_t kb, const v4i (&w)[kCB], const uint4& raw) {
    if (first) {  // wave-uniform
      const uint2 codes = quant_codes8(raw, scale, rscale, mode);
      if (mine_row) *reinterpret_cast<uint2*>(xq_dst + (size_t)kb * kBlockBytes) = codes;
    }
    if constexpr (CB > 0) {
      const v4i xa = {(int)raw.x, (int)raw.y, (int)raw.z, (int)raw.w};  // (zeros where the lane has no value)
#pragma unroll
      for (int b = 0; b < CB; ++b)
        acc[b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, xa), __builtin_bit_cast(v8bf, w[b]),
                                                         acc[b], 0, 0, 0);
    }
  };
  v4f z[kCB];  // (at a group boundary: every row the sums of its own group's pass)
#pragma unroll 1
  for (uint32_t grp = glo; grp <= ghi; ++grp) {  // workgroup-uniform: one trip except at a group boundary
    const bool first = grp == glo;
    if (CB > 0 && !first) {
      if (__builtin_amdgcn_ballot_w64(rowgrp == grp) == 0) continue;
#pragma unroll
      for (int b = 0; b < kCB; ++b) acc[b] = v4f{0.f, 0.f, 0.f, 0.f};
    }
    v4i wa[kCB], wb2[kCB];
    uint4 ra, rb;
    request(grp, wave, wa, ra);
    request(grp, wave + 16u, wb2, rb);
#pragma unroll 1
    for (uint32_t kb = wave; kb < a.KB; kb += 32u) {
      work(first, kb, wa, ra);
      request(grp, kb + 32u, wa, ra);
      if (kb + 16u >= a.KB) break;  // wave-uniform
      work(first, kb + 16u, wb2, rb);
      request(grp, kb + 48u, wb2, rb);
    }
    if constexpr (CB == 0) break;
    if (ghi > glo) keep_group_rows<kCB>(acc, rowgrp, grp, first, [&](int b, int e, float v) { z[b][e] = v; });
  }
  if constexpr (CB > 0) {
    if (ghi > glo) {
#pragma unroll
      for (int b = 0; b < kCB; ++b) acc[b] = z[b];
    }
    __syncthreads();  // the rows are spent: their bytes take the wave tiles
    quant_lora_store_z<kCB, 16u>(a, acc, reinterpret_cast<float (*)[kCB][4][64]>(ql_lds), zs, pb, half16,
                                   [&](uint32_t r) -> int { return row_src[r]; }, r0, r0 + R);
  }
}

}  // namespace w8a8
