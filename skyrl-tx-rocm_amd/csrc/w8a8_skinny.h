// Skinny-M (decode) path, M <= 32 rows: the weight is streamed exactly once from HBM.
//   1. skinny_quant_kernel   one workgroup per row: (RMSNorm,) absmax, scale, int8 codes in
//                            MFMA operand order; where a loop asks for it, B regrouped for the stream kernel.
//                            LoRA-A units ride along: z_part[chunk][m][:] = x[m, chunk] @
//                            A[idx[m]][chunk, :] in float32 (with RMSNorm every unit forms the row's
//                            inverse RMS for itself: a few KiB from the L2 against a launch of its own).
//   2. skinny_stream_kernel  every workgroup owns 16 or 32 weight columns for all of K: its eight waves
//                            stream the weight once from HBM straight into MFMA operands (no LDS:
//                            every byte is used once), are reduced through LDS, and the workgroup
//                            finishes its columns: (float(acc) * sx) * sw + s * (z @ B[idx[m]])
//                            + residual, one bf16 cast, or the SwiGLU of the (gate, up) column pairs.
// Integer sums are exact and the float32 sums have a fixed order: results are bit-identical
// from run to run.  No atomics, no data crosses workgroups inside a launch.
#pragma once
#include "../../include/mi355_w8a8.h"
#include "w8a8_device.h"
#include "w8a8_gemm.h"

namespace w8a8 {

constexpr int kSkinnyMaxRows = 32;
constexpr uint32_t kSkinnyMaxZChunks = 16;
constexpr uint32_t kSkinnyZChunkK = 1024;  // K elements per LoRA-A work unit (per row)

// Ranks of a row of the regrouped B (skinny_regroup_b): 1 KiB holds whole rows.
__host__ __device__ inline uint32_t skinny_b_ranks(uint32_t r) { return r <= 16u ? 16u : 32u; }
// Two slices of 16 columns to a workgroup, or one: slices of 16 columns while 32-column units would leave CUs idle
// (fewer than 512 units: two workgroups share a CU); SwiGLU and residual decide for themselves (a gate/up
// pair is two slices; the residual's dword gather serves one column).
inline bool skinny_pairs(uint32_t n, bool swiglu, bool residual) {
  return swiglu || (!residual && (n & 1u) == 0 && n_padded(n) / 128u * 4u >= 512u);
}
// Calls that can keep B regrouped: one slice, one row half, whole column quads, and values enough.  Per call of a loop, B
// gathered / regrouped: 12288 x 4096, 16 rows of rank 32 20.4 / 18.9 us, 8 rows 17.9 / 17.3, 9 rows of rank 16 16.5 / 15.8;
// 2560 x 6144, 16 rows of rank 32 16.2 / 13.8, 9 rows of rank 16 11.9 / 11.3; below that, where the host bounds a call,
// level or 0.3 slower (4096 x 2560, 4 rows of rank 16 10.0 / 10.4, 8 rows 10.3 / 10.3).
inline bool skinny_b_can_be_kept(uint32_t m, uint32_t n, uint32_t r, bool swiglu) {
  return !swiglu && m <= 16u && r <= 32u && m * r > 128u && (n & 3u) == 0;
}

struct SkinnyLayout {
  uint64_t z_part, row_scaling, bsel, total;
  uint32_t pairs_per_wave, z_chunks, z_chunk_k;
};

// keep_b: with the regrouped B of m rows of rank r
inline SkinnyLayout skinny_layout(uint32_t k, bool keep_b = false, uint32_t m = 0u, uint32_t n = 0u, uint32_t r = 0u) {
  SkinnyLayout L{};
  const uint32_t n_pairs = k_padded(k) / 64u;
  L.pairs_per_wave = (n_pairs + 7u) / 8u;
  uint32_t zc = (k + kSkinnyZChunkK - 1u) / kSkinnyZChunkK;
  uint32_t zk = kSkinnyZChunkK;
  while (zc > kSkinnyMaxZChunks) { zk *= 2u; zc = (k + zk - 1u) / zk; }
  L.z_chunks = zc;
  L.z_chunk_k = zk;
  L.z_part = 0;
  L.row_scaling = (uint64_t)kSkinnyMaxZChunks * kSkinnyMaxRows * kMaxRank * 4u;
  L.bsel = L.row_scaling + 256u;
  L.total = L.bsel + (keep_b ? (uint64_t)(n_padded(n) / 16u) * m * skinny_b_ranks(r) * 32u + 1024u : 0u);  // (whole KiBs are read)
  return L;
}

// ---------------------------------------------------------------------------------------
struct SkinnyQuantArgs {
  const uint16_t* x;     // bf16 [M, K]
  const float* gamma;    // f32 [K] or null
  float eps;
  uint32_t M, K, K_pad, KB;
  unsigned char* xq;     // packed codes, one 32-row block [KB][1 KiB]
  float* sx;             // f32 [32]
  int8_t* codes_rm;      // optional row-major copy
  float* scales_rm;      // optional
  uint16_t* xn_aux;      // bf16 [M, K] normalized rows for the caller (RMSNorm only) or null
  // LoRA-A work units that share the launch (they need only x, not the codes)
  const uint16_t* lora_a;  // bf16 [n_adapters, K, r] or null
  const int32_t* idx;      // adapter per row or null
  float* z_part;           // f32 [z_chunks][32][kMaxRank]
  uint32_t n_adapters, r, z_chunks, z_chunk_k, n_z_units;
  const float* lora_scaling;  // f32 [n_adapters] or null
  float* row_scaling;      // f32 [32]: lora_scaling[idx[m]], written here for the stream kernel
  // B regrouped for the stream kernel, by blocks behind the LoRA-A units (sixteen items of a row and 128 columns each)
  const uint16_t* lora_b;  // bf16 [n_adapters, r, N]
  uint16_t* bsel;          // or null
  uint32_t N, n_groups;    // n_groups = N_pad / 128
};

// B of row m's adapter in the order in which the stream kernel's units of 16 columns read it, 128 columns of it:
// bsel[8 G + u][m][p][c][t] = B[idx[m]][2 t + p][128 G + 4 (16 (u & 1) + c) + u / 2], zeros beyond the rank.  A wave; two
// ranks at a time.
__device__ inline void skinny_regroup_b(const SkinnyQuantArgs& a, uint32_t item) {
  const uint32_t lane = threadIdx.x & 63u, m = item / a.n_groups, G = item % a.n_groups;
  if (m >= a.M) return;
  int ad = a.idx ? a.idx[m] : 0;
  ad = ad < 0 ? 0 : (ad >= (int)a.n_adapters ? (int)a.n_adapters - 1 : ad);
  const uint32_t quad = lane & 31u, p = lane >> 5, col = 128u * G + 4u * quad, ranks = skinny_b_ranks(a.r);
  const uint16_t* src = a.lora_b + (size_t)ad * a.r * a.N + (col < a.N ? col : 0u);
  uint16_t* dst = a.bsel + (((size_t)(8u * G + (quad >> 4)) * a.M + m) * 2u + p) * (8u * ranks) + (quad & 15u) * (ranks / 2u);
  const size_t next = (size_t)2u * a.M * ranks * 16u;  // the next column of the quad: two units on
#pragma unroll 4
  for (uint32_t t = 0; t < ranks / 2u; ++t) {
    const uint32_t r = 2u * t + p;
    uint2 v = *reinterpret_cast<const uint2*>(src + (size_t)(r < a.r ? r : 0u) * a.N);
    if (r >= a.r) v = make_uint2(0u, 0u);
    dst[t] = (uint16_t)v.x; dst[next + t] = (uint16_t)(v.x >> 16);
    dst[2u * next + t] = (uint16_t)v.y; dst[3u * next + t] = (uint16_t)(v.y >> 16);
  }
}

// Inverse RMS of row xr by a workgroup of 1024 threads (float64 sum, IEEE division and square root), the
// same value in every workgroup that forms it: v holds the thread's 2 x 8 values of the row.
__device__ inline float skinny_inverse_rms(const float (&v)[2][8], uint32_t K, float eps, double* red_sum) {
  double ss = 0.0;
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int e = 0; e < 8; ++e) ss += (double)v[j][e] * (double)v[j][e];
  ss = wave_sum(ss);
  if ((threadIdx.x & 63u) == 0) red_sum[threadIdx.x >> 6] = ss;
  __syncthreads();
  double tot = 0.0;
#pragma unroll
  for (int w = 0; w < 16; ++w) tot += red_sum[w];
  const float var = (float)(tot / (double)K);
  return 1.0f / sqrtf(var + eps);
}
__device__ inline void skinny_row_values(const uint16_t* __restrict__ xr, uint32_t K, float (&v)[2][8]) {
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const uint32_t k0 = (j * 1024u + threadIdx.x) * 8u;
    uint4 raw = make_uint4(0, 0, 0, 0);
    if (k0 < K) raw = *reinterpret_cast<const uint4*>(xr + k0);
    const uint32_t w[4] = {raw.x, raw.y, raw.z, raw.w};
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      v[j][2 * e] = __uint_as_float(w[e] << 16);
      v[j][2 * e + 1] = __uint_as_float(w[e] & 0xffff0000u);
    }
  }
}

// z_part[ch][m][:] = x[m, chunk ch] @ A[idx[m]][chunk ch, :] in float32.  Thread (kl, q)
// accumulates rank columns 8q..8q+7 over the rows k = k_begin + kl + kpt*j; lanes with equal q are
// reduced by a fixed butterfly and the waves are added in wave order.  With RMS the row's values are the
// normalized ones, bf16((x * inv) * gamma), formed here as the quantizer forms them.
template <int THREADS, bool RMS>
__device__ inline void skinny_lora_a_unit(const uint16_t* __restrict__ xsrc, const float* __restrict__ gamma, float inv, const uint16_t* __restrict__ lora_a,
                                          const int32_t* __restrict__ idx, float* __restrict__ z_part,
                                          uint32_t unit, uint32_t K, uint32_t n_adapters, uint32_t r,
                                          uint32_t z_chunks, uint32_t z_chunk_k, float (*zw)[64]) {
  constexpr uint32_t kWaves = THREADS / 64;
  const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
  const uint32_t m = unit / z_chunks, ch = unit % z_chunks;
  int ad = idx ? idx[m] : 0;
  ad = ad < 0 ? 0 : (ad >= (int)n_adapters ? (int)n_adapters - 1 : ad);
  const uint16_t* Ar = lora_a + (size_t)ad * K * r;
  const uint16_t* xr = xsrc + (size_t)m * K;
  const uint32_t rch = (r + 7u) / 8u;  // 8-wide rank chunks
  const uint32_t rch2 = rch <= 1u ? 1u : (rch <= 2u ? 2u : (rch <= 4u ? 4u : 8u));
  const uint32_t kpt = THREADS / rch2;
  const uint32_t q = tid % rch2, kl = tid / rch2;
  float accz[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  const uint32_t k_begin = ch * z_chunk_k;
  uint32_t k_end = k_begin + z_chunk_k;
  if (k_end > K) k_end = K;
  if (q < rch) {
    if ((r & 7u) == 0) {
      // four rows of A per round, their loads issued together (same order of additions as a plain loop)
      for (uint32_t k = k_begin + kl; k < k_end; k += 4u * kpt) {
        v8us w[4];
        float xv[4], gv[4];
#pragma unroll
        for (uint32_t u = 0; u < 4; ++u) {
          const uint32_t ku = k + u * kpt;
          const bool in = ku < k_end;
          const v8us zero = {0, 0, 0, 0, 0, 0, 0, 0};
          w[u] = in ? *reinterpret_cast<const v8us*>(Ar + (size_t)ku * r + q * 8u) : zero;
          xv[u] = in ? bf16_bits_to_f32(xr[ku]) : 0.f;
          gv[u] = (RMS && in) ? gamma[ku] : 0.f;
        }
        if (RMS) {
#pragma unroll
          for (uint32_t u = 0; u < 4; ++u) xv[u] = bf16_round_f32((xv[u] * inv) * gv[u]);
        }
#pragma unroll
        for (uint32_t u = 0; u < 4; ++u) {
          if (k + u * kpt < k_end) {
#pragma unroll
            for (int e = 0; e < 8; ++e) accz[e] = fmaf(xv[u], bf16_bits_to_f32(w[u][e]), accz[e]);
          }
        }
      }
    } else {
      for (uint32_t k = k_begin + kl; k < k_end; k += kpt) {
        float xv = bf16_bits_to_f32(xr[k]);
        if (RMS) xv = bf16_round_f32((xv * inv) * gamma[k]);
        const uint16_t* src = Ar + (size_t)k * r + q * 8u;
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (q * 8u + e < r) accz[e] = fmaf(xv, bf16_bits_to_f32(src[e]), accz[e]);
      }
    }
  }
  const auto add = [](float x, float y) { return x + y; };
#pragma unroll
  for (int e = 0; e < 8; ++e) {  // the steps rch2, 2 rch2, .., 32
    if (rch2 < 2u) accz[e] = lane_step<1>(accz[e], add);
    if (rch2 < 4u) accz[e] = lane_step<2>(accz[e], add);
    if (rch2 < 8u) accz[e] = lane_step<4>(accz[e], add);
    accz[e] = lane_step<8>(accz[e], add);
    accz[e] = lane_step<16>(accz[e], add);
    accz[e] = lane_step<32>(accz[e], add);
  }
  if (lane < rch2) {
#pragma unroll
    for (int e = 0; e < 8; ++e) zw[wave][lane * 8u + e] = accz[e];
  }
  __syncthreads();
  if (tid < (uint32_t)kMaxRank) {
    float sum = zw[0][tid];
#pragma unroll
    for (uint32_t w = 1; w < kWaves; ++w) sum += zw[w][tid];
    z_part[((size_t)ch * kSkinnyMaxRows + m) * kMaxRank + tid] = (tid < r) ? sum : 0.f;
  }
}

template <bool RMS>
__global__ __launch_bounds__(1024) void skinny_quant_kernel(SkinnyQuantArgs a) {
  __shared__ float red_max[16];
  __shared__ double red_sum[16];
  __shared__ float zw[16][64];
  if (blockIdx.x >= a.M + a.n_z_units) {
    skinny_regroup_b(a, (blockIdx.x - a.M - a.n_z_units) * 16u + (threadIdx.x >> 6));
    return;
  }
  if (blockIdx.x >= a.M) {
    const uint32_t unit = blockIdx.x - a.M;
    float inv = 1.0f;
    if (RMS) {
      float v[2][8];
      skinny_row_values(a.x + (size_t)(unit / a.z_chunks) * a.K, a.K, v);
      inv = skinny_inverse_rms(v, a.K, a.eps, red_sum);
    }
    skinny_lora_a_unit<1024, RMS>(a.x, a.gamma, inv, a.lora_a, a.idx, a.z_part, unit, a.K, a.n_adapters, a.r, a.z_chunks,
                                  a.z_chunk_k, zw);
    return;
  }
  const uint32_t m = blockIdx.x;
  const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
  const uint16_t* xr = a.x + (size_t)m * a.K;
  float v[2][8];
  skinny_row_values(xr, a.K, v);
  if (RMS) {
    const float inv = skinny_inverse_rms(v, a.K, a.eps, red_sum);
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const uint32_t k0 = (j * 1024u + tid) * 8u;
      if (k0 < a.K) {
        const float4 g0 = *reinterpret_cast<const float4*>(a.gamma + k0);
        const float4 g1 = *reinterpret_cast<const float4*>(a.gamma + k0 + 4);
        const float gm[8] = {g0.x, g0.y, g0.z, g0.w, g1.x, g1.y, g1.z, g1.w};
        uint32_t packed[4];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          float t = v[j][e] * inv;
          t = t * gm[e];
          const uint32_t b = f32_to_bf16_bits(t);
          v[j][e] = __uint_as_float(b << 16);
          if (e & 1) packed[e >> 1] |= b << 16; else packed[e >> 1] = b;
        }
        const uint4 o = make_uint4(packed[0], packed[1], packed[2], packed[3]);
        if (a.xn_aux) *reinterpret_cast<uint4*>(a.xn_aux + (size_t)m * a.K + k0) = o;
      }
    }
  }
  float amax = 0.0f;
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int e = 0; e < 8; ++e) amax = fmaxf(amax, fabsf(v[j][e]));
  amax = wave_max(amax);
  if (lane == 0) red_max[wave] = amax;
  __syncthreads();
  amax = 0.0f;
#pragma unroll
  for (int w = 0; w < 16; ++w) amax = fmaxf(amax, red_max[w]);
  const float scale = amax > 0.0f ? amax / 127.0f : 1.0f, rscale = __builtin_amdgcn_rcpf(scale);
  const bool ordinary = code_scale_ordinary(scale);
  if (tid == 0) {
    a.sx[m] = scale;
    if (a.scales_rm) a.scales_rm[m] = scale;
    if (a.lora_scaling) {
      int ad = a.idx ? a.idx[m] : 0;
      ad = ad < 0 ? 0 : (ad >= (int)a.n_adapters ? (int)a.n_adapters - 1 : ad);
      a.row_scaling[m] = a.lora_scaling[ad];
    }
  }
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const uint32_t k0 = (j * 1024u + tid) * 8u;
    if (k0 >= a.K_pad) continue;
    uint32_t lo = 0, hi = 0;
    if (k0 < a.K) {
      float q[2][4];
      if (ordinary) {  // workgroup-uniform; a NaN (which the row's maximum passes over) takes the lower limit either way
#pragma unroll
        for (int e = 0; e < 8; ++e) q[e >> 2][e & 3] = fmaxf(code_quotient(v[j][e], scale, rscale), -127.0f);
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) q[e >> 2][e & 3] = fminf(fmaxf(v[j][e] / scale, -127.0f), 127.0f);
      }
      lo = code_bytes4(q[0]);
      hi = code_bytes4(q[1]);
      if (a.codes_rm) *reinterpret_cast<uint2*>(a.codes_rm + (size_t)m * a.K + k0) = make_uint2(lo, hi);
    }
    *reinterpret_cast<uint2*>(a.xq + packed_offset(m, k0, a.KB)) = make_uint2(lo, hi);
  }
}

// ---------------------------------------------------------------------------------------
constexpr uint32_t kSkinnyStreamWaves = 8;   // waves of a stream workgroup; they split K
constexpr uint32_t kSkinnyStreamThreads = kSkinnyStreamWaves * 64u;

struct SkinnyStreamArgs {
  const unsigned char* xq;   // packed codes of the single 32-row block
  const unsigned char* wp;   // packed weight
  const float* z_part;       // f32 [z_chunks][32][kMaxRank]
  const float* sx;           // f32 [32]
  const float* sw;           // f32 [N]
  const uint16_t* lora_b;    // bf16 [n_adapters, r, N] or null
  const uint16_t* bsel;      // B regrouped (skinny_regroup_b; NS = 1, RB = 1), or null: gathered from lora_b
  const float* row_scaling;  // f32 [32]: lora_scaling[idx[m]] (from the quantizer launch)
  const int32_t* idx;        // adapter per row or null
  const uint16_t* residual;  // bf16 [M, N] or null
  uint16_t* out;             // bf16 [M, N], or [M, N / 2] with swiglu
  int32_t* aux_acc;          // int32 [M, N] or null
  uint32_t M, N, K, KB, pairs_per_wave, n_adapters, r, z_chunks, n_groups;
  uint32_t swiglu;
  uint32_t z_off;            // bytes of the staged B in front of the staged z partials (skinny_stream_lds)
  uint32_t tail_off;         // ... of both (or of the accumulators that take their place), in front of the rest
};

// LDS of a stream workgroup: [staged B rows | staged z partials], the same bytes later the waves'
// accumulators; behind them z, the per-output scales and the odd-rank sums.
struct SkinnyStreamLds { uint32_t z_off, tail_off, bytes; };
constexpr uint32_t kSkinnyZlStride = 65;  // floats between two rows of z: four rows a wave reads at a time in four banks
constexpr uint32_t kSkinnyTailBytes = 16u * kSkinnyZlStride * 4u + 5u * 2048u + 2u * 1024u + 64u;
inline SkinnyStreamLds skinny_stream_lds(uint32_t m, uint32_t r, uint32_t z_chunks, uint32_t ns, uint32_t rb, bool kept_b) {
  SkinnyStreamLds L{};
  const uint32_t rows = m < 16u ? m : 16u, rpad = round_up(r, 4u);
  const uint32_t per_piece = r <= 32u ? 8u : 4u;  // rows of z per KiB
  const uint32_t b_bytes = kept_b ? round_up(rows * skinny_b_ranks(r) * 32u, 1024u) : rows * rpad * 64u;
  L.z_off = r ? round_up(b_bytes + 4u * 64u, 1024u) : 0u;
  const uint32_t staged = L.z_off + (r ? z_chunks * ((rows + per_piece - 1u) / per_piece) * 1024u : 0u);
  const uint32_t red = kSkinnyStreamWaves * ns * rb * 1024u;
  L.tail_off = staged > red ? staged : red;
  L.bytes = L.tail_off + kSkinnyTailBytes;
  return L;
}

// Every workgroup owns NS slices of 16 packed weight columns for all of K and finishes them itself;
// nothing crosses workgroups.
//  * Its eight waves each stream a K range of the weight from HBM straight into
//    v_mfma_i32_16x16x64_i8 operands (a lane loads its 16 bytes from the 1 KiB fragment blocks:
//    column c of a block pair's four 16-wide k chunks) and are reduced through LDS.  KP is what a wave
//    keeps in flight: KP 64-wide k steps of every slice; a longer share of K takes further rounds.
//  * Finish: (float(acc) * sx) * sw + s * (z @ B) + residual, one bf16 cast, or SwiGLU.  z[m][r] is the
//    fixed-order sum of the LoRA-A partials; the rank sum runs as an even and an odd chain.
// Slice (nb, half) is the original columns 128 G + 4 (16 half + c) + j, c = 0..15, of column block
// nb = 4 G + j.  NS = 2 takes j = 2 p and 2 p + 1: adjacent column pairs, so a dword of B (or of the output)
// is both columns, and a fused gate/up projection's (gate, up) pair ends in one thread.  The units of a
// 128-column group share stretches of B and of memory pages; they get workgroup ids that land on one XCD
// (ids are dealt round-robin to the XCDs).
//
// Bound by HBM, and for short weights by the latency of the launch.  What the finish step works with (the
// rows' B, the z partials, scales, residual) takes no registers -- the MFMA operands take all there are --
// the waves copy it into the LDS with direct-to-LDS loads, the first loads they issue (a wave's loads return
// in order), and form the low-rank term from there while the weight is on its way.  B is gathered as dwords
// (64 per instruction: four ranks x sixteen columns) straight from its [rank, N] rows: half or all of every
// 64 bytes fetched is used, and no regrouped copy of it is written and read back, which cost 2 x 25 MB for
// sixteen adapters of a 24576-wide projection whenever an adapter had changed.  A loop that keeps its adapters has B
// regrouped once (skinny_regroup_b) and then finds a unit's in whole KiBs.
// Measured: 4096 x 24576 with SwiGLU, 16 rows, 16 adapters of rank 32: 22.9 us for 126 MB (5.5 TB/s), the whole
// call 29 us against 139 us on 128 x 128 tiles behind the tiled quantizer (which such a call took before);
// 2560 x 6144, one row, rank 64: 8.1 us against 18.3 us with B's loads behind the weight's; 12288 x 4096,
// 16 rows: 14.6 us, 13.0 us from the regrouped B.
// Rows 16..31 (RB = 2) share the weight operands; their B is staged in a second step behind the stream.
template <int NS, int RB, int KP>
__global__ __launch_bounds__(kSkinnyStreamThreads, (NS + RB) * KP <= 24 ? 4 : 2)
void skinny_stream_kernel(SkinnyStreamArgs a) {
  extern __shared__ __attribute__((aligned(1024))) unsigned char sk_lds[];
  const uint32_t tid = threadIdx.x, lane = tid & 63u;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  constexpr uint32_t kUnits = 8u / NS;  // of a 128-column group
  const uint32_t slot = blockIdx.x >> 3;
  const uint32_t grp = (slot / kUnits) * 8u + (blockIdx.x & 7u), unit = slot % kUnits;
  if (grp >= a.n_groups) return;
  const uint32_t j0 = NS == 2 ? (unit >> 1) * 2u : unit >> 1, chalf = unit & 1u;
  const uint32_t c16 = lane & 15u, q = lane >> 4;        // MFMA operand: column / row c16, k chunk q
  const uint32_t pc = 16u * chalf + c16;                 // packed column inside its block
  // byte offsets inside a pair of 1 KiB blocks: chunk q sits in block q/2, k half q%2
  const uint32_t w_lane_off = (q >> 1) * kBlockBytes + (pc + 32u * (q & 1u)) * 16u;
  // (rows beyond M repeat the last one: fewer cache lines, and their results are dropped)
  const uint32_t xrow0 = c16 < a.M ? c16 : a.M - 1u, xrow1 = c16 + 16u < a.M ? c16 + 16u : a.M - 1u;
  const uint32_t x_chunk = (q >> 1) * kBlockBytes + 512u * (q & 1u);
  const uint32_t n_pairs = a.KB >> 1;
  uint32_t p0 = wave * a.pairs_per_wave, p1 = p0 + a.pairs_per_wave;
  if (p0 > n_pairs) p0 = n_pairs;
  if (p1 > n_pairs) p1 = n_pairs;
  // Buffer resources that end with the wave's share of K: a step beyond it reads zeros without touching
  // memory, so the loads need no clamps and the MFMAs no conditions (and no 64-bit address per load).
  __amdgpu_buffer_rsrc_t wrsrc[NS];
#pragma unroll
  for (int s = 0; s < NS; ++s)
    wrsrc[s] = __builtin_amdgcn_make_buffer_rsrc(const_cast<unsigned char*>(a.wp) + (size_t)(grp * 4u + j0 + s) * a.KB * kBlockBytes,
                                                 0, (int)(p1 * 2u * kBlockBytes), 0x00020000);
  const __amdgpu_buffer_rsrc_t xrsrc =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<unsigned char*>(a.xq), 0, (int)(p1 * 2u * kBlockBytes), 0x00020000);
  const uint32_t x_lane_off0 = x_chunk + xrow0 * 16u, x_lane_off1 = x_chunk + xrow1 * 16u;

  // ---- finish step mapping: thread -> output row, columns fn .. fn + NS - 1, and (RB = 1) a rank parity.
  // Each use derives it anew from the thread id behind an opaque copy: kept across the stream it would take
  // registers that the operands in flight need.
  struct Finish {
    uint32_t t8, t256, lane, fe, frow16, frow, c16, fn, srow, scol;
    bool valid;
  };
  auto finish_map = [&]() -> Finish {
    uint32_t t = threadIdx.x;
    asm volatile("" : "+v"(t));
    Finish f;
    f.t8 = t >> 8; f.t256 = t & 255u; f.lane = t & 63u;
    f.fe = (t >> 6) & 3u;
    f.c16 = t & 15u;
    f.frow16 = 4u * (f.lane >> 4) + f.fe;                  // row inside its half
    f.frow = (RB == 2 ? 16u * f.t8 : 0u) + f.frow16;
    f.fn = 128u * grp + 4u * (16u * chalf + f.c16) + j0;
    f.valid = f.frow < a.M && f.fn < a.N;                  // (NS = 2 needs an even N: both columns exist or none)
    // Lanes without an output read element 0 instead of selecting on the loaded value.
    f.srow = f.valid ? f.frow : 0u;
    f.scol = f.valid ? f.fn : 0u;
    return f;
  };
  const bool lora = a.lora_b != nullptr;
  const bool kept_b = NS == 1 && RB == 1 && a.bsel != nullptr;  // kernel-uniform
  // an odd number of values in B: the dword gathers would read two bytes behind it (NS = 2: N is even)
  const bool odd_b = NS == 1 && (a.n_adapters & a.r & a.N & 1u);
  const uint32_t rpad = (a.r + 3u) & ~3u;
  const uint32_t rp = a.r <= 32u ? 32u : 64u;            // ranks of a staged z row
  uint32_t* const bst = reinterpret_cast<uint32_t*>(sk_lds);
  const float* const zst = reinterpret_cast<const float*>(sk_lds + a.z_off);
  int* const red = reinterpret_cast<int*>(sk_lds);       // [wave][slice][row half][4][64], once the staged data is spent
  float* const zl = reinterpret_cast<float*>(sk_lds + a.tail_off);
  uint32_t* const fst = reinterpret_cast<uint32_t*>(zl + 16u * kSkinnyZlStride);  // [5][512]: sx, sw, scaling, residual, sw of the second column
  float* const low_odd = reinterpret_cast<float*>(fst + 5u * 512u);               // [NS][256]
  uint32_t* const odd_base = reinterpret_cast<uint32_t*>(low_odd + 512u);          // [16]
  const uint32_t lds0 = (uint32_t)(uintptr_t)(lptr_t)sk_lds;
  const uint32_t fst_addr = lds0 + a.tail_off + 16u * kSkinnyZlStride * 4u + wave * 256u;

  // adapters of the rows this wave stages (wave, wave + 8, ...)
  int ads[2 * RB];
#pragma unroll
  for (uint32_t i = 0; i < 2u * RB; ++i) {
    const uint32_t m = wave + 8u * i;
    int ad = (lora && a.idx && m < a.M) ? a.idx[m] : 0;
    ad = ad < 0 ? 0 : (ad >= (int)a.n_adapters ? (int)a.n_adapters - 1 : ad);
    ads[i] = __builtin_amdgcn_readfirstlane(ad);
  }
  // B rows and z partials of rows 16 hf .. 16 hf + 15 on their way into the LDS
  auto stage_half = [&](uint32_t hf) {
    const uint32_t rows = a.M - 16u * hf < 16u ? a.M - 16u * hf : 16u;
    if (kept_b) {  // 1 KiB at a time, whole rows of one row quad (the quads 64 bytes apart: bank groups of their own)
      const uint32_t row_bytes = skinny_b_ranks(a.r) * 32u, pieces = (rows * row_bytes + 1023u) / 1024u, quad_bytes = 4u * row_bytes;
      const unsigned char* src = reinterpret_cast<const unsigned char*>(a.bsel) + (size_t)(grp * 8u + unit) * a.M * row_bytes;
      for (uint32_t i = wave; i < pieces; i += kSkinnyStreamWaves)
        lds_load_1k(src, i * 1024u + lane * 16u, lds0 + i * 1024u + (i * 1024u / quad_bytes) * 64u);
    } else
#pragma unroll
    for (uint32_t mi = 0; mi < 2u; ++mi) {
      const uint32_t m = wave + 8u * mi;
      if (m >= rows) break;
      const int ad = (RB == 2 && hf) ? ads[RB == 2 ? 2 + mi : mi] : ads[mi];
      // (the gathers are dwords on 4-byte boundaries: an adapter that starts in the middle of one -- odd N and
      // rank -- is addressed from the boundary in front of it)
      const size_t e0 = (size_t)ad * a.r * a.N;
      const uint32_t odd0 = (uint32_t)(e0 & 1u);
      if (lane == 0) odd_base[m] = odd0;
      const uint16_t* brow = a.lora_b + (e0 - odd0);
      const uint32_t dst = lds0 + m * rpad * 64u + (m >> 2) * 64u;
      uint32_t col = 128u * grp + 4u * pc + j0;
      if (col + NS > a.N) col = 0u;
      if (!(odd_b && ad + 1 == (int)a.n_adapters)) {
        for (uint32_t i = 0; i < rpad / 4u; ++i) {
          uint32_t rr = 4u * i + q;
          rr = rr < a.r ? rr : a.r - 1u;
          lds_gather_dword(brow, ((rr * a.N + col + odd0) * 2u) & ~3u, dst + i * 256u);
        }
      } else {  // B's last value has no whole dword: it is loaded by itself
        for (uint32_t i = 0; i < rpad / 4u; ++i) {
          uint32_t rr = 4u * i + q;
          rr = rr < a.r ? rr : a.r - 1u;
          if (rr + 1u == a.r && col + 1u == a.N) bst[(dst - lds0) / 4u + i * 64u + lane] = brow[rr * a.N + col + odd0];
          else lds_gather_dword(brow, ((rr * a.N + col + odd0) * 2u) & ~3u, dst + i * 256u);
        }
      }
    }
    const uint32_t per_piece = 1024u / (rp * 4u), pieces = (rows + per_piece - 1u) / per_piece;
    const uint32_t lanes_row = rp / 4u;  // lanes of 16 bytes per row
    for (uint32_t i = wave; i < pieces * a.z_chunks; i += kSkinnyStreamWaves) {
      const uint32_t ch = i / pieces, pi = i % pieces;
      const uint32_t row = 16u * hf + pi * per_piece + lane / lanes_row;
      const uint32_t voff = ((ch * (uint32_t)kSkinnyMaxRows + row) * (uint32_t)kMaxRank) * 4u + (lane % lanes_row) * 16u;
      lds_load_1k(reinterpret_cast<const unsigned char*>(a.z_part), voff, lds0 + a.z_off + i * 1024u);
    }
  };
  // z of the staged rows, then the thread's share of the low-rank term (every wave has its pieces: a
  // barrier stands in front)
  auto low_rank = [&](uint32_t hf, float (&low)[NS]) {
    const Finish f = finish_map();
    const uint32_t rows = a.M - 16u * hf < 16u ? a.M - 16u * hf : 16u;
    const uint32_t per_piece = 1024u / (rp * 4u), chunk_stride = (rows + per_piece - 1u) / per_piece * 256u;
    for (uint32_t zi = tid; zi < rows * rp; zi += kSkinnyStreamThreads) {
      float s4[4] = {0.f, 0.f, 0.f, 0.f};  // four interleaved partial sums, combined in a fixed order
      for (uint32_t ch = 0; ch < a.z_chunks; ch += 4u) {
#pragma unroll
        for (uint32_t u = 0; u < 4u; ++u)
          if (ch + u < a.z_chunks) s4[u] += zst[(ch + u) * chunk_stride + zi];
      }
      zl[(zi / rp) * kSkinnyZlStride + zi % rp] = ((s4[0] + s4[1]) + s4[2]) + s4[3];
    }
    __syncthreads();
    if ((RB == 1 || f.t8 == hf) && f.frow < a.M) {
      const uint32_t* bl = bst + f.frow16 * rpad * 16u + (f.frow16 >> 2) * 16u + f.c16;
      const float* zr = zl + f.frow16 * kSkinnyZlStride;
      const uint32_t odd_row = NS == 1 ? odd_base[f.frow16] : 0u;
      const uint32_t r0 = RB == 2 ? 0u : f.t8, step = RB == 2 ? 1u : 2u;
      if (kept_b) {
        const uint32_t ranks = skinny_b_ranks(a.r);
        const uint16_t* bk = reinterpret_cast<const uint16_t*>(sk_lds) + f.frow16 * ranks * 16u + (f.frow16 >> 2) * 32u + (f.t8 * 16u + f.c16) * (ranks / 2u);
        for (uint32_t t0 = 0; t0 < ranks / 2u; t0 += 8u) {  // (z and B are zeros beyond the rank: they add nothing)
          const v8us b8 = *reinterpret_cast<const v8us*>(bk + t0);
#pragma unroll
          for (uint32_t e = 0; e < 8u; ++e) low[0] = fmaf(zr[2u * (t0 + e) + f.t8], bf16_bits_to_f32(b8[e]), low[0]);
        }
      } else
#pragma unroll 2
      for (uint32_t r = r0; r < a.r; r += step) {
        const uint32_t w = bl[r * 16u];
        const float z = zr[r];
        if constexpr (NS == 2) {
          low[0] = fmaf(z, __uint_as_float(w << 16), low[0]);
          low[1] = fmaf(z, __uint_as_float(w & 0xffff0000u), low[1]);
        } else {
          const bool odd = ((r * a.N + f.scol + odd_row) & 1u) != 0;  // which half of the dword holds the column
          low[0] = fmaf(z, __uint_as_float(odd ? w & 0xffff0000u : w << 16), low[0]);
        }
      }
    }
    if constexpr (RB == 1) {  // the two rank parities of an output, added in a fixed order
      if (f.t8 == 1u) {
#pragma unroll
        for (int s = 0; s < NS; ++s) low_odd[s * 256 + f.t256] = low[s];
      }
      __syncthreads();
      if (f.t8 == 0u) {
#pragma unroll
        for (int s = 0; s < NS; ++s) low[s] = low[s] + low_odd[s * 256 + f.t256];
      }
    }
  };

  if (lora) stage_half(0);  // kernel-uniform
  if (RB == 2 || wave < 4u) {  // the output threads: thread tid finds its values at fst[.][tid]
    const Finish f = finish_map();
    const uint32_t srow = f.srow, scol = f.scol, res_elem = srow * a.N + scol;  // (M * N is below 2^32)
    lds_gather_dword(a.sx, srow * 4u, fst_addr);
    lds_gather_dword(a.sw, scol * 4u, fst_addr + 2048u);
    if (lora) lds_gather_dword(a.row_scaling, srow * 4u, fst_addr + 4096u);
    if (a.residual) {  // (the last of an odd number of values: as above)
      if (NS == 1 && (a.M & a.N & 1u) && res_elem + 1u == a.M * a.N) fst[1536u + threadIdx.x] = a.residual[res_elem];
      else lds_gather_dword(a.residual, (res_elem * 2u) & ~3u, fst_addr + 6144u);
    }
    if constexpr (NS == 2) lds_gather_dword(a.sw, (scol + 1u < a.N ? scol + 1u : scol) * 4u, fst_addr + 8192u);
  }

  // accumulators take turns, so that no MFMA waits for the one before it (integer sums: any order)
  constexpr int kTurns = NS * RB >= 4 ? 1 : 4 / (NS * RB);
  v4i acc[kTurns][NS][RB];
  float low[NS];
#pragma unroll
  for (int s = 0; s < NS; ++s) low[s] = 0.f;

  // One round: KP steps of every slice requested, then multiplied.  The first one forms the low-rank term in
  // between (and starts the accumulators, which so take no registers while it does).
  auto round = [&](uint32_t base, auto first) {
    v4i wf[KP][NS], xf[KP][RB];
    // (the codes first: they come from the L2 and are in the registers long before the weight, whose
    // requests the memory takes at its own pace)
#pragma unroll
    for (uint32_t t = 0; t < (uint32_t)KP; ++t)
#pragma unroll
      for (int b = 0; b < RB; ++b)
        xf[t][b] = __builtin_amdgcn_raw_buffer_load_b128(xrsrc, (b ? x_lane_off1 : x_lane_off0) + (base + t) * 2u * kBlockBytes, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (uint32_t t = 0; t < (uint32_t)KP; ++t)
#pragma unroll
      for (int s = 0; s < NS; ++s)  // (non-temporal)
        wf[t][s] = __builtin_amdgcn_raw_buffer_load_b128(wrsrc[s], w_lane_off + (base + t) * 2u * kBlockBytes, 0, 2);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (decltype(first)::value) {
      if (lora) {  // kernel-uniform: the low-rank term, while the weight is on its way
        // the staged operands are the wave's oldest loads: a wait that leaves the code and weight loads
        // outstanding has them
        asm volatile("s_waitcnt vmcnt(%0)" :: "n"(KP * (NS + RB)) : "memory");
        __syncthreads();  // ... and the other waves' pieces
        low_rank(0u, low);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int u = 0; u < kTurns; ++u)
#pragma unroll
        for (int s = 0; s < NS; ++s)
#pragma unroll
          for (int b = 0; b < RB; ++b) acc[u][s][b] = v4i{0, 0, 0, 0};
    }
#pragma unroll
    for (uint32_t t = 0; t < (uint32_t)KP; ++t)
#pragma unroll
      for (int s = 0; s < NS; ++s)
#pragma unroll
        for (int b = 0; b < RB; ++b)
          acc[t % kTurns][s][b] = __builtin_amdgcn_mfma_i32_16x16x64_i8(xf[t][b], wf[t][s], acc[t % kTurns][s][b], 0, 0, 0);
  };
  round(p0, std::true_type{});
#pragma unroll 1
  for (uint32_t base = p0 + (uint32_t)KP; base < p1; base += (uint32_t)KP) round(base, std::false_type{});
  if constexpr (RB == 2) {
    if (lora) {  // rows 16..31: their B and z into the same bytes
      __syncthreads();
      stage_half(1);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
      low_rank(1u, low);
    }
  }
  __syncthreads();  // the staged operands are spent
#pragma unroll
  for (int s = 0; s < NS; ++s)
#pragma unroll
    for (int b = 0; b < RB; ++b)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        int v = acc[0][s][b][e];
#pragma unroll
        for (int u = 1; u < kTurns; ++u) v += acc[u][s][b][e];
        red[(((wave * NS + s) * RB + b) * 4u + e) * 64u + lane] = v;
      }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (without LoRA nothing has waited for the staged scales yet)
  __syncthreads();
  const Finish f = finish_map();
  if ((RB == 1 && f.t8 == 1u) || !f.valid) return;
  const float f_sx = __uint_as_float(fst[tid]);
  const float f_s = lora ? __uint_as_float(fst[1024u + tid]) : 0.f;
  float y[NS];
  int sum[NS];
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    sum[s] = 0;
#pragma unroll
    for (uint32_t w = 0; w < kSkinnyStreamWaves; ++w)
      sum[s] += red[(((w * NS + s) * RB + (RB == 2 ? f.t8 : 0u)) * 4u + f.fe) * 64u + f.lane];
    y[s] = ((float)sum[s] * f_sx) * __uint_as_float(fst[(s == 0 ? 512u : 2048u) + tid]);
    if (lora) {
      const float l = low[s] * f_s;
      y[s] = y[s] + l;
    }
  }
  const size_t o = (size_t)f.frow * a.N + f.fn;
  if (a.aux_acc) {
#pragma unroll
    for (int s = 0; s < NS; ++s) a.aux_acc[o + s] = sum[s];
  }
  if constexpr (NS == 2) {
    const uint32_t pair = pack_bf16x2(y[0], y[1]);
    if (a.swiglu) {  // kernel-uniform: gate and up are rounded to bf16 first
      a.out[(size_t)f.frow * (a.N >> 1) + (f.fn >> 1)] =
          (uint16_t)f32_to_bf16_bits(swiglu_f32(__uint_as_float(pair << 16), __uint_as_float(pair & 0xffff0000u)));
    } else {
      *reinterpret_cast<uint32_t*>(a.out + o) = pair;
    }
  } else {
    if (a.residual) {
      const uint32_t w = fst[1536u + tid];
      y[0] = y[0] + __uint_as_float((o & 1u) ? w & 0xffff0000u : w << 16);
    }
    a.out[o] = (uint16_t)f32_to_bf16_bits(y[0]);
  }
}

}  // namespace w8a8
