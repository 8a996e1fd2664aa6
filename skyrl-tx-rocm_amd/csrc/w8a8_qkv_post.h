// Qwen3.5 attention input stage behind the fused QKV projection
// (skyrl/tx/kernels/qwen3_5_qkv_lora.py:216-286): split the interleaved projection, RMSNorm with
// (1 + weight) over every Q and K head, partial RoPE on Q and K, V and the Q gates copied out.
// The projection itself (RMSNorm prologue, W8A8 GEMM, LoRA) is the ordinary forward call; this
// kernel reads its bf16 output once and writes q, k, v, gate once (memory-bound).
//
// Layout of a fused row: per kv head one group [q_0 g_0 ... q_{qpk-1} g_{qpk-1} k v], every chunk
// head_dim wide (qwen3_5_qkv_lora.py:40-46).  One workgroup per row; a wave takes a (q, gate) or a
// (k, v) pair at a time.
#pragma once
#include "w8a8_device.h"

namespace w8a8 {

constexpr uint32_t kQkvMaxHeadDim = 512;

// sum / D in float64, rounded to float32; a power of two is divided by as a product, which is exact and a sixth of the instructions.
__device__ inline float qkv_mean(double sum, uint32_t D) {
  return (float)((D & (D - 1u)) == 0u ? sum * (1.0 / (double)D) : sum / (double)D);  // (kernel-uniform; 1 / D is formed once)
}
// Four elements a lane and piece of the two chunks of a unit.  A wave asks for the next unit's before it works on one, and for its
// first before the rotation's table is formed; the norm weights stay in registers.  Instructions bound it as much as memory
// (40960 heads of 300 each, float64 sums and two divisions among them: the loads ahead alone gave the pull-back 0.2 us; the rest
// is the mean as a product and the weights held).  2048 rows of 16 + 4 heads of 256: forward 22.6 us, now 21.1 (84 MB, 4.0 TB/s);
// backward 40.8, now 31.5 (126 MB).
// NP: pieces, one for heads of up to 256.
template <uint32_t NP> struct QkvPieces { uint2 a[NP], b[NP]; };
template <uint32_t NP>
__device__ inline void qkv_fetch(QkvPieces<NP>& t, const uint16_t* a, const uint16_t* b, uint32_t D, uint32_t lane) {
#pragma unroll
  for (uint32_t j = 0; j < NP; ++j) {
    const uint32_t i = 4u * lane + 256u * j;
    t.a[j] = t.b[j] = make_uint2(0, 0);
    if (i < D) {
      t.a[j] = *reinterpret_cast<const uint2*>(a + i);
      t.b[j] = *reinterpret_cast<const uint2*>(b + i);
    }
  }
}
// Norm weight i as float32: the tensor may be bf16 (the model's own; converted by the caller it took a launch of 2 us for each).
__device__ inline float qkv_weight(const float* w, uint32_t i, bool bf16) {
  return bf16 ? bf16_bits_to_f32(reinterpret_cast<const uint16_t*>(w)[i]) : w[i];  // (kernel-uniform)
}
// 1 + weight of the lane's elements
template <uint32_t NP>
__device__ inline void qkv_weights(float4 (&w)[NP], const float* src, bool bf16, uint32_t D, uint32_t lane) {
#pragma unroll
  for (uint32_t j = 0; j < NP; ++j) {
    const uint32_t i = 4u * lane + 256u * j;
    float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
    if (i < D) {
      if (bf16) {
        const uint2 r = *reinterpret_cast<const uint2*>(reinterpret_cast<const uint16_t*>(src) + i);
        v = make_float4(__uint_as_float(r.x << 16), __uint_as_float(r.x & 0xffff0000u), __uint_as_float(r.y << 16), __uint_as_float(r.y & 0xffff0000u));
      } else {
        v = *reinterpret_cast<const float4*>(src + i);
      }
    }
    w[j] = make_float4(1.0f + v.x, 1.0f + v.y, 1.0f + v.z, 1.0f + v.w);
  }
}

struct QkvPostArgs {
  const uint16_t* fused;   // bf16 [M, width]
  const float* q_w;        // f32 [D] delta weights of the Q norm (w_bf16: bf16, like k_w)
  const float* k_w;        // f32 [D]
  const int32_t* pos;      // int32 [M]
  uint16_t* q;             // bf16 [M, Hq, D]
  uint16_t* k;             // bf16 [M, Hkv, D]
  uint16_t* v;             // bf16 [M, Hkv, D]
  uint16_t* gate;          // bf16 [M, Hq * D]
  uint32_t M, Hq, Hkv, D, rot, width;
  float theta, eps;
  uint32_t w_bf16;
};

template <uint32_t NP>
__global__ __launch_bounds__(256) void qkv_post_kernel(QkvPostArgs a) {
  __shared__ float sn[kQkvMaxHeadDim / 2], cs[kQkvMaxHeadDim / 2];
  __shared__ float buf[4][kQkvMaxHeadDim];
  const uint32_t row = blockIdx.x, tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
  if (row >= a.M) return;
  const uint32_t half = a.rot / 2u;
  const uint32_t qpk = a.Hq / a.Hkv;
  const uint32_t group_width = (qpk * 2u + 2u) * a.D;
  const uint16_t* frow = a.fused + (size_t)row * a.width;
  const uint32_t units = a.Hq + a.Hkv;
  // four consecutive elements per lane (8-byte accesses) where the geometry allows it
  const bool vec4 = (a.D & 3u) == 0 && (half & 3u) == 0 && (a.width & 3u) == 0;
  auto chunk = [&](uint32_t u) -> const uint16_t* {  // of a unit's head; the one that passes through lies D behind it
    return frow + (u < a.Hq ? u / qpk * group_width + (u % qpk) * 2u * a.D : (u - a.Hq) * group_width + qpk * 2u * a.D);
  };
  QkvPieces<NP> next;
  float4 wq[NP], wk[NP];
  if (vec4) {
    if (wave < units) qkv_fetch(next, chunk(wave), chunk(wave) + a.D, a.D, lane);
    qkv_weights(wq, a.q_w, a.w_bf16 != 0u, a.D, lane);
    qkv_weights(wk, a.k_w, a.w_bf16 != 0u, a.D, lane);
  }
  // angle[i] = position / theta^(2 i / rot), all float32 (qwen3_5_qkv_lora.py:119-127)
  const float position = (float)a.pos[row];
  for (uint32_t i = tid; i < half; i += 256u) {
    const float fraction = (2.0f * (float)i) / (float)a.rot;
    const float angle = position / powf(a.theta, fraction);
    sn[i] = sinf(angle);
    cs[i] = cosf(angle);
  }
  __syncthreads();
  for (uint32_t u = wave; u < units; u += 4u) {  // wave-uniform
    const bool is_q = u < a.Hq;
    const uint32_t g = is_q ? u / qpk : u - a.Hq;
    const uint32_t off = g * group_width + (is_q ? (u % qpk) * 2u * a.D : qpk * 2u * a.D);
    const float* w = is_q ? a.q_w : a.k_w;
    uint16_t* normed = is_q ? a.q + ((size_t)row * a.Hq + u) * a.D : a.k + ((size_t)row * a.Hkv + g) * a.D;
    uint16_t* copied = is_q ? a.gate + ((size_t)row * a.Hq + u) * a.D : a.v + ((size_t)row * a.Hkv + g) * a.D;
    if (vec4) {
      const QkvPieces<NP> t = next;
      if (u + 4u < units) qkv_fetch(next, chunk(u + 4u), chunk(u + 4u) + a.D, a.D, lane);
      // the second chunk of the pair (gate or v) passes through
#pragma unroll
      for (uint32_t j = 0; j < NP; ++j)
        if (4u * lane + 256u * j < a.D) *reinterpret_cast<uint2*>(copied + 4u * lane + 256u * j) = t.b[j];
      // RMSNorm over the head: mean = float(sum_f64(x^2) / D), inv = 1 / sqrt(mean + eps) (IEEE),
      // n = bf16((x * inv) * (1 + w)); D <= 512: at most two pieces per lane, kept in registers
      const uint2 (&raw)[NP] = t.a;
      double ss = 0.0;
#pragma unroll
      for (uint32_t j = 0; j < NP; ++j) {
        const uint32_t i = 4u * lane + 256u * j;
        if (i < a.D) {
          const float x0 = __uint_as_float(raw[j].x << 16), x1 = __uint_as_float(raw[j].x & 0xffff0000u);
          const float x2 = __uint_as_float(raw[j].y << 16), x3 = __uint_as_float(raw[j].y & 0xffff0000u);
          ss += (double)x0 * (double)x0 + (double)x1 * (double)x1 + (double)x2 * (double)x2 + (double)x3 * (double)x3;
        }
      }
      ss = wave_sum(ss);
      const float mean = qkv_mean(ss, a.D);
      const float inv = 1.0f / sqrtf(mean + a.eps);
#pragma unroll
      for (uint32_t j = 0; j < NP; ++j) {
        const uint32_t i = 4u * lane + 256u * j;
        if (i < a.D) {
          const float4 w4 = is_q ? wq[j] : wk[j];
          const float x[4] = {__uint_as_float(raw[j].x << 16), __uint_as_float(raw[j].x & 0xffff0000u),
                              __uint_as_float(raw[j].y << 16), __uint_as_float(raw[j].y & 0xffff0000u)};
          const float wv[4] = {w4.x, w4.y, w4.z, w4.w};
          float4 n4;
          float* np_ = &n4.x;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            float y = x[e] * inv;
            y = y * wv[e];
            np_[e] = bf16_round_f32(y);
          }
          *reinterpret_cast<float4*>(&buf[wave][i]) = n4;
        }
      }
      // the wave reads what other lanes of the same wave wrote: LDS operations of a wave complete
      // in order, the barrier-free hand-over only needs them drained
      __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (uint32_t j = 0; j < NP; ++j) {
        const uint32_t i = 4u * lane + 256u * j;
        if (i < a.D) {
          float4 o4 = *reinterpret_cast<const float4*>(&buf[wave][i]);
          if (i < a.rot) {
            // halves (i, i + rot / 2): [first cos - second sin, first sin + second cos], products in float32
            float* o = &o4.x;
            if (i < half) {
              const float4 s2 = *reinterpret_cast<const float4*>(&buf[wave][i + half]);
              const float* sp = &s2.x;
#pragma unroll
              for (int e = 0; e < 4; ++e) o[e] = o[e] * cs[i + e] - sp[e] * sn[i + e];
            } else {
              const float4 f2 = *reinterpret_cast<const float4*>(&buf[wave][i - half]);
              const float* fp = &f2.x;
#pragma unroll
              for (int e = 0; e < 4; ++e) o[e] = fp[e] * sn[i - half + e] + o[e] * cs[i - half + e];
            }
          }
          *reinterpret_cast<uint2*>(normed + i) = make_uint2(pack_bf16x2(o4.x, o4.y), pack_bf16x2(o4.z, o4.w));
        }
      }
      __builtin_amdgcn_s_waitcnt(0xc07f);
      __builtin_amdgcn_wave_barrier();  // buf[wave] is rewritten by the next unit
      continue;
    }
    // general geometry: one element per lane and step
    for (uint32_t i = lane; i < a.D; i += 64u) copied[i] = frow[off + a.D + i];
    double ss = 0.0;
    for (uint32_t i = lane; i < a.D; i += 64u) {
      const float x = bf16_bits_to_f32(frow[off + i]);
      ss += (double)x * (double)x;
    }
    ss = wave_sum(ss);
    const float mean = (float)(ss / (double)a.D);
    const float inv = 1.0f / sqrtf(mean + a.eps);
    for (uint32_t i = lane; i < a.D; i += 64u) {
      const float x = bf16_bits_to_f32(frow[off + i]);
      float t = x * inv;
      t = t * (1.0f + qkv_weight(w, i, a.w_bf16 != 0u));
      buf[wave][i] = bf16_round_f32(t);
    }
    __builtin_amdgcn_s_waitcnt(0xc07f);
    __builtin_amdgcn_wave_barrier();
    for (uint32_t i = lane; i < a.D; i += 64u) {
      float o = buf[wave][i];
      if (i < a.rot) {
        if (i < half) o = buf[wave][i] * cs[i] - buf[wave][i + half] * sn[i];
        else o = buf[wave][i - half] * sn[i - half] + buf[wave][i] * cs[i - half];
      }
      normed[i] = (uint16_t)f32_to_bf16_bits(o);
    }
    __builtin_amdgcn_s_waitcnt(0xc07f);
    __builtin_amdgcn_wave_barrier();
  }
}

// ---------------------------------------------------------------------------------------
// Pull-back of the kernel above (qwen3_5_qkv_lora.py:391-425): the transposed partial rotation on
// the Q and K cotangents, the RMSNorm pull-back of every Q and K head against the raw projection,
// and the re-interleave with the gate and V cotangents into the cotangent of the fused projection.
// Optionally the cotangents of the two head-norm weights (sums over rows and heads).
//
// Per head, float32 in the order of _apply_partial_rope_transpose (:148-164) and
// _delta_rms_norm_vjp (:97-116):
//   u  = bf16([first cos + second sin, second cos - first sin]) on the rotated part of dy
//   n  = x inv,  p = u (1 + w),  mu = mean(p n),  dx = bf16(inv (p - n mu)),  dw += u n
struct QkvPostBwdArgs {
  const uint16_t* fused;   // bf16 [M, width] raw projection
  const float* q_w;        // f32 [D]
  const float* k_w;        // f32 [D]
  const int32_t* pos;      // int32 [M]
  const uint16_t* dq;      // bf16 [M, Hq, D]
  const uint16_t* dk;      // bf16 [M, Hkv, D]
  const uint16_t* dv;      // bf16 [M, Hkv, D]
  const uint16_t* dgate;   // bf16 [M, Hq * D]
  uint16_t* dfused;        // bf16 [M, width]
  float* partial;          // f32 [gridDim.x][2][D] when the weight cotangents are wanted
  uint32_t M, Hq, Hkv, D, rot, width;
  float theta, eps;
  uint32_t w_bf16;
};

// V consecutive elements per lane and piece (V = 4: 8-byte accesses; V = 1: any geometry); a head
// has at most NP pieces per lane.  Workgroups stride over the rows so that the
// weight cotangents accumulate in registers; WGRAD = false leaves them out altogether.
template <int V, bool WGRAD, uint32_t NP = kQkvMaxHeadDim / (64u * V)>
__global__ __launch_bounds__(256) void qkv_post_bwd_kernel(QkvPostBwdArgs a) {
  __shared__ float sn[kQkvMaxHeadDim / 2], cs[kQkvMaxHeadDim / 2];
  __shared__ float buf[4][kQkvMaxHeadDim];
  const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
  const uint32_t half = a.rot / 2u;
  const uint32_t qpk = a.Hq / a.Hkv;
  const uint32_t group_width = (qpk * 2u + 2u) * a.D;
  const uint32_t units = a.Hq + a.Hkv;
  float wq[NP * V], wk[NP * V];
#pragma unroll
  for (uint32_t e = 0; e < NP * V; ++e) wq[e] = wk[e] = 0.0f;

  QkvPieces<NP> next;  // x and dy of the wave's next unit (V = 4)
  uint2 next_copy[NP];
  float4 one_q[NP], one_k[NP];
  if constexpr (V == 4) {
    qkv_weights(one_q, a.q_w, a.w_bf16 != 0u, a.D, lane);
    qkv_weights(one_k, a.k_w, a.w_bf16 != 0u, a.D, lane);
  }
  auto unit_off = [&](uint32_t u) -> uint32_t {
    return u < a.Hq ? u / qpk * group_width + (u % qpk) * 2u * a.D : (u - a.Hq) * group_width + qpk * 2u * a.D;
  };
  auto fetch = [&](uint32_t row, uint32_t u) {
    const size_t at = u < a.Hq ? ((size_t)row * a.Hq + u) * a.D : ((size_t)row * a.Hkv + (u - a.Hq)) * a.D;
    qkv_fetch(next, a.fused + (size_t)row * a.width + unit_off(u), (u < a.Hq ? a.dq : a.dk) + at, a.D, lane);
    const uint16_t* copy = (u < a.Hq ? a.dgate : a.dv) + at;
#pragma unroll
    for (uint32_t j = 0; j < NP; ++j)
      if (4u * lane + 256u * j < a.D) next_copy[j] = *reinterpret_cast<const uint2*>(copy + 4u * lane + 256u * j);
  };
  for (uint32_t row = blockIdx.x; row < a.M; row += gridDim.x) {
    if constexpr (V == 4) {
      if (wave < units) fetch(row, wave);
    }
    __syncthreads();  // the tables of the previous row are no longer read
    const float position = (float)a.pos[row];
    for (uint32_t i = tid; i < half; i += 256u) {
      const float fraction = (2.0f * (float)i) / (float)a.rot;
      const float angle = position / powf(a.theta, fraction);
      sn[i] = sinf(angle);
      cs[i] = cosf(angle);
    }
    __syncthreads();
    const uint16_t* frow = a.fused + (size_t)row * a.width;
    uint16_t* orow = a.dfused + (size_t)row * a.width;
    for (uint32_t u = wave; u < units; u += 4u) {  // wave-uniform
      const bool is_q = u < a.Hq;
      const uint32_t g = is_q ? u / qpk : u - a.Hq;
      const uint32_t off = g * group_width + (is_q ? (u % qpk) * 2u * a.D : qpk * 2u * a.D);
      const float* w = is_q ? a.q_w : a.k_w;
      const uint16_t* dy = is_q ? a.dq + ((size_t)row * a.Hq + u) * a.D : a.dk + ((size_t)row * a.Hkv + g) * a.D;
      const uint16_t* dcopy = is_q ? a.dgate + ((size_t)row * a.Hq + u) * a.D : a.dv + ((size_t)row * a.Hkv + g) * a.D;
      float x[NP * V], d[NP * V];
      double ss = 0.0;
      QkvPieces<NP> t;
      uint2 t_copy[NP];
      if constexpr (V == 4) {
        t = next;
#pragma unroll
        for (uint32_t j = 0; j < NP; ++j) t_copy[j] = next_copy[j];
        if (u + 4u < units) fetch(row, u + 4u);
      }
#pragma unroll
      for (uint32_t j = 0; j < NP; ++j) {
        const uint32_t i = V * lane + 64u * V * j;
        if (i < a.D) {
          if constexpr (V == 4) {
            *reinterpret_cast<uint2*>(orow + off + a.D + i) = t_copy[j];
            const uint2 xr = t.a[j], dr = t.b[j];
            x[4 * j + 0] = __uint_as_float(xr.x << 16); x[4 * j + 1] = __uint_as_float(xr.x & 0xffff0000u);
            x[4 * j + 2] = __uint_as_float(xr.y << 16); x[4 * j + 3] = __uint_as_float(xr.y & 0xffff0000u);
            d[4 * j + 0] = __uint_as_float(dr.x << 16); d[4 * j + 1] = __uint_as_float(dr.x & 0xffff0000u);
            d[4 * j + 2] = __uint_as_float(dr.y << 16); d[4 * j + 3] = __uint_as_float(dr.y & 0xffff0000u);
          } else {
            orow[off + a.D + i] = dcopy[i];
            x[j] = bf16_bits_to_f32(frow[off + i]);
            d[j] = bf16_bits_to_f32(dy[i]);
          }
#pragma unroll
          for (int e = 0; e < V; ++e) {
            ss += (double)x[V * j + e] * (double)x[V * j + e];
            buf[wave][i + e] = d[V * j + e];
          }
        } else {
#pragma unroll
          for (int e = 0; e < V; ++e) x[V * j + e] = d[V * j + e] = 0.0f;
        }
      }
      ss = wave_sum(ss);
      const float mean = qkv_mean(ss, a.D);
      const float inv = 1.0f / sqrtf(mean + a.eps);
      // the rotation pairs element i with i +- rot / 2, held by another lane of this wave
      __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
      __builtin_amdgcn_wave_barrier();
      float n[NP * V], p[NP * V];
      double sp = 0.0;
#pragma unroll
      for (uint32_t j = 0; j < NP; ++j) {
        const uint32_t i = V * lane + 64u * V * j;
        if (i < a.D) {
#pragma unroll
          for (int e = 0; e < V; ++e) {
            const uint32_t c = i + e;
            float uo = d[V * j + e];
            if (c < a.rot) {
              if (c < half) uo = uo * cs[c] + buf[wave][c + half] * sn[c];
              else uo = uo * cs[c - half] - buf[wave][c - half] * sn[c - half];
              uo = bf16_round_f32(uo);
            }
            d[V * j + e] = uo;
            n[V * j + e] = x[V * j + e] * inv;
            float one = 0.0f;
            if constexpr (V == 4) {
              const float4 o4 = is_q ? one_q[j] : one_k[j];
              one = e == 0 ? o4.x : e == 1 ? o4.y : e == 2 ? o4.z : o4.w;
            } else {
              one = 1.0f + qkv_weight(w, c, a.w_bf16 != 0u);
            }
            p[V * j + e] = uo * one;
            sp += (double)(p[V * j + e] * n[V * j + e]);
          }
        }
      }
      sp = wave_sum(sp);
      const float mu = qkv_mean(sp, a.D);
#pragma unroll
      for (uint32_t j = 0; j < NP; ++j) {
        const uint32_t i = V * lane + 64u * V * j;
        if (i < a.D) {
          float o[V];
#pragma unroll
          for (int e = 0; e < V; ++e) {
            o[e] = inv * (p[V * j + e] - n[V * j + e] * mu);
            if (WGRAD) {
              const float t = d[V * j + e] * n[V * j + e];
              wq[V * j + e] += is_q ? t : 0.0f;
              wk[V * j + e] += is_q ? 0.0f : t;
            }
          }
          if constexpr (V == 4) {
            *reinterpret_cast<uint2*>(orow + off + i) = make_uint2(pack_bf16x2(o[0], o[1]), pack_bf16x2(o[2], o[3]));
          } else {
            orow[off + i] = (uint16_t)f32_to_bf16_bits(o[0]);
          }
        }
      }
      __builtin_amdgcn_s_waitcnt(0xc07f);
      __builtin_amdgcn_wave_barrier();  // buf[wave] is rewritten by the next unit
    }
  }
  if (WGRAD) {
    // the four waves' sums, wave 0 first; buf is free once every wave is past its rows
    for (uint32_t which = 0; which < 2; ++which) {
      __syncthreads();
#pragma unroll
      for (uint32_t j = 0; j < NP; ++j) {
        const uint32_t i = V * lane + 64u * V * j;
        if (i < a.D) {
#pragma unroll
          for (int e = 0; e < V; ++e) buf[wave][i + e] = which == 0 ? wq[V * j + e] : wk[V * j + e];
        }
      }
      __syncthreads();
      for (uint32_t i = tid; i < a.D; i += 256u)
        a.partial[((size_t)blockIdx.x * 2u + which) * a.D + i] = ((buf[0][i] + buf[1][i]) + buf[2][i]) + buf[3][i];
    }
  }
}

// out[c] = sum over the n_parts rows of partial[part][col0 + c].  A workgroup takes 16 columns; its
// 16 lanes per column sum every 16th part each (lane l: parts l, l + 16, ...), then lane 0 adds the
// 16 sums in lane order: a fixed order whatever the launch.
struct ColumnSumArgs {
  const float* partial;  // f32 [n_parts][stride]
  float* out;            // f32 [cols]
  uint32_t n_parts, stride, cols, col0;
};

__global__ __launch_bounds__(256) void column_sum_kernel(ColumnSumArgs a) {
  __shared__ float red[16][17];
  const uint32_t cl = threadIdx.x & 15u, pl = threadIdx.x >> 4;
  const uint32_t c = blockIdx.x * 16u + cl;
  float s = 0.0f;
  if (c < a.cols) {
#pragma unroll 4
    for (uint32_t p = pl; p < a.n_parts; p += 16u) s += a.partial[(size_t)p * a.stride + a.col0 + c];
  }
  red[pl][cl] = s;
  __syncthreads();
  if (pl == 0 && c < a.cols) {
    float t = red[0][cl];
#pragma unroll
    for (uint32_t l = 1; l < 16; ++l) t += red[l][cl];
    a.out[c] = t;
  }
}

}  // namespace w8a8
