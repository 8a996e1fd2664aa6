// Entry points that the torch mirror's autograd rule of the group-scaled linear calls.  They are not part of the
// public C header: a binding of another framework keeps the reference's rule for these weights.
#pragma once
#include "../../include/mi355_w8a8.h"

extern "C" {

/*
 * Backward of the group-scaled linear with one adapter (skyrl/tx/kernels/quantized_lora.py:337-394):
 * dx = dy @ deq(W).T + rs @ A.T with rs = (dy @ B.T) * s, dA = x.T @ rs, dB = ((x @ A).T @ dy) * s,
 * ds = sum(dy * ((x @ A) @ B)); float32 products and sums (a dequantized weight value is carried as its exact
 * split into bf16 terms), every cotangent cast once.  k and n multiples of 8.
 */
#define MI355_W8A8_FLAG_GQ_BF16_SCALES 2u /* every w_scales value is a bf16 value: two terms hold code * scale exactly */
typedef struct mi355_w8a8_gq_bwd_problem {
  uint32_t struct_size;      /* sizeof(mi355_w8a8_gq_bwd_problem) */
  uint32_t flags;            /* GQ_BF16_SCALES, SKIP_GEMM (no dx; dx is not written) */
  uint32_t m, k, k_pad, n;
  uint32_t group_size;       /* multiple of 32, divides k_pad */
  uint32_t weight_bits;      /* 4 or 8 */
  uint32_t rank;             /* 0 = no LoRA, <= 64 */
  uint32_t reserved;
  const void* x;             /* bf16 [m, k]; needed for the LoRA cotangents */
  const void* dy;            /* bf16 [m, n] */
  const void* w_packed;      /* from mi355_w8a8_gq_pack_weight_v1 */
  const float* w_scales;     /* f32 [k_pad / group_size, n] */
  const void* lora_a;        /* bf16 [k, rank] or NULL */
  const void* lora_b;        /* bf16 [rank, n] or NULL */
  const float* lora_scaling; /* f32 [1] or NULL */
  void* dx;                  /* bf16 [m, k] */
  void* d_lora_a;            /* bf16 [k, rank] or NULL */
  void* d_lora_b;            /* bf16 [rank, n] or NULL */
  float* d_lora_scaling;     /* f32 [1] or NULL */
  void* workspace;           /* >= mi355_w8a8_gq_bwd_workspace_bytes(...), 256-byte aligned */
  uint64_t workspace_bytes;
} mi355_w8a8_gq_bwd_problem;

uint64_t mi355_w8a8_gq_bwd_workspace_bytes(uint32_t m, uint32_t k, uint32_t k_pad, uint32_t n, uint32_t group_size,
                                           uint32_t rank);
int mi355_w8a8_gq_linear_bwd_v1(const mi355_w8a8_gq_bwd_problem* problem, void* stream);

}  // extern "C"
