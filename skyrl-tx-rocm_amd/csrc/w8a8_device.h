// Device-side helpers and the packed operand layout shared by every kernel of the
// W8A8 LoRA linear path (gfx950 only: wave64, MFMA, 160 KiB LDS).
//
// Packed int8 operand layout ("fragment order").  Both GEMM operands are stored as
// 1 KiB blocks of 32 rows (activation rows, or weight output columns) x 32 k.  Inside
// a block, lane l of a wavefront owns 16 consecutive bytes:
//     row-in-block = l % 32,   k-in-block = 16 * (l / 32) + byte
// which is exactly one v_mfma_i32_32x32x32_i8 A or B operand, so a wave fetches an
// operand with a single 16-byte-per-lane load of a contiguous 1 KiB chunk.  Blocks are
// ordered [row_block][k_block].  Weight columns are additionally permuted inside every
// group of 128: packed column 128g + 32j + c holds original column 128g + 4c + j, so a lane
// of the MFMA output owns four consecutive original columns (two (gate, up) pairs of a fused
// gate/up projection) in the four adjacent 32-column blocks of its wave.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace w8a8 {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef unsigned short v8us __attribute__((ext_vector_type(8)));

constexpr int kBlk = 32;          // rows / columns / k per fragment block
constexpr int kBlockBytes = 1024; // bytes of one fragment block
constexpr int kTileM = 256;
constexpr int kTileN = 256;
constexpr int kTileK = 128;
constexpr int kMaxAdapters = 64;
constexpr int kMaxRank = 64;
constexpr int kMaxKSplit = 8;

__host__ __device__ inline uint32_t round_up(uint32_t v, uint32_t a) { return (v + a - 1) / a * a; }
__host__ __device__ inline uint32_t k_padded(uint32_t k) { return round_up(k, kTileK); }
__host__ __device__ inline uint32_t n_padded(uint32_t n) { return round_up(n, kTileN); }

// original weight column of packed column c
__host__ __device__ inline uint32_t packed_to_orig_col(uint32_t c) {
  return (c & ~127u) + 4u * (c & 31u) + ((c >> 5) & 3u);
}
// packed column of original column n (inverse of the above)
__host__ __device__ inline uint32_t orig_to_packed_col(uint32_t n) {
  return (n & ~127u) + 32u * (n & 3u) + ((n & 127u) >> 2);
}
// byte offset of element (row r, k) of a packed operand with kb k-blocks per row block
__host__ __device__ inline size_t packed_offset(uint32_t r, uint32_t k, uint32_t kb) {
  return ((size_t)(r >> 5) * kb + (k >> 5)) * kBlockBytes + ((r & 31u) + 32u * ((k & 31u) >> 4)) * 16u +
         (k & 15u);
}

__device__ inline float bf16_bits_to_f32(uint32_t bits16) { return __uint_as_float(bits16 << 16); }

// float pair -> packed bf16x2, round to nearest even (one v_cvt_pk_bf16_f32; NaN stays NaN)
__device__ inline uint32_t pack_bf16x2(float lo, float hi) {
  typedef float v2f __attribute__((ext_vector_type(2)));
  typedef __bf16 v2bf __attribute__((ext_vector_type(2)));
  const v2f v = {lo, hi};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, v2bf));
}
// float -> bf16 bits, round to nearest even
__device__ inline uint32_t f32_to_bf16_bits(float f) { return pack_bf16x2(f, 0.0f) & 0xffffu; }
__device__ inline float bf16_round_f32(float f) { return bf16_bits_to_f32(f32_to_bf16_bits(f)); }

// Largest |value| of eight bf16 values against a running maximum of pairs: |bf16| compares like its 15
// magnitude bits as an integer (a NaN ends above every number and the scale then falls back to 1, as the
// reference's comparison amax > 0 does).
__device__ inline uint32_t bf16_absmax_pairs(uint32_t amax_bits, const uint4& raw) {
  typedef unsigned short us2 __attribute__((ext_vector_type(2)));
  us2 mx = __builtin_bit_cast(us2, amax_bits);
  mx = __builtin_elementwise_max(mx, __builtin_bit_cast(us2, raw.x & 0x7fff7fffu));
  mx = __builtin_elementwise_max(mx, __builtin_bit_cast(us2, raw.y & 0x7fff7fffu));
  mx = __builtin_elementwise_max(mx, __builtin_bit_cast(us2, raw.z & 0x7fff7fffu));
  mx = __builtin_elementwise_max(mx, __builtin_bit_cast(us2, raw.w & 0x7fff7fffu));
  return __builtin_bit_cast(uint32_t, mx);
}

// ---- int8 codes of bf16 values: code = rint(v / scale), the quotient correctly rounded, with scale = amax / qmax for
// the largest |v|.  q0 = v * r (r: the hardware reciprocal) is corrected by its remainder v - q0 * scale, which a fused
// multiply-add forms exactly: three operations, no division and no look at how near a tie the quotient lies.  (Ties are
// common here: v and amax are bf16 values, and 127 v / amax is a half integer for every third value or so of a row whose
// amax is a power of two.  The form before, one product and a division for the 512 values of a wave where one of them lay
// near a tie, took that division for every other piece: 28 vector operations a value, now 7.)  That the codes are those
// of the division was checked for every pair of bf16 significands and every reciprocal within two units of the last place;
// powers of two drop out while scale and r are ordinary numbers (tests/test_quotient.py).
__device__ inline float code_quotient(float v, float scale, float r) {
  const float q0 = v * r;
  return __builtin_fmaf(__builtin_fmaf(-q0, scale, v), r, q0);
}
// The codes of four quotients q, -128.5 <= q < 127.5, byte e the e-th: 1.5 * 2^23 has a last place of one, so the sum's low byte
// is the quotient rounded to nearest even in two's complement.
__device__ inline uint32_t code_bytes4(const float (&q)[4]) {
  uint32_t m[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) m[e] = __float_as_uint(q[e] + 12582912.0f);
  const uint32_t lo = __builtin_amdgcn_perm(m[1], m[0], 0x0c0c0400u), hi = __builtin_amdgcn_perm(m[3], m[2], 0x0c0c0400u);
  return __builtin_amdgcn_perm(hi, lo, 0x05040100u);
}
__device__ inline bool code_scale_ordinary(float scale) { return scale > 1e-30f && scale < 1e30f; }

// f(integral_constant 0), f(1), ..: an unrolled loop whose index is a constant expression.
template <class F, int... S>
__device__ inline __attribute__((always_inline)) void each_of(F&& f, std::integer_sequence<int, S...>) {
  (f(std::integral_constant<int, S>{}), ...);
}

// One step of a butterfly over the wave: op(v, the value of lane ^ O) for an op that commutes, without the LDS.  Rows of 16
// and halves of 32 change places by the permlane swaps, which leave both operands in every lane; below that the data
// parallel moves carry the value (lane ^ 4 as reversed quads in a reversed half row).  __shfl_xor goes through the LDS pipe,
// 130 clocks a step against some ten: moe_route_kernel for 16 tokens, eight selections of 12 steps, 7.1 us, 4.4 now; an MLP's
// 16 decode rows (two launches of skinny_quant_kernel) 46.6 us, 45.3 now.
// Every lane of the wave must be active.
template <int O>
__device__ inline void lane_pair(uint32_t v, uint32_t& a, uint32_t& b) {
  static_assert(O == 1 || O == 2 || O == 4 || O == 8 || O == 16 || O == 32, "a lane bit");
  if constexpr (O == 32) {
    const auto s = __builtin_amdgcn_permlane32_swap(v, v, false, false);
    a = s[0]; b = s[1];
  } else if constexpr (O == 16) {
    const auto s = __builtin_amdgcn_permlane16_swap(v, v, false, false);
    a = s[0]; b = s[1];
  } else {
    constexpr int kCtrl = O == 8 ? 0x128 : O == 4 ? 0x141 : O == 2 ? 0x4e : 0xb1;  // row_ror:8, row_half_mirror, quad_perm
    int t = (int)v;
    if constexpr (O == 4) t = __builtin_amdgcn_update_dpp(t, t, 0x1b, 0xf, 0xf, true);
    a = v;
    b = (uint32_t)__builtin_amdgcn_update_dpp(t, t, kCtrl, 0xf, 0xf, true);
  }
}
template <int O, typename T, typename Op>
__device__ inline T lane_step(T v, Op op) {
  static_assert(sizeof(T) == 4 || sizeof(T) == 8, "one or two registers");
  if constexpr (sizeof(T) == 4) {
    uint32_t a, b;
    lane_pair<O>(__builtin_bit_cast(uint32_t, v), a, b);
    return op(__builtin_bit_cast(T, a), __builtin_bit_cast(T, b));
  } else {
    const uint64_t w = __builtin_bit_cast(uint64_t, v);
    uint32_t a0, b0, a1, b1;
    lane_pair<O>((uint32_t)w, a0, b0);
    lane_pair<O>((uint32_t)(w >> 32), a1, b1);
    return op(__builtin_bit_cast(T, (uint64_t)a1 << 32 | a0), __builtin_bit_cast(T, (uint64_t)b1 << 32 | b0));
  }
}
// The steps 32, 16, .., 1: the value of the whole wave in every lane.
template <typename T, typename Op>
__device__ inline T wave_fold(T v, Op op) {
  v = lane_step<32>(v, op);
  v = lane_step<16>(v, op);
  v = lane_step<8>(v, op);
  v = lane_step<4>(v, op);
  v = lane_step<2>(v, op);
  return lane_step<1>(v, op);
}
__device__ inline float wave_max(float v) { return wave_fold(v, [](float a, float b) { return fmaxf(a, b); }); }
__device__ inline int wave_min(int v) { return wave_fold(v, [](int a, int b) { return a < b ? a : b; }); }
template <typename T>
__device__ inline T wave_sum(T v) { return wave_fold(v, [](T a, T b) { return a + b; }); }

// Inclusive scan of values with identity 0 over the wave, in data parallel moves as above: inside the rows of 16, then the last
// lane of a row to the next, then lane 31 to the upper half.
template <typename Op>
__device__ inline uint32_t wave_scan(uint32_t v, Op op) {
  v = op(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xf, 0xf, false));  // row_shr:1, 2, 4, 8
  v = op(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xf, 0xf, false));
  v = op(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xf, 0xf, false));
  v = op(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xf, 0xf, false));
  v = op(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xa, 0xf, false));  // row_bcast:15
  return op(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xc, 0xf, false));  // row_bcast:31
}
__device__ inline uint32_t wave_scan(uint32_t v) { return wave_scan(v, [](uint32_t a, uint32_t b) { return a + b; }); }
// the value of the lane before, 0 in lane 0
__device__ inline uint32_t lane_before(uint32_t v) { return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x138, 0xf, 0xf, false); }

// s_waitcnt vmcnt(N) only (gfx9 encoding: vmcnt[3:0]|[15:14], expcnt[6:4], lgkmcnt[11:8])
template <int N>
__device__ inline void wait_vmcnt() {
  static_assert(N >= 0 && N < 64, "vmcnt is a 6-bit counter");
  __builtin_amdgcn_s_waitcnt(0x0F70 | (N & 15) | ((N >> 4) << 14));
}
__device__ inline void wait_vmcnt0() { wait_vmcnt<0>(); }

// Workgroup barrier for LDS hand-over that does not wait for outstanding global loads: the
// caller decides with wait_vmcnt<N>() how many direct-to-LDS loads may stay in flight.  The
// wave first drains its own LDS operations, so data it read is in registers and data it wrote
// is visible once every wave has passed.
__device__ inline void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

typedef const __attribute__((address_space(1))) void* gptr_t;
typedef __attribute__((address_space(3))) void* lptr_t;

// One wave copies 1 KiB: lane l moves 16 bytes global[src + 16 l] -> LDS[dst + 16 l].
__device__ inline void load_1k_to_lds(const unsigned char* src_lane, unsigned char* lds_dst_uniform) {
  __builtin_amdgcn_global_load_lds((gptr_t)src_lane, (lptr_t)lds_dst_uniform, 16, 0, 0);
}
// A gather of 64 dwords by one wave: lane l moves 4 bytes global[base + voff] (voff a multiple of 4, any
// place) -> LDS[lds_addr_uniform + 4 l].
__device__ inline void lds_gather_dword(const void* base_uniform, uint32_t voff, uint32_t lds_addr_uniform) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dword %0, %1"
               :: "v"(voff), "s"(base_uniform), "s"(lds_addr_uniform) : "memory", "m0");
}
// The same as an assembly statement the compiler keeps no books on (it treats the builtin as an access
// that may touch the LDS and then drains every counter at its next wait): lane l moves 16 bytes
// global[base + voff] -> LDS[lds_addr_uniform + 16 l]; inactive lanes move nothing.  The caller waits
// with s_waitcnt vmcnt and a barrier before the LDS is read.
__device__ inline void lds_load_1k(const unsigned char* base_uniform, uint32_t voff, uint32_t lds_addr_uniform) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
               :: "v"(voff), "s"(base_uniform), "s"(lds_addr_uniform) : "memory", "m0");
}
// two KiB, one behind the other at both ends (an instruction's offset counts for the LDS as well) ...
__device__ inline void lds_load_2k(const unsigned char* base_uniform, uint32_t voff, uint32_t lds_addr_uniform) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1\n\tglobal_load_lds_dwordx4 %0, %1 offset:1024"
               :: "v"(voff), "s"(base_uniform), "s"(lds_addr_uniform) : "memory", "m0");
}
// ... the second from second_uniform + 1024; for data that is read once (non-temporal)
template <bool ONCE>
__device__ inline void lds_load_2k(const unsigned char* base_uniform, const unsigned char* second_uniform, uint32_t voff, uint32_t lds_addr_uniform) {
  if constexpr (ONCE)
    asm volatile("s_mov_b32 m0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1 nt\n\tglobal_load_lds_dwordx4 %0, %2 offset:1024 nt"
                 :: "v"(voff), "s"(base_uniform), "s"(second_uniform), "s"(lds_addr_uniform) : "memory", "m0");
  else
    asm volatile("s_mov_b32 m0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1\n\tglobal_load_lds_dwordx4 %0, %2 offset:1024"
                 :: "v"(voff), "s"(base_uniform), "s"(second_uniform), "s"(lds_addr_uniform) : "memory", "m0");
}
__device__ inline void lds_load_1k_once(const unsigned char* base_uniform, uint32_t voff, uint32_t lds_addr_uniform) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1 nt"
               :: "v"(voff), "s"(base_uniform), "s"(lds_addr_uniform) : "memory", "m0");
}

}  // namespace w8a8
