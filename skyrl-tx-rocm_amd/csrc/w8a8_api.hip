// C ABI of the MI355X W8A8 LoRA linear forward path: argument validation, workspace
// carving and kernel launches.  Nothing here synchronises, allocates or keeps state.
#include "../../include/mi355_w8a8.h"
#include "w8a8_gq_bwd_api.h"
#include "w8a8_bwd_split.h"

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstring>
#include <mutex>

#include "w8a8_device.h"
#include "w8a8_gemm.h"
#include "w8a8_grouped.h"
#include "w8a8_gemm16.h"
#include "w8a8_calibration.h"
#include "w8a8_prologue.h"
#include "w8a8_skinny.h"
#include "w8a8_backward.h"
#include "w8a8_qkv_post.h"
#include "w8a8_fused_bwd.h"
#include "w8a8_moe.h"
#include "w8a8_gq.h"
#include "w8a8_gq_bwd.h"

using namespace w8a8;

// Workspace of mi355_w8a8_forward_static_ws_v1: one copy per GPU, held until the process ends.  In host
// code this name is a stand-in, not a device address: the per-device address comes from
// hipGetSymbolAddress (static_workspace() below) and only that pointer is handed to kernels.
static __device__ __align__(256) unsigned char scratch[MI355_W8A8_STATIC_WORKSPACE_BYTES];

namespace {

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mutex;
void* g_scratch_ptr[kMaxDevices] = {};

// Device address of `scratch` on the current device (looked up once per device), or null.
void* static_workspace() {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return nullptr;
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (!g_scratch_ptr[dev]) {
    void* ptr = nullptr;
    if (hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)) != hipSuccess) {
      (void)hipGetLastError();
      return nullptr;
    }
    g_scratch_ptr[dev] = ptr;
  }
  return g_scratch_ptr[dev];
}

constexpr uint32_t kMaxK = 16384;
constexpr uint32_t kMaxRows = 1u << 20;
constexpr uint32_t kMaxN = 1u << 20;

inline uint64_t align256(uint64_t v) { return (v + 255u) & ~uint64_t(255); }

struct WsLayout {
  uint64_t xq, sx, zp, at, bp, row_scale, row_inv, src_row, slot_group, blk_range, tile_ctr, skinny, total;
  uint64_t split_z, split_bytes;  // the last part: a call that finds no room for it does without
  uint32_t slots, nkk, K_pad, KB, n_steps, steps_per_wave;
  uint32_t rows_bound;  // the slots that can hold rows (a multiple of 32)
};

// number of 16-wide rank chunks the kernels are instantiated for (rank padded with zeros)
inline uint32_t rank_chunks(uint32_t rank) { return rank == 0 ? 0u : (rank <= 16u ? 1u : (rank <= 32u ? 2u : 4u)); }

// Between the skinny-M limit and this many rows a call without SwiGLU may run the skinny-M kernels
// on chunks of 32 rows: the weight is streamed once per chunk (the later passes from the last-level
// cache), whatever the adapters.  Where it may is what mi355_w8a8_forward_path reports and what callers go by;
// whether it does is chunks_pay's choice.
constexpr uint32_t kSkinnyChunkedMaxRows = 96;
inline bool skinny_chunks_possible(uint32_t m, uint32_t k, uint32_t n) {
  if (m > kSkinnyChunkedMaxRows || k < 4096u || (uint64_t)k_padded(k) * n_padded(n) > (64ull << 20)) return false;
  return k >= 8192u || (m <= 64u && n_padded(n) <= 4096u);
}

// Grouped slots a call of m rows and n_groups adapters can need when every adapter's rows start on a
// 32-slot block boundary (sum of the groups' sizes rounded up to 32).
inline uint32_t padded_rows_bound(uint32_t m, uint32_t n_groups) {
  return round_up(m + 31u * (n_groups < m ? n_groups : m), 32u);
}
// Whether a routed call may lay its groups out that way: the
// empty slots cost no time -- neither the quantizer's workgroups (16 slots each, one resident per CU) nor
// the GEMM's tiles (512 resident tiles of 128 x 128, 256 of 256 x 256) need another round on the chip
// than the packed layout does.
inline bool padded_groups_fit(uint32_t m, uint32_t n, uint32_t n_groups, bool wide_tiles = false) {
  if (n_groups < 2u || m > kPaddedRouteMaxRows) return false;
  const uint32_t rows = padded_rows_bound(m, n_groups), base = round_up(m, 32u);
  auto rounds = [](uint64_t items, uint64_t resident) { return (items + resident - 1u) / resident; };
  if (rounds(rows / 16u, 256u) != rounds(base / 16u, 256u)) return false;
  const uint32_t tile_m = wide_tiles ? (uint32_t)kTileM : (uint32_t)kGemm128TileM;
  const uint64_t per_row = n_padded(n) / (wide_tiles ? (uint32_t)kG16TileN : (uint32_t)kGemmTileN);
  const uint64_t resident = wide_tiles ? 256u : 512u;
  return rounds((uint64_t)(round_up(rows, tile_m) / tile_m) * per_row, resident) ==
         rounds((uint64_t)(round_up(base, tile_m) / tile_m) * per_row, resident);
}

// Tiles of 192 x 256 instead of 256 x 256 where they fill the chip's rounds of 256 tiles better.  A round of them takes 0.79 of
// the time; beside the rounds the tiles themselves count as much, which is a compromise and no fit: a partly filled round is shorter than a
// full one, but not by its share.  Of 57 other calls of 1142 to 4031 rows over eight projections that take it, 56 are faster with it
// (whole call 0.77 to 0.996 of the time); 2086 rows of 4096 -> 24576, where the two sides of the rule are 2 % apart, take 1.016.
// The GEMM, 256 / 192
// rows, us: 2560 -> 6144, rank 64, 1536 rows (144 / 192 tiles) 42.1 / 33.5, 1900 (192 / 240) 46.3 / 35.1, 2800 (264 / 360) 80.9 / 63.1, 3900 (384 /
// 504) 88.2 / 67.1; 2560 -> 10240, rank 64, 2048 (320 / 440) 83.3 / 67.6; 12288 -> 4096, rank 32, 3003 (192 / 256) 134.5 / 120.3; 4096 -> 24576, rank
// 32, 1281 (576 / 672) 154.9 / 135.3, 3003 (1152 / 1536) 278 / 269, 2300 (864 / 1152) 213 / 224, 2800 (1056 / 1440) 263 / 275.
inline uint64_t gemm16_tiles(uint32_t rows_bound, uint32_t n, uint32_t tile_rows) {
  return (uint64_t)((rows_bound + tile_rows - 1u) / tile_rows) * (n_padded(n) / (uint32_t)kG16TileN);
}
inline bool gemm16_short_tiles(uint32_t rows_bound, uint32_t n, uint32_t flags) {
  const uint64_t t6 = gemm16_tiles(rows_bound, n, 192u), t8 = gemm16_tiles(rows_bound, n, 256u);
  return !(flags & MI355_W8A8_FLAG_TILE_256X256) && ((t6 + 255u) / 256u * 256u + t6) * 79u < ((t8 + 255u) / 256u * 256u + t8) * 100u;
}
// the rounds of such a call, in hundredths of one of 256 x 256 tiles
inline uint64_t gemm16_rounds(uint32_t rows_bound, uint32_t n, uint32_t flags) {
  return gemm16_short_tiles(rows_bound, n, flags) ? (gemm16_tiles(rows_bound, n, 192u) + 255u) / 256u * 79u : (gemm16_tiles(rows_bound, n, 256u) + 255u) / 256u * 100u;
}

// 64 x 128 tiles of a call whose slots end at rows_bound, the waves of a workgroup splitting K (w8a8_gemm_ksplit_kernel), and
// whether it takes them: while all are resident at once, one to a CU (up to 256) or two.  Beyond, the 128 x 128 geometry moves
// fewer bytes.  Whole call, the other prologue in front of the 128 x 128 tiles: 4096 -> 2560, rank 64: 333 rows 34 us against 51, 700 (480 tiles)
// 46 against 52; 2560 -> 6144, rank 64: 128 rows 29 / 42, 333 rows (480) 39 / 43; 1024 -> 3072, rank 16 19 / 25;
// 12288 -> 4096, rank 32: 333 rows 55 / 102; SwiGLU 1024 -> 6144, 333 rows 24 / 26.  As three rounds of pairs 2560 -> 6144, 700 rows 59 / 48.
constexpr uint32_t kKSplitMaxTiles = 512u;
inline uint32_t ksplit_tiles_m(uint32_t rows_bound) { return (rows_bound + (uint32_t)kGemm64TileM - 1u) / (uint32_t)kGemm64TileM; }
inline bool ksplit_fits(uint32_t rows_bound, uint32_t n) { return ksplit_tiles_m(rows_bound) * ((n + 127u) / 128u) <= kKSplitMaxTiles; }
inline uint32_t ksplit_tiles(uint32_t rows_bound, uint32_t n) { return ksplit_tiles_m(rows_bound) * ((n + 127u) / 128u); }
// Whether a routed call that the K-split tiles fit without padding puts its groups on block boundaries all the same.  A block of several groups runs its
// epilogue and its LoRA-A once for each, a matter of the rank and of how many groups share 32 rows; the empty slots cost tiles, which
// matters where those then run two to a CU, or no longer on these kernels at all, and the more the longer K is.
// Whole call, packed / on boundaries.  Same number to a CU: 2560 -> 6144, 4 adapters of rank 64, 333 rows 38 us / 37 and up.  From one to two: 8192 -> 8192, 8 adapters
// of rank 16, 64 rows 60 / 52, rank 64, 97 rows 68 / 62, 256 53 / 62; 2560 -> 6144, 8 of rank 16, 160 rows 31 / 27, of rank 32, 256 31 / 33; 4096 -> 2560, 8 of rank 64, 768 rows 42 / 46; 1024 -> 3072, 4 of rank
// 64, 520 rows 28 / 25.  From one to behind each other: 4096 -> 24576, 4 of rank 64, 33 rows 59 / 63; 4096 -> 4096, 24 of rank 16, 300 rows 40 / 53.  From two: 8192 -> 8192, 8 of rank 16, 400 rows
// 79 / 91; 2048 -> 10960 SwiGLU, 8 adapters, 200 rows, rank 64 54 / 45, rank 32 42 / 39, at 160 rows rank 16 32 / 37; 4096 -> 4096, 4 of rank 32, 1024 rows 52 / 55; 256 -> 4096 level.  Many rows of rank
// 64: 4096 -> 2560, 4 adapters, 1600 rows 62 / 58, 2560 -> 1024, 2000 rows 41 / 38.
// Many groups of rank 64, rows dealt at random: 12288 -> 6144, 24 adapters, 54 rows 187 / 143; 4096 -> 5120, 24, 155 rows 74 / 68; 4096 -> 6144, 16, 323 rows 71 / 68;
// 6144 -> 2048, 64, 1124 rows 128 / 105; 8192 -> 1024, 64, 1271 rows 125 / 115 (1000 rows 115 / 111, 700 rows 106 / 108).
inline bool ksplit_padding_pays(uint32_t m, uint32_t k, uint32_t n, uint32_t groups, uint32_t nkk) {
  const uint32_t packed = ksplit_tiles(round_up(m, 32u), n), padded = ksplit_tiles(padded_rows_bound(m, groups), n);
  if (padded <= 256u || (packed > 256u && padded <= kKSplitMaxTiles)) return true;
  if (nkk > 2u && (m >= 1280u || (groups > 32u && m >= 960u))) return true;
  const uint64_t group_work = ((uint64_t)m * k / groups) >> 10;
  if (padded <= kKSplitMaxTiles) return k <= 1536u || group_work <= (nkk > 2u ? 100u : 70u);
  if (k <= 512u) return true;
  if (nkk > 2u && m / groups <= (packed <= 256u ? (k <= 4096u ? 8u : 4u) : (k <= 4096u ? 32u : 16u))) return true;
  if (packed <= 256u) return group_work <= (nkk > 2u ? 24u : 16u);
  return group_work <= (nkk > 2u ? (k <= 2048u ? 140u : 70u) : (nkk == 2u && k <= 2048u ? 70u : 16u));
}
// Chunks or 128 x 128 tiles where a call may run on chunks.  Tiles run one to a CU, two (1.5 times as long) or behind each other, by
// the slots of the call's groups on block boundaries, and bring every adapter's A and B into operand order first; a chunk takes 11 to 30 us
// whatever the adapters.  Chunks / tiles in us.  No adapters: 12288 x 4096 at 64 rows 33 / 50-64, at 96 49 / 63; 8192 x 1024 at 96 34 / 42; 4096 x 2560 at 64
// 17 / 25; 8192 x 8192 at 40 40 / 36-43, at 65 62 / 43.  One to a CU: 12288 x 4096, rank 16 at 64 45 / 48, at 72 60 / 46, rank 64 at 48 50 / 54, at 64 58 / 54; 6144 x 4096, rank 16
// at 64 30 / 31, rank 64 at 56 41 / 37; 4096 x 2560, rank 16 at 48 24 / 24, at 64 27 / 24, sixteen adapters 27 / 28, rank 64 at 48 33 / 31, at 64 39 / 32; 8192 x 1024, rank 64, 16 adapters
// at 56 45 / 48, 48 at 64 49 / 69, at 96 75 / 70, 48 of rank 32 at 67 53 / 57; 8192 x 8192, rank 64 at 33 64 / 42.  In pairs: 12288 x 4096, 16 adapters of rank 16 at 96 69 / 74; 9728 x 2560, 24 of rank 16 at 96
// 62 / 63; 6144 x 4096, 16 of rank 64 at 64 49 / 57; 8192 x 8192, 8 of rank 64 at 33 66 / 63, of rank 8 at 40 53 / 57, of rank 32 at 37 57 / 61; 8192 x 6144, 16 of rank 16 at 33 48 / 56, of rank 64 at 48 70 / 69, at 64 84 / 72; 12288 x
// 5120, 16 of rank 64 at 64 94 / 94.  Behind each other: 8192 x 8192, 16 of rank 16 at 64 61 / 87, at 72 83 / 88, 48 of rank 16 at 33 53 / 252, at 96 94 / 119; 12288 x 5120, 24 of
// rank 16 at 96 104 / 121.
inline bool chunks_pay(uint32_t m, uint32_t k, uint32_t n, uint32_t slots, uint32_t groups, uint32_t nkk) {
  const bool narrow = n_padded(n) <= 4096u;
  if (!nkk) return narrow;
  const uint32_t tiles = ksplit_tiles(slots, n);
  if (tiles <= 256u) {
    if (!narrow) return false;
    if (nkk <= 2u) return m <= (groups > 32u ? 80u : (k >= 6144u || groups > 8u ? 64u : 48u));
    return m <= (k >= 8192u && groups > 8u ? (groups > 32u ? 80u : 64u) : 48u);
  }
  if (narrow) return true;
  if (tiles <= kKSplitMaxTiles) return groups > (nkk > 2u ? 8u : 7u) && m <= 64u && m <= k / 170u;
  return groups > 16u || m <= 64u;
}
// Whether such a call's prologue leaves z in quarters (quant_lora_kernel's SPLIT form) instead of packed.  The prologue is a chain over K
// that four workgroups to a half block shorten: 333 x 4096, rank 64 14 us / 22 packed, 333 x 12288, rank 32 22 / 41, 1000 x 1032 10 / 12.  But every tile then
// reads four floats where it reads three bf16 terms and splits them itself, in pairs behind its main loop.  Whole call, quarters / packed: rank 16
// 256 -> 4096, 1024 rows (512 tiles) 16.6 us / 17.7, 4096 -> 2560, 1400 rows 42 / 45; rank 32 256 -> 4096, 768 rows (384) 4 % slower, 1024 -> 3072, 1024 rows (384) 2 %,
// 2048 -> 2048, 1024 rows 8 % faster, 1024 -> 1024, 1400 rows 4 % slower; rank 64 256 -> 4096, 768 rows 24.0 / 19.6, 512 -> 2048, 2000 rows 31.0 / 24.0, 1024 -> 3072, 1024 rows 29.0 / 25.4,
// 520 rows (216) 4 % slower, 2048 -> 2048, 1400 rows (352) 36.7 / 33.7, 640 rows level, 4096 -> 2560, 1400 rows (440) 50.7 / 47.9, 768 rows 10 % faster, 8192 -> 8192, 400 rows (448) 60.8 / 69.2.
constexpr uint32_t kSplitZMinKRank64 = 2048u;
inline bool split_z_pays(uint32_t m, uint32_t k, uint32_t nkk, uint32_t tiles) {
  if (nkk <= 1u) return true;
  if (nkk > 2u && k < kSplitZMinKRank64) return false;
  return k >= m * (nkk / 2u) * (tiles > 256u ? 2u : 1u);
}
// Bytes of z's four quarters for a call that may leave them, or 0.
constexpr uint32_t kSplitZMaxRows = 2048;
inline uint64_t split_z_bytes(uint32_t m, uint32_t n, uint32_t n_groups, uint32_t rank) {
  if (!rank || m <= (uint32_t)kSkinnyMaxRows || m > kSplitZMaxRows || !ksplit_fits(round_up(m, 32u), n)) return 0u;
  return (uint64_t)padded_rows_bound(m, n_groups < 2u ? 1u : n_groups) * rank_chunks(rank) * 256u;
}

WsLayout make_layout(uint32_t m, uint32_t k, uint32_t n, uint32_t n_groups, uint32_t rank, bool routed,
                     bool pad_groups = false, bool keep_b = false) {
  WsLayout w{};
  w.K_pad = k_padded(k);
  w.KB = w.K_pad / 32u;
  w.rows_bound = pad_groups ? padded_rows_bound(m, n_groups) : round_up(m, 32u);
  w.slots = round_up(w.rows_bound, kTileM);
  (void)routed;
  w.nkk = rank_chunks(rank);
  w.n_steps = (k + 63u) / 64u;
  w.steps_per_wave = (w.n_steps + 15u) / 16u;
  uint64_t off = 0;
  // The LoRA operands a caller may vouch for (MI355_W8A8_FLAG_LORA_PACK_VALID) come first: their sizes and
  // so their places depend on (k, n, n_adapters, rank) only -- not on m, the path or the slot layout -- so
  // calls of different row counts on one workspace find them where an earlier call left them.
  w.at = off; off += rank ? align256((uint64_t)n_groups * w.KB * w.nkk * kBlockBytes) : 0u;  // A in operand order
  w.bp = off; off += rank ? align256((uint64_t)n_groups * (n_padded(n) / 32u) * w.nkk * kBlockBytes) : 0u;
  w.xq = off; off += align256((uint64_t)w.slots * w.K_pad);
  w.sx = off; off += align256((uint64_t)w.slots * 4u);
  w.row_scale = off; off += align256((uint64_t)m * 4u);
  w.row_inv = off; off += align256((uint64_t)m * 4u);
  w.src_row = off; off += align256((uint64_t)w.slots * 4u);
  w.slot_group = off; off += align256((uint64_t)w.slots * 4u);
  w.blk_range = off; off += align256((uint64_t)(w.slots / 32u) * 4u);
  w.tile_ctr = off; off += 1024u;  // two sets of eight counters, 64 bytes apart
  w.zp = off; off += rank ? align256((uint64_t)(w.slots / 32u) * w.nkk * 3u * kBlockBytes) : 0u;
  w.skinny = off; off += align256(skinny_layout(k, keep_b, m, n, rank).total);
  w.split_bytes = split_z_bytes(m, n, n_groups, rank);
  w.split_z = off; off += w.split_bytes;
  w.total = off;
  return w;
}

inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }
inline bool overlaps(const void* a, uint64_t an, const void* b, uint64_t bn) {
  if (!a || !b || an == 0 || bn == 0) return false;
  const uintptr_t a0 = reinterpret_cast<uintptr_t>(a), b0 = reinterpret_cast<uintptr_t>(b);
  return a0 < b0 + bn && b0 < a0 + an;
}

inline int launch_status() { return hipGetLastError() == hipSuccess ? MI355_W8A8_OK : MI355_W8A8_ERR_LAUNCH; }

int launch_quant(const QuantArgs& a, hipStream_t s) {
  const uint32_t need = (a.K + 511u) / 512u;
  const dim3 grid((a.M + 3u) / 4u), block(256);
#define W8A8_Q(NCH)                                                              \
  if (need <= NCH) {                                                             \
    hipLaunchKernelGGL((quant_rows_kernel<NCH>), grid, block, 0, s, a);          \
    return launch_status();                                                      \
  }
  W8A8_Q(1) W8A8_Q(2) W8A8_Q(4) W8A8_Q(8) W8A8_Q(16) W8A8_Q(24) W8A8_Q(32)
#undef W8A8_Q
  return MI355_W8A8_ERR_UNSUPPORTED;
}

// LoRA-A projection.  Up to 32 ranks (nkk: 16-wide rank chunks) the operands travel through LDS in whole
// cache lines (the staged form of the kernel); beyond, two rank blocks per wave leave no room for that.
int launch_lora_a(const LoraAArgs& la, uint32_t nkk, dim3 grid, hipStream_t s) {
  if (nkk > 2u) {
    hipLaunchKernelGGL((lora_a_kernel<2>), grid, dim3(1024), 0, s, la);
    return launch_status();
  }
  if (hipFuncSetAttribute(reinterpret_cast<const void*>(&lora_a_kernel<1, true>),
                          hipFuncAttributeMaxDynamicSharedMemorySize, kLoraAStageBytes) != hipSuccess)
    return MI355_W8A8_ERR_LAUNCH;
  hipLaunchKernelGGL((lora_a_kernel<1, true>), grid, dim3(1024), kLoraAStageBytes, s, la);
  return launch_status();
}

template <int EPI, int NKK, int MODE>
int launch_gemm_one(const GemmArgs& g, hipStream_t s) {
  // persistent grid: two workgroups per CU, a multiple of 8
  const uint32_t ntile = g.tiles_m * g.tiles_n;
  const uint32_t want = ((ntile + 7u) / 8u) * 8u;
  const dim3 grid(want < 512u ? want : 512u), block(256);
  constexpr uint32_t lds_bytes = MODE == kModeDense128 ? kGemmStages * kGemm128StageBytes : kGemmLdsBytes;
  if (hipFuncSetAttribute(reinterpret_cast<const void*>(&w8a8_gemm_kernel<EPI, NKK, MODE>),
                          hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes) != hipSuccess)
    return MI355_W8A8_ERR_LAUNCH;
  hipLaunchKernelGGL((w8a8_gemm_kernel<EPI, NKK, MODE>), grid, block, lds_bytes, s, g);
  return launch_status();
}

template <int EPI, int MODE = kModeDense>
int launch_gemm(const GemmArgs& g, uint32_t nkk, hipStream_t s) {
  switch (nkk) {
    case 0: return launch_gemm_one<EPI, 0, MODE>(g, s);
    case 1: return launch_gemm_one<EPI, 1, MODE>(g, s);
    case 2: return launch_gemm_one<EPI, 2, MODE>(g, s);
    case 4: return launch_gemm_one<EPI, 4, MODE>(g, s);
    default: return MI355_W8A8_ERR_UNSUPPORTED;
  }
}

template <int EPI, int NKK, bool PAIR, bool CHUNKS>
int launch_gemm_ksplit_one(const GemmKSplitArgs& g, hipStream_t s) {
  constexpr int lds_bytes = PAIR ? kGemm64LdsBytes / 2 : kGemm64LdsBytes;
  if (hipFuncSetAttribute(reinterpret_cast<const void*>(&w8a8_gemm_ksplit_kernel<EPI, NKK, PAIR, CHUNKS>),
                          hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes) != hipSuccess)
    return MI355_W8A8_ERR_LAUNCH;
  hipLaunchKernelGGL((w8a8_gemm_ksplit_kernel<EPI, NKK, PAIR, CHUNKS>), dim3(round_up(g.tiles_m * g.tiles_n, 8u)), dim3(256), lds_bytes, s, g);
  return launch_status();
}

template <int EPI, bool CHUNKS = false>
int launch_gemm_ksplit(const GemmKSplitArgs& g, uint32_t nkk, hipStream_t s) {
  const bool pair = g.tiles_m * g.tiles_n > 256u;
  switch (nkk) {
    case 0: return pair ? launch_gemm_ksplit_one<EPI, 0, true, false>(g, s) : launch_gemm_ksplit_one<EPI, 0, false, false>(g, s);
    case 1: return pair ? launch_gemm_ksplit_one<EPI, 1, true, CHUNKS>(g, s) : launch_gemm_ksplit_one<EPI, 1, false, CHUNKS>(g, s);
    case 2: return pair ? launch_gemm_ksplit_one<EPI, 2, true, CHUNKS>(g, s) : launch_gemm_ksplit_one<EPI, 2, false, CHUNKS>(g, s);
    case 4: return pair ? launch_gemm_ksplit_one<EPI, 4, true, CHUNKS>(g, s) : launch_gemm_ksplit_one<EPI, 4, false, CHUNKS>(g, s);
    default: return MI355_W8A8_ERR_UNSUPPORTED;
  }
}

template <int EPI, int NKK, int RB>
int launch_grouped_one(const GemmArgs& g, hipStream_t s) {
  // one workgroup per CU; how many tiles there are stands in the tile table
  const uint32_t want = round_up(g.tiles_m * g.tiles_n, 8u);
  constexpr uint32_t lds_bytes = grouped_lds_bytes(RB);
  if (hipFuncSetAttribute(reinterpret_cast<const void*>(&w8a8_grouped_kernel<EPI, NKK, RB>),
                          hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes) != hipSuccess)
    return MI355_W8A8_ERR_LAUNCH;
  hipLaunchKernelGGL((w8a8_grouped_kernel<EPI, NKK, RB>), dim3(want < 256u ? want : 256u), dim3(kGroupedThreads), lds_bytes, s, g);
  return launch_status();
}

template <int EPI, int RB>
int launch_grouped(const GemmArgs& g, uint32_t nkk, hipStream_t s) {
  switch (nkk) {
    case 0: return launch_grouped_one<EPI, 0, RB>(g, s);
    case 1: return launch_grouped_one<EPI, 1, RB>(g, s);
    case 2: return launch_grouped_one<EPI, 2, RB>(g, s);
    case 4: return launch_grouped_one<EPI, 4, RB>(g, s);
    default: return MI355_W8A8_ERR_UNSUPPORTED;
  }
}

template <int EPI, int NKK, int NW = 4, int MF = 8>
int launch_gemm16_one(const GemmArgs& g, hipStream_t s) {
  // persistent grid: one workgroup per CU (two in the 256 x 128 geometry), a multiple of 8 so that every
  // XCD gets the same share
  using Geo = G16Geo<NW, MF>;
  const uint32_t ntile = g.tiles_m * g.tiles_n;
  const uint32_t want = ((ntile + 7u) / 8u) * 8u;
  const dim3 grid(want < (uint32_t)Geo::kResident ? want : (uint32_t)Geo::kResident), block(Geo::kThreads);
  if (hipFuncSetAttribute(reinterpret_cast<const void*>(&w8a8_gemm16_kernel<EPI, NKK, NW, MF>),
                          hipFuncAttributeMaxDynamicSharedMemorySize, Geo::kLdsBytes) != hipSuccess)
    return MI355_W8A8_ERR_LAUNCH;
  hipLaunchKernelGGL((w8a8_gemm16_kernel<EPI, NKK, NW, MF>), grid, block, Geo::kLdsBytes, s, g);
  return launch_status();
}

template <int EPI, int NW = 4, int MF = 8>
int launch_gemm16(const GemmArgs& g, uint32_t nkk, hipStream_t s) {
  switch (nkk) {
    case 0: return launch_gemm16_one<EPI, 0, NW, MF>(g, s);
    case 1: return launch_gemm16_one<EPI, 1, NW, MF>(g, s);
    case 2: return launch_gemm16_one<EPI, 2, NW, MF>(g, s);
    case 4: return launch_gemm16_one<EPI, 4, NW, MF>(g, s);
    default: return MI355_W8A8_ERR_UNSUPPORTED;
  }
}

int validate_common(uint32_t m, uint32_t k, uint32_t n) {
  if (m == 0 || k == 0 || n == 0) return MI355_W8A8_ERR_SHAPE;
  if (m > kMaxRows || n > kMaxN) return MI355_W8A8_ERR_UNSUPPORTED;
  if (k % 8u) return MI355_W8A8_ERR_UNSUPPORTED;
  if (k_padded(k) > kMaxK) return MI355_W8A8_ERR_UNSUPPORTED;
  if ((uint64_t)m * n >= (1ull << 32) - (1ull << 20)) return MI355_W8A8_ERR_UNSUPPORTED;  // 32-bit offsets
  return MI355_W8A8_OK;
}

template <int NS, int RB, int KP>
int launch_skinny_stream_one(const SkinnyStreamArgs& a, uint32_t lds_bytes, hipStream_t s) {
  if (hipFuncSetAttribute(reinterpret_cast<const void*>(&skinny_stream_kernel<NS, RB, KP>),
                          hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes) != hipSuccess)
    return MI355_W8A8_ERR_LAUNCH;
  // 8 / NS units per 128-column group; groups are dealt to the eight XCD residues of the block index
  const dim3 grid(((a.n_groups + 7u) / 8u) * (64u / NS)), block(kSkinnyStreamThreads);
  hipLaunchKernelGGL((skinny_stream_kernel<NS, RB, KP>), grid, block, lds_bytes, s, a);
  return launch_status();
}

// The stream kernel's instantiation: KP covers a wave's share of K in one round where registers allow it
// (KP * (NS + RB) operands of four registers), so that all of it is in flight at once.
int launch_skinny_stream(SkinnyStreamArgs& a, hipStream_t s) {
  const bool pairs = skinny_pairs(a.N, a.swiglu != 0, a.residual != nullptr);
  const uint32_t rb = a.M > 16u ? 2u : 1u, ns = pairs ? 2u : 1u, ppw = a.pairs_per_wave;
  const SkinnyStreamLds L = skinny_stream_lds(a.M, a.lora_b ? a.r : 0u, a.z_chunks, ns, rb, a.bsel != nullptr);
  a.z_off = L.z_off; a.tail_off = L.tail_off;
  if (ns == 1u && rb == 1u) {
    if (ppw <= 4u) return launch_skinny_stream_one<1, 1, 4>(a, L.bytes, s);
    if (ppw <= 8u) return launch_skinny_stream_one<1, 1, 8>(a, L.bytes, s);
    if (ppw <= 12u) return launch_skinny_stream_one<1, 1, 12>(a, L.bytes, s);
    return launch_skinny_stream_one<1, 1, 24>(a, L.bytes, s);
  }
  if (ns == 1u) {
    if (ppw <= 4u) return launch_skinny_stream_one<1, 2, 4>(a, L.bytes, s);
    if (ppw <= 8u) return launch_skinny_stream_one<1, 2, 8>(a, L.bytes, s);
    return launch_skinny_stream_one<1, 2, 12>(a, L.bytes, s);
  }
  if (rb == 1u) {
    if (ppw <= 4u) return launch_skinny_stream_one<2, 1, 4>(a, L.bytes, s);
    if (ppw <= 8u) return launch_skinny_stream_one<2, 1, 8>(a, L.bytes, s);
    return launch_skinny_stream_one<2, 1, 12>(a, L.bytes, s);
  }
  if (ppw <= 4u) return launch_skinny_stream_one<2, 2, 4>(a, L.bytes, s);
  return launch_skinny_stream_one<2, 2, 8>(a, L.bytes, s);
}

// Skinny-M path: quantize (+ LoRA-A units) -> stream the weight and finish.
int launch_skinny(const mi355_w8a8_problem* p, unsigned char* xq, float* sx, unsigned char* sws, uint32_t K_pad,
                  uint32_t KB, hipStream_t s, bool allow_kept_b = true) {
  const bool rms = p->rms_gamma != nullptr;
  const bool lora = p->n_adapters > 0;
  const bool skip_prologue = (p->flags & MI355_W8A8_FLAG_SKIP_PROLOGUE) != 0;
  // B regrouped per unit: written by this call, or kept from an earlier one
  const bool can_keep_b = allow_kept_b && lora && skinny_b_can_be_kept(p->m, p->n, p->rank, (p->flags & MI355_W8A8_FLAG_SWIGLU) != 0) &&
                          !skinny_pairs(p->n, false, p->residual != nullptr);
  const bool write_b = can_keep_b && !skip_prologue && (p->flags & MI355_W8A8_FLAG_DECODE_B_WRITE);
  const bool use_b = write_b || (can_keep_b && (p->flags & MI355_W8A8_FLAG_DECODE_B_KEPT));
  const SkinnyLayout L = skinny_layout(p->k);
  int st;
  if (!skip_prologue) {
    SkinnyQuantArgs q{};
    q.x = static_cast<const uint16_t*>(p->x);
    q.gamma = p->rms_gamma;
    q.eps = p->rms_eps;
    q.M = p->m; q.K = p->k; q.K_pad = K_pad; q.KB = KB;
    q.xq = xq; q.sx = sx;
    q.codes_rm = p->aux_x_codes; q.scales_rm = p->aux_x_scales;
    q.xn_aux = static_cast<uint16_t*>(p->aux_normalized);
    q.lora_a = static_cast<const uint16_t*>(p->lora_a);
    q.idx = p->adapter_indices;
    q.z_part = reinterpret_cast<float*>(sws + L.z_part);
    q.n_adapters = p->n_adapters; q.r = p->rank; q.z_chunks = L.z_chunks; q.z_chunk_k = L.z_chunk_k;
    q.n_z_units = lora ? p->m * L.z_chunks : 0u;
    q.lora_scaling = lora ? p->lora_scaling : nullptr;
    q.row_scaling = reinterpret_cast<float*>(sws + L.row_scaling);
    q.N = p->n; q.n_groups = n_padded(p->n) / 128u;
    if (write_b) { q.lora_b = static_cast<const uint16_t*>(p->lora_b); q.bsel = reinterpret_cast<uint16_t*>(sws + L.bsel); }
    const dim3 grid(p->m + q.n_z_units + (write_b ? (p->m * q.n_groups + 15u) / 16u : 0u)), block(1024);
    if (rms) hipLaunchKernelGGL((skinny_quant_kernel<true>), grid, block, 0, s, q);
    else hipLaunchKernelGGL((skinny_quant_kernel<false>), grid, block, 0, s, q);
    if ((st = launch_status())) return st;
  }
  if (p->flags & MI355_W8A8_FLAG_SKIP_GEMM) return MI355_W8A8_OK;
  SkinnyStreamArgs a{};
  a.xq = xq;
  a.wp = static_cast<const unsigned char*>(p->w_packed);
  a.z_part = reinterpret_cast<const float*>(sws + L.z_part);
  a.sx = sx; a.sw = p->w_scales;
  a.lora_b = lora ? static_cast<const uint16_t*>(p->lora_b) : nullptr;
  a.bsel = use_b ? reinterpret_cast<const uint16_t*>(sws + L.bsel) : nullptr;
  a.idx = p->adapter_indices;
  a.row_scaling = reinterpret_cast<const float*>(sws + L.row_scaling);
  a.residual = static_cast<const uint16_t*>(p->residual);
  a.out = static_cast<uint16_t*>(p->out);
  a.aux_acc = p->aux_acc;
  a.M = p->m; a.N = p->n; a.K = p->k; a.KB = KB;
  a.pairs_per_wave = L.pairs_per_wave;
  a.n_adapters = p->n_adapters; a.r = lora ? p->rank : 0u; a.z_chunks = L.z_chunks;
  a.n_groups = n_padded(p->n) / 128u;
  a.swiglu = (p->flags & MI355_W8A8_FLAG_SWIGLU) ? 1u : 0u;
  return launch_skinny_stream(a, s);
}

enum Required { kReqNone = 0, kReqLinear = 1, kReqGateUp = 2, kReqResidual = 3 };

// Which kernels a forward call of these dimensions runs (an MI355_W8A8_PATH_* value), or a negative
// status for a contradictory request.  The choice depends on the dimensions and the flags only.
int choose_forward_path(uint32_t m, uint32_t k, uint32_t n, uint32_t flags) {
  const bool swiglu = (flags & MI355_W8A8_FLAG_SWIGLU) != 0;
  bool skinny = m <= (uint32_t)kSkinnyMaxRows && !(flags & MI355_W8A8_FLAG_FORCE_TILED);
  if (flags & MI355_W8A8_FLAG_FORCE_SKINNY) {
    if (m > (uint32_t)kSkinnyMaxRows) return MI355_W8A8_ERR_UNSUPPORTED;
    skinny = true;
  }
  if (skinny) return MI355_W8A8_PATH_SKINNY;
  if (!swiglu && skinny_chunks_possible(m, k, n) &&
      !(flags & (MI355_W8A8_FLAG_FORCE_TILED | MI355_W8A8_FLAG_TILE_256X128 | MI355_W8A8_FLAG_TILE_256X256 |
                 MI355_W8A8_FLAG_TILE_128X128 | MI355_W8A8_FLAG_TILE_256X128_PAIR)))
    return MI355_W8A8_PATH_SKINNY_CHUNKS;
  // 256 x 256 tiles (one 8-wave workgroup per CU, 16 x 16 x 64 MFMAs) once they fill half the CUs;
  // below that the 256 x 128 geometry (two 4-wave workgroups per CU) has twice the tiles to spread.
  // Measured on the Qwen3-4B QKV projection (K = 2560, N = 6144, rank-64 adapters): at 192 tiles
  // (M = 2048) the GEMM takes 55 us against 73 us; at 48-80 tiles the two are level.
  bool wide = (uint64_t)(round_up(m, kTileM) / kTileM) * (n_padded(n) / kG16TileN) >= 128u;
  if (flags & MI355_W8A8_FLAG_TILE_256X128) wide = false;
  if (flags & MI355_W8A8_FLAG_TILE_256X256) wide = true;
  if (k_padded(k) < kG16MinKPad) wide = false;  // its stage schedule needs at least six 64-wide k steps
  // 128 x 128 tiles (32 x 128 per wave) while all of them are resident at once (two workgroups per
  // CU): a wave then carries half the MFMAs and half the epilogue of the 256 x 128 geometry and the
  // call spreads over four times the CUs.  Measured (call, rank-64 adapters): K = 2560, N = 6144 at
  // M = 512: 62 us against 84; K = 4096, N = 2560 at M = 2048: 88 against 105; beyond 512 tiles the
  // larger geometries win (K = 2560, N = 6144 at M = 2048: 97 us against 85 on 256 x 256).
  const bool small = (uint64_t)(round_up(m, (uint32_t)kGemm128TileM) / (uint32_t)kGemm128TileM) * (n_padded(n) / kGemmTileN) <= 512u;
  const uint32_t forced = flags & (MI355_W8A8_FLAG_TILE_256X128 | MI355_W8A8_FLAG_TILE_256X256 | MI355_W8A8_FLAG_TILE_128X128 |
                                   MI355_W8A8_FLAG_TILE_256X128_PAIR);
  if (forced & (forced - 1u)) return MI355_W8A8_ERR_SHAPE;  // two geometries asked for
  if (forced == MI355_W8A8_FLAG_TILE_256X128_PAIR)  // (its stage schedule needs at least six 64-wide k steps, too)
    return k_padded(k) < kG16MinKPad ? MI355_W8A8_PATH_TILED_256X128 : MI355_W8A8_PATH_TILED_256X128_PAIR;
  if (forced == MI355_W8A8_FLAG_TILE_128X128 || (!forced && small)) return MI355_W8A8_PATH_TILED_128X128;
  return wide ? MI355_W8A8_PATH_TILED_256X256 : MI355_W8A8_PATH_TILED_256X128;
}

template <int CB, bool RMS>
int launch_quant_rows_one(const QuantLoraRowsArgs& a, hipStream_t s) {
  const uint32_t lds_bytes = quant_lora_rows_lds_bytes(a.q.K, CB);
  if (hipFuncSetAttribute(reinterpret_cast<const void*>(&quant_lora_rows_kernel<CB, RMS>),
                          hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes) != hipSuccess)
    return MI355_W8A8_ERR_LAUNCH;
  hipLaunchKernelGGL((quant_lora_rows_kernel<CB, RMS>), dim3(a.q.n_half_blocks * (16u / a.rows_per_wg)), dim3(1024), lds_bytes, s, a);
  return launch_status();
}

template <bool RMS>
int launch_quant_rows(const QuantLoraRowsArgs& a, uint32_t nkk, hipStream_t s) {
  switch (nkk) {
    case 0: return launch_quant_rows_one<0, RMS>(a, s);
    case 1: return launch_quant_rows_one<1, RMS>(a, s);
    case 2: return launch_quant_rows_one<2, RMS>(a, s);
    default: return launch_quant_rows_one<4, RMS>(a, s);
  }
}

int launch_quant_split(const QuantLoraSplitArgs& q, bool normalize, hipStream_t s) {
  const dim3 grid(q.n_half_blocks * 4u), block(256);
#define W8A8_QS(CB)                                                                                        \
  if (normalize) hipLaunchKernelGGL((quant_lora_kernel<CB, true, 4, true>), grid, block, 0, s, q);         \
  else hipLaunchKernelGGL((quant_lora_kernel<CB, false, 4, true>), grid, block, 0, s, q)
  switch (q.nkk) {
    case 1: W8A8_QS(1); break;
    case 2: W8A8_QS(2); break;
    default: W8A8_QS(4); break;
  }
#undef W8A8_QS
  return launch_status();
}

// Which of the two prologues a tiled call takes: quant_lora_rows_kernel (the rows held in the LDS: no launch for their statistics,
// and a second group among sixteen rows costs little) or quant_lora_kernel (x read twice, two workgroups per CU,
// A fetched once per sixteen rows whatever K is).  `boundaries`: the groups follow each other without padding, so
// that sixteen rows may belong to several.  Prologue in us, rows held / read twice, back to back:
//   no LoRA: 4096 x 4096 RMSNorm 20.8 / 23.4, 184 x 12288 RMSNorm 36 / 48, 1024 x 12288 34 / 35; 2048 x 12288 63 / 38.
//   boundaries: 48 x 4096, 8 adapters of rank 32, RMSNorm 32 / 52; 4096 x 4096 34 / 40; 8192 x 4096 62 / 68;
//     48 x 12288 72 / 155, 512 x 12288 (128 workgroups) 65 / 73, 1024 x 12288 72 / 59.
//   operands kept: 4096 x 2560, rank 16 21 / 28, 333 x 4096 level; 6000 x 4096, rank 64, groups padded 54 / 51;
//     184 x 12288 RMSNorm 46 / 51, without the norm 40 / 36.
//   operands laid out by this call, groups padded: 1024 x 4096, rank 32 29 / 26, 333 x 4096, rank 64 25 / 23.
// (Packed groups that happen to meet on block boundaries take the second form 1-2 % of a call faster, 4096 x 2560 -> 6144
// 92 / 94; the layout is not known here.)
bool prologue_keeps_rows(uint32_t rows_bound, uint32_t k, bool rms, bool lora, bool pack, bool boundaries) {
  const uint32_t per_wg = quant_lora_rows_per_wg(k), wgs = (rows_bound + per_wg - 1u) / per_wg;
  if (per_wg < 16u) {  // K > 4608: A fetched for fewer rows
    if (!lora) return wgs <= 256u;
    return wgs <= 128u && (boundaries || (rms && !pack));
  }
  if (!lora || boundaries) return true;
  return !pack && (wgs <= 256u || k <= 2304u);  // (two workgroups of up to 2304 k share a CU)
}

// Whether a call's LoRA-A projection passes through quant_lora_store_z whatever its routing: the tiled paths, but not where the K-split
// tiles, which may take it in quarters, could fit (they fit fewer rows first: the unpadded count decides).
bool forward_keeps_z(uint32_t m, uint32_t k, uint32_t n, uint32_t n_adapters, uint32_t rank, uint32_t flags) {
  if (!n_adapters || !rank || rank > (uint32_t)kMaxRank || validate_common(m, k, n)) return false;
  const int path = choose_forward_path(m, k, n, flags);
  if (path < 0 || path == MI355_W8A8_PATH_SKINNY || path == MI355_W8A8_PATH_SKINNY_CHUNKS) return false;
  return path != MI355_W8A8_PATH_TILED_128X128 || !ksplit_fits(round_up(m, 32u), n);
}

int run_forward(const mi355_w8a8_problem* p, hipStream_t s, Required req) {
  if (!p) return MI355_W8A8_ERR_NULL;
  float* z_rows = nullptr;
  uint32_t rows_per_index = 1;
  if (p->struct_size == sizeof(mi355_w8a8_problem_z)) {
    const mi355_w8a8_problem_z* const whole = reinterpret_cast<const mi355_w8a8_problem_z*>(p);
    z_rows = whole->z;
    rows_per_index = whole->rows_per_index > 1u ? whole->rows_per_index : 1u;
  } else if (p->struct_size != sizeof(mi355_w8a8_problem)) return MI355_W8A8_ERR_STRUCT;
  int st = validate_common(p->m, p->k, p->n);
  if (st) return st;
  if (z_rows && !forward_keeps_z(p->m, p->k, p->n, p->n_adapters, p->rank, p->flags)) return MI355_W8A8_ERR_UNSUPPORTED;
  if (!p->x || !p->w_packed || !p->w_scales || !p->out) return MI355_W8A8_ERR_NULL;
  const bool swiglu = (p->flags & MI355_W8A8_FLAG_SWIGLU) != 0;
  const bool rms = p->rms_gamma != nullptr;
  const bool lora = p->n_adapters > 0;
  if (req == kReqLinear && (swiglu || rms || p->residual)) return MI355_W8A8_ERR_SHAPE;
  if (req == kReqGateUp && (!swiglu || !rms)) return MI355_W8A8_ERR_SHAPE;
  if (req == kReqResidual && (!p->residual || swiglu)) return MI355_W8A8_ERR_SHAPE;
  if (swiglu && (p->n & 1u)) return MI355_W8A8_ERR_SHAPE;
  if (swiglu && p->residual) return MI355_W8A8_ERR_UNSUPPORTED;
  if ((p->flags & MI355_W8A8_FLAG_FORCE_TILED) && (p->flags & MI355_W8A8_FLAG_FORCE_SKINNY))
    return MI355_W8A8_ERR_SHAPE;
  if (lora) {
    if (!p->lora_a || !p->lora_b || !p->lora_scaling) return MI355_W8A8_ERR_NULL;
    if (p->rank == 0 || p->rank > (uint32_t)kMaxRank) return MI355_W8A8_ERR_UNSUPPORTED;
    if (p->n_adapters > (uint32_t)kMaxAdapters) return MI355_W8A8_ERR_UNSUPPORTED;
  } else if (p->adapter_indices) {
    return MI355_W8A8_ERR_SHAPE;
  }
  if (rows_per_index > 1u && (!p->adapter_indices || p->m % rows_per_index)) return MI355_W8A8_ERR_SHAPE;
  if (p->aux_normalized && !rms) return MI355_W8A8_ERR_SHAPE;
  const uint32_t n_out = swiglu ? p->n / 2u : p->n;
  const uint64_t out_bytes = (uint64_t)p->m * n_out * 2u;
  const uint64_t x_bytes = (uint64_t)p->m * p->k * 2u;
  if (!aligned16(p->x) || !aligned16(p->w_packed) || !aligned16(p->out) || !aligned16(p->w_scales) ||
      !aligned16(p->lora_a) || !aligned16(p->lora_b) || !aligned16(p->residual) ||
      !aligned16(p->rms_gamma) || !aligned16(p->adapter_indices) || !aligned16(z_rows))
    return MI355_W8A8_ERR_ALIGN;
  const uint64_t z_bytes = (uint64_t)p->m * p->rank * 4u;
  if (overlaps(z_rows, z_bytes, p->out, out_bytes) || overlaps(z_rows, z_bytes, p->x, x_bytes) ||
      overlaps(z_rows, z_bytes, p->workspace, p->workspace_bytes) || overlaps(p->out, out_bytes, p->x, x_bytes) || overlaps(p->out, out_bytes, p->residual, out_bytes) ||
      overlaps(p->out, out_bytes, p->w_packed, mi355_w8a8_packed_weight_bytes(p->k, p->n)) ||
      overlaps(p->out, out_bytes, p->lora_b, (uint64_t)p->n_adapters * p->rank * p->n * 2u) ||
      overlaps(p->out, out_bytes, p->lora_a, (uint64_t)p->n_adapters * p->rank * p->k * 2u) ||
      overlaps(p->out, out_bytes, p->workspace, p->workspace_bytes))
    return MI355_W8A8_ERR_ALIAS;

  const bool routed = lora && p->adapter_indices && p->n_adapters > 1;
  // The workspace is always sized for the routed layout so one allocation serves every call.
  const uint64_t need = mi355_w8a8_workspace_bytes(p->m, p->k, p->n, p->n_adapters, p->rank, p->flags);
  if (!p->workspace) return MI355_W8A8_ERR_WORKSPACE;
  if (p->workspace_bytes < need - split_z_bytes(p->m, p->n, p->n_adapters, lora ? p->rank : 0u)) return MI355_W8A8_ERR_WORKSPACE;
  if (reinterpret_cast<uintptr_t>(p->workspace) & 255u) return MI355_W8A8_ERR_ALIGN;
  const int reported = choose_forward_path(p->m, p->k, p->n, p->flags);
  if (reported < 0) return reported;
  if (rows_per_index > 1u && (reported == MI355_W8A8_PATH_SKINNY || reported == MI355_W8A8_PATH_SKINNY_CHUNKS)) return MI355_W8A8_ERR_UNSUPPORTED;
  int path = reported;
  if (path == MI355_W8A8_PATH_SKINNY_CHUNKS) {
    const uint32_t groups = routed ? p->n_adapters : 1u, slots = groups > 1u ? padded_rows_bound(p->m, groups) : round_up(p->m, 32u);
    if (!chunks_pay(p->m, p->k, p->n, slots, groups, lora ? rank_chunks(p->rank) : 0u))
      path = choose_forward_path(p->m, p->k, p->n, p->flags | MI355_W8A8_FLAG_FORCE_TILED);
  }
  // groups on block boundaries: only where the empty slots cost no round on the chip, or less than they save
  const bool may_ksplit = path == MI355_W8A8_PATH_TILED_128X128 && !(p->flags & MI355_W8A8_FLAG_TILE_128X128);
  const bool pad_groups =
      routed && ((path == MI355_W8A8_PATH_TILED_128X128 && padded_groups_fit(p->m, p->n, p->n_adapters) &&
                  (!may_ksplit || !ksplit_fits(round_up(p->m, 32u), p->n) ||
                   ksplit_padding_pays(p->m, p->k, p->n, p->n_adapters, rank_chunks(p->rank))) &&
                  // (in the place of chunks on the K-split tiles only, which they fit unpadded: sums_again)
                  (reported != MI355_W8A8_PATH_SKINNY_CHUNKS || ksplit_fits(padded_rows_bound(p->m, p->n_adapters), p->n))) ||
                 (path == MI355_W8A8_PATH_TILED_256X256 && padded_groups_fit(p->m, p->n, p->n_adapters, true) &&
                  gemm16_rounds(padded_rows_bound(p->m, p->n_adapters), p->n, p->flags) <= gemm16_rounds(round_up(p->m, 32u), p->n, p->flags)));
  const WsLayout w = make_layout(p->m, p->k, p->n, p->n_adapters, lora ? p->rank : 0u, routed, pad_groups);
  unsigned char* ws = static_cast<unsigned char*>(p->workspace);
  int32_t* src_row = reinterpret_cast<int32_t*>(ws + w.src_row);
  int32_t* slot_group = reinterpret_cast<int32_t*>(ws + w.slot_group);
  int32_t* blk_range = reinterpret_cast<int32_t*>(ws + w.blk_range);

  (void)hipGetLastError();  // drop a stale error so it is not blamed on these launches

  const bool skinny = path == MI355_W8A8_PATH_SKINNY;
  if (skinny) {
    return launch_skinny(p, ws + w.xq, reinterpret_cast<float*>(ws + w.sx), ws + w.skinny, w.K_pad, w.KB, s);
  }
  if (reported == MI355_W8A8_PATH_SKINNY_CHUNKS) {
    // The chunks overwrite each other's prologue results, so there is no GEMM-only or prologue-only
    // rerun of such a call (nor of one that takes tiles in their place); the choice of path must not depend on those flags either
    // (a GEMM-only tiled call would read tables no tiled prologue has written).
    if (p->flags & (MI355_W8A8_FLAG_SKIP_PROLOGUE | MI355_W8A8_FLAG_SKIP_GEMM)) return MI355_W8A8_ERR_UNSUPPORTED;
  }
  if (path == MI355_W8A8_PATH_SKINNY_CHUNKS) {
    for (uint32_t row0 = 0; row0 < p->m; row0 += (uint32_t)kSkinnyMaxRows) {
      mi355_w8a8_problem sub = *p;
      sub.m = p->m - row0 < (uint32_t)kSkinnyMaxRows ? p->m - row0 : (uint32_t)kSkinnyMaxRows;
      sub.x = static_cast<const unsigned char*>(p->x) + (size_t)row0 * p->k * 2u;
      sub.out = static_cast<unsigned char*>(p->out) + (size_t)row0 * p->n * 2u;
      if (p->residual) sub.residual = static_cast<const unsigned char*>(p->residual) + (size_t)row0 * p->n * 2u;
      if (p->adapter_indices) sub.adapter_indices = p->adapter_indices + row0;
      if (p->aux_x_codes) sub.aux_x_codes = p->aux_x_codes + (size_t)row0 * p->k;
      if (p->aux_x_scales) sub.aux_x_scales = p->aux_x_scales + row0;
      if (p->aux_acc) sub.aux_acc = p->aux_acc + (size_t)row0 * p->n;
      if (p->aux_normalized)
        sub.aux_normalized = static_cast<unsigned char*>(p->aux_normalized) + (size_t)row0 * p->k * 2u;
      // the chunks share the workspace: they run one after the other on the stream
      if ((st = launch_skinny(&sub, ws + w.xq, reinterpret_cast<float*>(ws + w.sx), ws + w.skinny, w.K_pad, w.KB, s, false)))
        return st;
    }
    return MI355_W8A8_OK;
  }

  const bool skip_prologue = (p->flags & MI355_W8A8_FLAG_SKIP_PROLOGUE) != 0;
  const bool skip_gemm = (p->flags & MI355_W8A8_FLAG_SKIP_GEMM) != 0;
  // Rows held in the LDS, or read twice behind a launch that takes their statistics (quant_lora_rows_kernel,
  // quant_lora_kernel).
  // (tiles in the place of chunks, which keep no packed operands and ignore what a caller vouches for, always pack)
  const bool pack = lora && (!(p->flags & MI355_W8A8_FLAG_LORA_PACK_VALID) || reported == MI355_W8A8_PATH_SKINNY_CHUNKS);
  // (neither the next two may depend on the measurement flags: a GEMM-only call reads what its prologue left)
  const bool ksplit = may_ksplit && ksplit_fits(w.rows_bound, p->n);
  const bool split_z = ksplit && w.split_bytes && split_z_pays(p->m, p->k, w.nkk, ksplit_tiles(w.rows_bound, p->n)) && p->workspace_bytes >= w.split_z + w.split_bytes;
  const bool rows_in_lds = !split_z && prologue_keeps_rows(w.rows_bound, p->k, rms, lora, pack, routed && !pad_groups);
  const bool route_inline = rows_in_lds && routed && !pack && p->m <= kInlineRouteMaxRows && rows_per_index == 1u;
  // launch 1: adapter routing, the rows' statistics and (unless the workspace holds them) the LoRA operands
  const uint32_t route_blocks = routed && !route_inline ? 1u : 0u, stat_blocks = rows_in_lds ? 0u : (p->m + 15u) / 16u;
  if (!skip_prologue && (route_blocks || stat_blocks || pack)) {
    LoraPrepArgs pa{};
    pa.idx = routed ? p->adapter_indices : nullptr;
    pa.src_row = src_row; pa.slot_group = slot_group; pa.blk_range = blk_range;
    pa.lora_a = static_cast<const uint16_t*>(p->lora_a);
    pa.lora_b = static_cast<const uint16_t*>(p->lora_b);
    pa.at = reinterpret_cast<uint16_t*>(ws + w.at);
    pa.bp = ws + w.bp;
    pa.M = p->m; pa.K = p->k; pa.N = p->n; pa.n_groups = p->n_adapters; pa.r = p->rank; pa.nkk = w.nkk;
    pa.ncb = n_padded(p->n) / 32u; pa.slots = w.slots;
    pa.route_blocks = route_blocks;
    pa.rows_per_index = rows_per_index;
    pa.route_pad = pad_groups ? 32u : 1u;
    pa.a_operand_kb = w.KB;  // the quantizer reads A in MFMA operand order
    pa.stat_blocks = stat_blocks;
    pa.stat_rows = p->m;
    pa.x = static_cast<const uint16_t*>(p->x);
    pa.gamma = p->rms_gamma; pa.eps = p->rms_eps;
    pa.row_scale = reinterpret_cast<float*>(ws + w.row_scale);
    pa.row_inv = reinterpret_cast<float*>(ws + w.row_inv);
    pa.scales_rm = p->aux_x_scales;
    pa.xn_aux = static_cast<uint16_t*>(p->aux_normalized);
    const uint64_t a_items = (uint64_t)p->n_adapters * w.KB * w.nkk * (p->rank % 4u ? 64u : 16u);
    const uint64_t b_items = (uint64_t)p->n_adapters * pa.ncb * w.nkk * (p->n % 4u ? 64u : 16u);
    pa.a_blocks = pack ? (uint32_t)((a_items + 1023u) / 1024u) : 0u;
    const uint32_t b_blocks = pack ? (uint32_t)((b_items + 1023u) / 1024u) : 0u;
    const dim3 grid(pa.route_blocks + pa.stat_blocks + pa.a_blocks + b_blocks), block(1024);
    if (rows_in_lds) hipLaunchKernelGGL((lora_prep_kernel<0>), grid, block, 0, s, pa);
    else if (rms) hipLaunchKernelGGL((lora_prep_kernel<2>), grid, block, 0, s, pa);
    else hipLaunchKernelGGL((lora_prep_kernel<1>), grid, block, 0, s, pa);
    if ((st = launch_status())) return st;
  }

  // launch 2: codes and LoRA-A projection
  QuantLoraArgs q{};
  // (normalized rows that the statistics launch has written for the caller are read as they are)
  const bool normalize = rms && (rows_in_lds || !p->aux_normalized);
  q.x = static_cast<const uint16_t*>(rms && !normalize ? p->aux_normalized : p->x);
  q.gamma = p->rms_gamma;
  q.row_scale = reinterpret_cast<const float*>(ws + w.row_scale);
  q.row_inv = reinterpret_cast<const float*>(ws + w.row_inv);
  q.M = p->m; q.K = p->k; q.K_pad = w.K_pad; q.KB = w.KB;
  q.n_half_blocks = w.rows_bound / 16u;
  q.src_row = routed ? src_row : nullptr;
  q.slot_group = routed ? slot_group : nullptr;
  q.blk_range = routed ? blk_range : nullptr;
  q.xq_packed = ws + w.xq;
  q.sx_slots = reinterpret_cast<float*>(ws + w.sx);
  q.at = lora ? reinterpret_cast<const uint16_t*>(ws + w.at) : nullptr;
  q.zp = ws + w.zp;
  q.r = p->rank; q.nkk = w.nkk;
  q.nterms = (p->flags & MI355_W8A8_FLAG_LORA_SPLIT2) ? 2u : 3u;
  q.tile_ctr = reinterpret_cast<uint32_t*>(ws + w.tile_ctr);
  q.group_pad = pad_groups ? 32u : 1u;
  q.z_rows = z_rows;
  if (!skip_prologue) {
    const dim3 grid(q.n_half_blocks), block(1024);
    if (split_z) {
      QuantLoraSplitArgs qs{q, reinterpret_cast<float*>(ws + w.split_z), w.rows_bound};
      if ((st = launch_quant_split(qs, normalize, s))) return st;
    } else if (rows_in_lds) {
      QuantLoraRowsArgs qr{};
      qr.q = q;
      qr.eps = p->rms_eps; qr.scales_rm = p->aux_x_scales; qr.xn_aux = static_cast<uint16_t*>(p->aux_normalized);
      if (route_inline) qr.route_idx = p->adapter_indices;
      qr.src_row = src_row; qr.slot_group = slot_group; qr.blk_range = blk_range;
      qr.n_groups = p->n_adapters; qr.slots = w.slots; qr.rows_per_wg = quant_lora_rows_per_wg(p->k); qr.row_stride = quant_lora_row_stride(p->k);
      if ((st = rms ? launch_quant_rows<true>(qr, lora ? w.nkk : 0u, s) : launch_quant_rows<false>(qr, lora ? w.nkk : 0u, s))) return st;
    } else {
#define W8A8_QL(CB)                                                                              \
  if (normalize) hipLaunchKernelGGL((quant_lora_kernel<CB, true>), grid, block, 0, s, q);        \
  else hipLaunchKernelGGL((quant_lora_kernel<CB, false>), grid, block, 0, s, q)
      switch (lora ? w.nkk : 0u) {
        case 0: W8A8_QL(0); break;
        case 1: W8A8_QL(1); break;
        case 2: W8A8_QL(2); break;
        default: W8A8_QL(4); break;
      }
#undef W8A8_QL
      if ((st = launch_status())) return st;
    }
    if (p->aux_x_codes) {
      hipLaunchKernelGGL(codes_row_major_kernel, dim3(w.rows_bound), dim3(256), 0, s, q.xq_packed, nullptr, q.src_row,
                         p->aux_x_codes, nullptr, p->m, p->k, w.KB);
      if ((st = launch_status())) return st;
    }
  } else if (!skip_gemm && path != MI355_W8A8_PATH_TILED_256X256) {
    // measurement calls: the tile counters of the 256 x 128 geometry's dynamic schedule still have to
    // start at zero (the 256 x 256 kernel has a static schedule and no counters)
    hipLaunchKernelGGL(zero_words_kernel, dim3(1), dim3(256), 0, s, q.tile_ctr, 256u);
    if ((st = launch_status())) return st;
  }

  if (skip_gemm) return MI355_W8A8_OK;
  GemmArgs g{};
  g.xq = ws + w.xq;
  g.wp = static_cast<const unsigned char*>(p->w_packed);
  g.sx = reinterpret_cast<const float*>(ws + w.sx);
  g.sw = p->w_scales;
  g.zp = lora ? ws + w.zp : nullptr;
  g.bp = lora ? ws + w.bp : nullptr;
  g.lora_scaling = p->lora_scaling;
  g.src_row = routed ? src_row : nullptr;
  g.slot_group = routed ? slot_group : nullptr;
  g.blk_range = routed ? blk_range : nullptr;
  g.residual = static_cast<const uint16_t*>(p->residual);
  g.out = p->out;
  g.M = p->m; g.N = p->n; g.K_pad = w.K_pad; g.KB = w.KB; g.slots = w.slots;
  g.total_rows = w.rows_bound;
  g.groups_per_weight = 1;
  g.tiles_m = w.slots / kTileM;
  g.tiles_n = n_padded(p->n) / kGemmTileN;
  g.rank = lora ? p->rank : 0u;
  g.tile_ctr = reinterpret_cast<uint32_t*>(ws + w.tile_ctr);
  const bool wide = path == MI355_W8A8_PATH_TILED_256X256;
  const bool pair = path == MI355_W8A8_PATH_TILED_256X128_PAIR;
  const bool small = path == MI355_W8A8_PATH_TILED_128X128;
  if (wide) g.tiles_n = n_padded(p->n) / kG16TileN;
  if (small) g.tiles_m = round_up(w.rows_bound, (uint32_t)kGemm128TileM) / (uint32_t)kGemm128TileM;
  if (p->aux_acc) {
    GemmArgs ga = g;
    ga.out = p->aux_acc;
    ga.residual = nullptr;
    if ((st = wide ? launch_gemm16_one<kEpiAcc, 0>(ga, s)
                   : (pair ? launch_gemm16_one<kEpiAcc, 0, 2>(ga, s)
                           : (small ? launch_gemm_one<kEpiAcc, 0, kModeDense128>(ga, s) : launch_gemm_one<kEpiAcc, 0, kModeDense>(ga, s)))))
      return st;
    g.tile_ctr += 128;  // the second counter set
  }
  if (wide && gemm16_short_tiles(w.rows_bound, p->n, p->flags)) {
    g.tiles_m = (w.rows_bound + 191u) / 192u;
    return swiglu ? launch_gemm16<kEpiSwiglu, 4, 6>(g, w.nkk, s) : launch_gemm16<kEpiPlain, 4, 6>(g, w.nkk, s);
  }
  if (wide) return swiglu ? launch_gemm16<kEpiSwiglu>(g, w.nkk, s) : launch_gemm16<kEpiPlain>(g, w.nkk, s);
  if (pair) return swiglu ? launch_gemm16<kEpiSwiglu, 2>(g, w.nkk, s) : launch_gemm16<kEpiPlain, 2>(g, w.nkk, s);
  if (ksplit) {
    GemmKSplitArgs gk{g, split_z ? reinterpret_cast<const float*>(ws + w.split_z) : nullptr, w.rows_bound, q.nterms};
    gk.tiles_m = ksplit_tiles_m(w.rows_bound);
    gk.tiles_n = (p->n + 127u) / 128u;
    if (reported == MI355_W8A8_PATH_SKINNY_CHUNKS) return launch_gemm_ksplit<kEpiPlain, true>(gk, w.nkk, s);  // (never SwiGLU)
    return swiglu ? launch_gemm_ksplit<kEpiSwiglu>(gk, w.nkk, s) : launch_gemm_ksplit<kEpiPlain>(gk, w.nkk, s);
  }
  if (small)
    return swiglu ? launch_gemm<kEpiSwiglu, kModeDense128>(g, w.nkk, s) : launch_gemm<kEpiPlain, kModeDense128>(g, w.nkk, s);
  return swiglu ? launch_gemm<kEpiSwiglu>(g, w.nkk, s) : launch_gemm<kEpiPlain>(g, w.nkk, s);
}

struct GroupedLayout {
  uint64_t xq, sx, zp, at, bp, row_scale, src_row, blk_range, tile_tab, total;
  uint32_t slots, nkk, K_pad, KB, tile_blocks, max_tiles;
};

// 32-row blocks that a GEMM tile holds at most, 4 or 8; the flags force either (8 only where K has the steps it
// needs).  8 once the groups average at least 96 rows, so that nearly every group is one tile, while those tiles
// still fill three quarters of the CUs and the epilogue's operands fit the ring (rank <= 16; beyond it the tall
// tile spills 60 to 212 bytes a lane).  Grouped call, 4 / 8, sizes rows x K x N: 48 groups of 200 x 1024 x 1024,
// rank 16: 63 / 59 us; 32 of 256 x 1024 x 1024 (128 tall tiles): 47 / 56; 128 of 128 x 2048 x 1536, rank 64: 240 / 273;
// 128 of 64 x 2048 x 1536, rank 16: 112 / 116.
uint32_t grouped_tile_blocks(uint32_t m, uint32_t k, uint32_t n, uint32_t n_groups, uint32_t rank, uint32_t flags) {
  if (k_padded(k) < kGroupedTallMinK) return 4u;
  if (flags & MI355_W8A8_FLAG_GROUPED_TILE64) return 4u;
  if (flags & MI355_W8A8_FLAG_GROUPED_TILE128) return 8u;
  const uint64_t tall_tiles = (uint64_t)(n_groups > m / 256u ? n_groups : m / 256u) * (n_padded(n) / kGroupedTileN);
  return (uint64_t)m >= 96ull * n_groups && rank <= 16u && tall_tiles >= 192u ? 8u : 4u;
}

GroupedLayout make_grouped_layout(uint32_t m, uint32_t k, uint32_t n, uint32_t n_groups, uint32_t rank,
                                  uint32_t flags) {
  GroupedLayout w{};
  w.K_pad = k_padded(k);
  w.KB = w.K_pad / 32u;
  w.tile_blocks = grouped_tile_blocks(m, k, n, n_groups, rank, flags);
  // every group is padded to a multiple of 32 slots: at most 31 padding slots per group
  w.slots = (uint32_t)(((uint64_t)m + 31u * (uint64_t)n_groups + 31u) / 32u * 32u);
  w.max_tiles = w.slots / 32u / w.tile_blocks + n_groups;
  w.nkk = rank_chunks(rank);
  uint64_t off = 0;
  // (the LoRA operands a caller may vouch for come first, as in make_layout: their places depend on
  // (k, n, n_groups, rank) only, not on the row count)
  w.at = off; off += rank ? align256((uint64_t)n_groups * w.KB * w.nkk * kBlockBytes) : 0u;
  w.bp = off; off += rank ? align256((uint64_t)n_groups * (n_padded(n) / 32u) * w.nkk * kBlockBytes) : 0u;
  w.xq = off; off += align256((uint64_t)w.slots * w.K_pad);
  w.sx = off; off += align256((uint64_t)w.slots * 4u);
  w.row_scale = off; off += align256((uint64_t)m * 4u);
  w.src_row = off; off += align256((uint64_t)w.slots * 4u);
  w.blk_range = off; off += align256((uint64_t)(w.slots / 32u) * 4u);
  w.tile_tab = off; off += align256(((uint64_t)w.max_tiles + 1u) * 8u);
  w.zp = off; off += rank ? align256((uint64_t)(w.slots / 32u) * w.nkk * 3u * kBlockBytes) : 0u;
  w.total = off;
  return w;
}

// Four waves per half block once more rows than 4096 come (a wave then has more of K to itself and the sum over
// the waves costs less), else sixteen (the pass is a chain of latencies); without LoRA there is no such sum and the line lies
// at twice the rows.  Prologue in us, 16 / 4 waves, rows x K:
//   128 groups, rank 16: 128 x 2048 17.6 / 18.5, 2048 19.1 / 19.2, 4096 21.8 / 22.2, 4608 29.8 / 26.1, 8192 32.6 / 30.1, 16384
//     54.8 / 46.9; 4096 x 768 14.4 / 14.6, 6144 19.3 / 17.4.  32 groups of 1024: 4096 14.3 / 14.3, 4608 18.2 / 16.3.
//   64 groups, rank 64: 512 x 2048 22.2 / 22.9, 4096 31.7 / 31.8, 4608 39.4 / 36.6, 32768 110 / 87.
//   128 groups, no LoRA: 128 x 2048 11.5 / 12.8, 4608 19.0 / 19.6, 8192 20.3 / 20.8, 12288 27.1 / 26.1, 16384 35.2 / 33.5.
int launch_grouped_quant(const QuantLoraArgs& q, uint32_t nkk, hipStream_t s) {
  const bool few_waves = q.M > (nkk ? 4096u : 8192u);
  const dim3 grid(q.n_half_blocks);
#define W8A8_GQL(CB)                                                                                          \
  if (few_waves) hipLaunchKernelGGL((quant_lora_kernel<CB, false, 4u>), grid, dim3(256), 0, s, q);            \
  else hipLaunchKernelGGL((quant_lora_kernel<CB, false, 16u>), grid, dim3(1024), 0, s, q)
  switch (nkk) {
    case 0: W8A8_GQL(0); break;
    case 1: W8A8_GQL(1); break;
    case 2: W8A8_GQL(2); break;
    default: W8A8_GQL(4); break;
  }
#undef W8A8_GQL
  return launch_status();
}

int run_grouped(const mi355_w8a8_grouped_problem* p, hipStream_t s) {
  if (!p) return MI355_W8A8_ERR_NULL;
  float* z_rows = nullptr;
  if (p->struct_size == sizeof(mi355_w8a8_grouped_problem_z)) z_rows = reinterpret_cast<const mi355_w8a8_grouped_problem_z*>(p)->z;
  else if (p->struct_size != sizeof(mi355_w8a8_grouped_problem)) return MI355_W8A8_ERR_STRUCT;
  int st = validate_common(p->m, p->k, p->n);
  if (st) return st;
  if (p->n_groups == 0) return MI355_W8A8_ERR_SHAPE;
  if (p->n_groups > (uint32_t)kMaxGroups) return MI355_W8A8_ERR_UNSUPPORTED;
  if (!p->x || !p->w_packed || !p->w_scales || !p->out || !p->group_sizes) return MI355_W8A8_ERR_NULL;
  const bool swiglu = (p->flags & MI355_W8A8_FLAG_SWIGLU) != 0;
  if (swiglu && (p->n & 1u)) return MI355_W8A8_ERR_SHAPE;
  const bool lora = p->rank > 0;
  if (lora) {
    if (!p->lora_a || !p->lora_b || !p->lora_scaling) return MI355_W8A8_ERR_NULL;
    if (p->rank > (uint32_t)kMaxRank) return MI355_W8A8_ERR_UNSUPPORTED;
  }
  const uint32_t gpw = p->groups_per_weight ? p->groups_per_weight : 1u;
  if (p->n_groups % gpw) return MI355_W8A8_ERR_SHAPE;
  const uint32_t n_out = swiglu ? p->n / 2u : p->n;
  const uint64_t out_bytes = (uint64_t)p->m * n_out * 2u;
  if (!aligned16(p->x) || !aligned16(p->w_packed) || !aligned16(p->out) || !aligned16(p->w_scales) ||
      !aligned16(p->lora_a) || !aligned16(p->lora_b) || !aligned16(z_rows) || (reinterpret_cast<uintptr_t>(p->group_sizes) & 3u))
    return MI355_W8A8_ERR_ALIGN;
  if (z_rows && !lora) return MI355_W8A8_ERR_SHAPE;
  const uint32_t x_repeat = p->x_row_map ? p->x_row_repeat : 1u;
  if (p->x_row_map && (x_repeat == 0 || (reinterpret_cast<uintptr_t>(p->x_row_map) & 3u)))
    return x_repeat == 0 ? MI355_W8A8_ERR_SHAPE : MI355_W8A8_ERR_ALIGN;
  // with a row map x holds one row per token unless the caller says otherwise; gathered reads are
  // clamped to these rows
  const uint32_t x_rows = (p->x_row_map && p->x_rows) ? p->x_rows : (p->m + x_repeat - 1u) / x_repeat;
  const uint64_t z_bytes = (uint64_t)p->m * p->rank * 4u;
  if (overlaps(p->out, out_bytes, p->x, (uint64_t)x_rows * p->k * 2u) ||
      overlaps(p->out, out_bytes, p->x_row_map, (uint64_t)p->m * 4u) ||
      overlaps(p->out, out_bytes, p->workspace, p->workspace_bytes) || overlaps(z_rows, z_bytes, p->out, out_bytes) ||
      overlaps(z_rows, z_bytes, p->x, (uint64_t)x_rows * p->k * 2u) || overlaps(z_rows, z_bytes, p->workspace, p->workspace_bytes))
    return MI355_W8A8_ERR_ALIAS;
  if ((p->flags & MI355_W8A8_FLAG_GROUPED_TILE64) && (p->flags & MI355_W8A8_FLAG_GROUPED_TILE128))
    return MI355_W8A8_ERR_SHAPE;
  const GroupedLayout w = make_grouped_layout(p->m, p->k, p->n, p->n_groups, p->rank, p->flags);
  if (!p->workspace || p->workspace_bytes < w.total) return MI355_W8A8_ERR_WORKSPACE;
  if (reinterpret_cast<uintptr_t>(p->workspace) & 255u) return MI355_W8A8_ERR_ALIGN;
  unsigned char* ws = static_cast<unsigned char*>(p->workspace);
  int32_t* src_row = reinterpret_cast<int32_t*>(ws + w.src_row);
  int32_t* blk_range = reinterpret_cast<int32_t*>(ws + w.blk_range);
  (void)hipGetLastError();

  // measurement only: a call with SKIP_PROLOGUE after a full call with the same arguments and workspace
  // re-runs only the GEMM kernel; SKIP_GEMM stops after routing / quantization / LoRA-A
  const bool skip_prologue = (p->flags & MI355_W8A8_FLAG_SKIP_PROLOGUE) != 0;
  const bool skip_gemm = (p->flags & MI355_W8A8_FLAG_SKIP_GEMM) != 0;
  if (skip_prologue && (p->aux_x_codes || p->aux_x_scales)) return MI355_W8A8_ERR_UNSUPPORTED;

  // Launch 1: the slot layout of the groups next to the rows' statistics and the LoRA operand layouts.  With a row map the
  // statistics are the source rows' (a token's row is read once, not once per expert), unless there are more of those than rows.
  const bool by_source = p->x_row_map && x_rows <= p->m;
  if (!skip_prologue) {
    LoraPrepArgs pa{};
    pa.src_row = src_row; pa.blk_range = blk_range;
    pa.group_sizes = p->group_sizes;
    pa.tile_tab = reinterpret_cast<uint64_t*>(ws + w.tile_tab); pa.tile_blocks = w.tile_blocks;
    pa.zero_out = static_cast<uint16_t*>(p->out); pa.zero_cols = n_out;
    pa.lora_a = static_cast<const uint16_t*>(p->lora_a);
    pa.lora_b = static_cast<const uint16_t*>(p->lora_b);
    pa.at = reinterpret_cast<uint16_t*>(ws + w.at);
    pa.bp = ws + w.bp;
    pa.M = p->m; pa.K = p->k; pa.N = p->n; pa.n_groups = p->n_groups; pa.r = p->rank; pa.nkk = w.nkk;
    pa.ncb = n_padded(p->n) / 32u; pa.slots = w.slots;
    // (the layout is filled slot by slot: a few workgroups, each with the prefix sums of its own)
    pa.route_blocks = (w.slots + 2047u) / 2048u < 16u ? (w.slots + 2047u) / 2048u : 16u;
    pa.a_operand_kb = w.KB;
    pa.stat_rows = by_source ? x_rows : p->m;
    pa.stat_blocks = (pa.stat_rows + 15u) / 16u;
    pa.x = static_cast<const uint16_t*>(p->x);
    if (p->x_row_map && !by_source) { pa.stat_map = p->x_row_map; pa.stat_div = x_repeat; pa.stat_limit = x_rows; }
    pa.row_scale = reinterpret_cast<float*>(ws + w.row_scale);
    uint32_t b_blocks = 0;
    // (a caller that vouches for the operand packs of an earlier call on this workspace keeps them)
    if (lora && !(p->flags & MI355_W8A8_FLAG_LORA_PACK_VALID)) {
      const uint64_t a_items = (uint64_t)p->n_groups * w.KB * w.nkk * (p->rank % 4u ? 64u : 16u);
      const uint64_t b_items = (uint64_t)p->n_groups * pa.ncb * w.nkk * (p->n % 4u ? 64u : 16u);
      pa.a_blocks = (uint32_t)((a_items + 1023u) / 1024u);
      b_blocks = (uint32_t)((b_items + 1023u) / 1024u);
    }
    hipLaunchKernelGGL((lora_prep_kernel<1>), dim3(pa.route_blocks + pa.stat_blocks + pa.a_blocks + b_blocks), dim3(1024), 0, s, pa);
    if ((st = launch_status())) return st;
  }

  // launch 2: codes and LoRA-A projection in one pass over the gathered rows
  if (!skip_prologue) {
    QuantLoraArgs q{};
    q.x = static_cast<const uint16_t*>(p->x);
    q.row_scale = reinterpret_cast<const float*>(ws + w.row_scale);
    q.M = p->m; q.K = p->k; q.K_pad = w.K_pad; q.KB = w.KB;
    q.n_half_blocks = w.slots / 16u;
    q.src_row = src_row; q.blk_range = blk_range;
    q.xq_packed = ws + w.xq;
    q.sx_slots = reinterpret_cast<float*>(ws + w.sx);
    q.at = lora ? reinterpret_cast<const uint16_t*>(ws + w.at) : nullptr;
    q.zp = ws + w.zp;
    q.r = p->rank; q.nkk = w.nkk;
    q.nterms = (p->flags & MI355_W8A8_FLAG_LORA_SPLIT2) ? 2u : 3u;
    q.group_pad = 32u;
    q.row_map = p->x_row_map; q.row_div = x_repeat; q.row_limit = x_rows; q.scale_by_source = by_source ? 1u : 0u;
    q.z_rows = z_rows;
    if ((st = launch_grouped_quant(q, lora ? w.nkk : 0u, s))) return st;
    if (p->aux_x_codes || p->aux_x_scales) {  // the caller's copies: of every row (some have no slot), then what the GEMM reads
      QuantArgs c{};
      c.x = static_cast<const uint16_t*>(p->x);
      c.M = p->m; c.K = p->k;
      c.codes_rm = p->aux_x_codes;
      c.scales_rm = p->aux_x_scales;
      c.row_map = p->x_row_map; c.row_div = x_repeat; c.row_limit = x_rows;
      if ((st = launch_quant(c, s))) return st;
      hipLaunchKernelGGL(codes_row_major_kernel, dim3(w.slots), dim3(256), 0, s, q.xq_packed, q.sx_slots, src_row,
                         p->aux_x_codes, p->aux_x_scales, p->m, p->k, w.KB);
      if ((st = launch_status())) return st;
    }
  }
  if (skip_gemm) return MI355_W8A8_OK;

  GemmArgs g{};
  g.xq = ws + w.xq;
  g.wp = static_cast<const unsigned char*>(p->w_packed);
  g.sx = reinterpret_cast<const float*>(ws + w.sx);
  g.sw = p->w_scales;
  g.zp = lora ? ws + w.zp : nullptr;
  g.bp = lora ? ws + w.bp : nullptr;
  g.lora_scaling = p->lora_scaling;
  g.src_row = src_row;
  g.slot_group = nullptr;
  g.blk_range = blk_range;
  g.residual = nullptr;
  g.out = p->out;
  g.w_group_stride = mi355_w8a8_packed_weight_bytes(p->k, p->n);
  g.M = p->m; g.N = p->n; g.K_pad = w.K_pad; g.KB = w.KB; g.slots = w.slots;
  g.total_rows = w.slots;
  g.tiles_m = w.max_tiles;
  g.tiles_n = n_padded(p->n) / kGroupedTileN;
  g.tile_tab = reinterpret_cast<const uint64_t*>(ws + w.tile_tab);
  g.rank = p->rank;
  g.groups_per_weight = gpw;
  const bool tall = w.tile_blocks == 8u;
  if (p->aux_acc) {
    GemmArgs ga = g;
    ga.out = p->aux_acc;
    if ((st = tall ? launch_grouped_one<kEpiAcc, 0, 8>(ga, s) : launch_grouped_one<kEpiAcc, 0, 4>(ga, s))) return st;
  }
  if (tall) return swiglu ? launch_grouped<kEpiSwiglu, 8>(g, w.nkk, s) : launch_grouped<kEpiPlain, 8>(g, w.nkk, s);
  return swiglu ? launch_grouped<kEpiSwiglu, 4>(g, w.nkk, s) : launch_grouped<kEpiPlain, 4>(g, w.nkk, s);
}

// ---------------------------------------------------------------------------------------
// backward
// ---------------------------------------------------------------------------------------
struct BwdLayout {
  BwdDxSplit split;
  uint64_t part;
  uint64_t dyp, swp, at, ap, rp, z, r_raw, rs, rpart, zpart, row_dot, src_row, slot_group, blk_range, group_off, partA, partB, total;
  uint64_t beyond;  // group-scaled calls
  uint32_t part_blocks;
  uint32_t slots, nkk, K_pad, KB, N_pad, NB, tiles_m, tiles_k, max_chunks, R, n_slices, groups_per_slice;
};

// Workgroups of the preparation that lay out A for the pull-back's epilogue.
uint32_t bwd_ap_blocks(uint32_t n_groups, uint32_t KB, uint32_t nkk) { return (uint32_t)(((uint64_t)n_groups * KB * nkk * 64u + 1023u) / 1024u); }

// K slices of z = x @ A: a call of few row blocks still fills the chip.  A slice keeps at least one 64-wide step for each of
// the 16 waves, and the count depends on K and N only, so that a grouped call and the dense calls over its groups add in the
// same order.
uint32_t bwd_z_slices(uint32_t k, uint32_t n_slices) {
  const uint32_t by_steps = (k + 63u) / 64u / 16u ? (k + 63u) / 64u / 16u : 1u;
  return by_steps < n_slices ? by_steps : n_slices;
}

// gq_k_pad: padded K of a group-scaled weight (its own k blocks, tiles of 128 k), or 0
BwdLayout make_bwd_layout(uint32_t m, uint32_t k, uint32_t n, uint32_t n_groups, uint32_t rank, uint32_t gq_k_pad = 0u) {
  BwdLayout w{};
  w.K_pad = gq_k_pad ? gq_k_pad : k_padded(k); w.KB = w.K_pad / 32u;
  w.N_pad = n_padded(n); w.NB = w.N_pad / 32u;
  w.slots = round_up(m, kTileM);
  w.tiles_m = w.slots / 256u;
  w.tiles_k = gq_k_pad ? (w.K_pad + 127u) / 128u : (w.K_pad + 255u) / 256u;
  w.nkk = rank_chunks(rank);
  w.R = w.nkk > 2u ? 64u : 32u;  // rank rows of a partial (32-wide rank blocks)
  w.max_chunks = (m + kBwdChunkRows - 1u) / kBwdChunkRows + n_groups;
  {  // dy is packed (and r accumulated) by workgroups that own a slice of the 128-column groups
    const uint32_t ng = w.N_pad / 128u;
    w.n_slices = (ng + 3u) / 4u < kBwdMaxSlices ? (ng + 3u) / 4u : kBwdMaxSlices;
    w.groups_per_slice = (ng + w.n_slices - 1u) / w.n_slices;
  }
  const uint32_t k_blocks = gq_k_pad ? 1u : 2u;  // of a wave's tile
  w.split = bwd_dx_split(w.tiles_m, w.tiles_k, w.NB, k_blocks);
  w.part_blocks = w.tiles_m > 1u ? 8u : (m + 31u) / 32u;
  uint64_t off = 0;
  w.part = off;
  if (w.split.sk_wgs)  // a partial tile per workgroup, and another wherever a tile ends inside its stages
    off += (uint64_t)(w.split.sk_wgs + w.tiles_m * w.tiles_k - w.split.direct_tiles) * w.part_blocks * kBwdPartBlockFloats * k_blocks * 4u;
  w.dyp = off; off += align256((uint64_t)w.slots * w.N_pad * 2u);
  w.swp = off; off += align256((uint64_t)(w.N_pad + kBwdScalePad) * 4u);  // a stage fetches 1 KiB of scales starting at its own 32
  w.src_row = off; off += align256((uint64_t)w.slots * 4u);
  w.slot_group = off; off += align256((uint64_t)w.slots * 4u);
  w.blk_range = off; off += align256((uint64_t)(w.slots / 32u) * 4u);
  w.group_off = off; off += align256((uint64_t)(kMaxAdapters + 1) * 4u);
  if (rank) {
    w.at = off; off += align256((uint64_t)n_groups * rank * k * 2u);
    w.ap = off; off += align256((uint64_t)n_groups * w.KB * w.nkk * kBlockBytes);
    w.rp = off; off += align256((uint64_t)(w.slots / 32u) * w.nkk * 3u * kBlockBytes);
    w.z = off; off += align256((uint64_t)w.slots * kBwdRankStride * 4u);
    w.r_raw = off; off += align256((uint64_t)w.slots * kBwdRankStride * 4u);
    w.rs = off; off += align256((uint64_t)w.slots * kBwdRankStride * 4u);
    w.rpart = off; off += align256((uint64_t)w.n_slices * w.slots * kBwdRankStride * 4u);
    w.zpart = off; off += align256((uint64_t)bwd_z_slices(k, w.n_slices) * w.slots * kBwdRankStride * 4u);
    w.row_dot = off; off += align256((uint64_t)w.slots * 8u);
    w.partA = off; off += align256((uint64_t)w.max_chunks * w.R * k * 4u);
    w.partB = off; off += align256((uint64_t)w.max_chunks * w.R * n * 4u);
    w.beyond = off; off += gq_k_pad ? align256((1u + bwd_ap_blocks(n_groups, w.KB, w.nkk)) * 4u) : 0u;
  }
  w.total = off;
  return w;
}

int validate_bwd_dims(uint32_t m, uint32_t k, uint32_t n, uint32_t n_adapters, uint32_t rank) {
  int st = validate_common(m, k, n);
  if (st) return st;
  if (n % 8u) return MI355_W8A8_ERR_UNSUPPORTED;
  if ((uint64_t)m * k >= (1ull << 32) - (1ull << 20)) return MI355_W8A8_ERR_UNSUPPORTED;  // 32-bit offsets
  if (n_adapters > (uint32_t)kMaxAdapters || rank > (uint32_t)kMaxRank) return MI355_W8A8_ERR_UNSUPPORTED;
  if (n_adapters && rank == 0) return MI355_W8A8_ERR_UNSUPPORTED;
  return MI355_W8A8_OK;
}

template <int NKK>
int launch_bwd_dx(const BwdDxArgs& g, bool rows128, hipStream_t s) {
  uint32_t want = ((g.direct_tiles + 7u) / 8u) * 8u;
  if (g.sk_wgs > want) want = g.sk_wgs;
  const dim3 grid(want < 256u ? want : 256u);
  const auto kernel = rows128 ? &bwd_dx_kernel<NKK> : &bwd_dx_wide_kernel<NKK>;
  if (hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, kBwdLdsBytes) != hipSuccess)
    return MI355_W8A8_ERR_LAUNCH;
  hipLaunchKernelGGL(kernel, grid, dim3(rows128 ? 512 : 256), kBwdLdsBytes, s, g);
  if (!g.sk_wgs) return launch_status();
  if (const int st = launch_status()) return st;
  const uint32_t split_tiles = g.tiles_m * g.tiles_k - g.direct_tiles;
  hipLaunchKernelGGL((bwd_dx_finish_kernel<NKK, 2>), dim3(split_tiles * 8u), dim3(256), 0, s, g);
  return launch_status();
}

// The stages of a backward call behind its routing tables: dy into operand order (with the partial
// sums of r = dy @ B.T), r and z finished, the pull-back GEMM, the LoRA cotangents.  The dense call
// and the grouped call differ only in who wrote the tables and in the per-tile weights.
struct BwdBody {
  uint32_t m, k, n, n_groups, rank;
  const void* x; const void* dy; const void* w_packed;
  const void* lora_b; const float* lora_scaling;
  void* dx; void* d_lora_a; void* d_lora_b; float* d_lora_scaling;
  bool lora, want_grads, skip_prologue, skip_gemm;
  // tables (null: identity routing, everything in group 0)
  const int32_t* src_row; const int32_t* slot_group; const int32_t* blk_range; const int32_t* group_off;
  // grouped calls only
  const int32_t* x_row; uint32_t x_rows;  // src_row and the rows of x where x is gathered, or null
  const int32_t* skip_range;  // blk_range again when blocks without rows are to be skipped
  const int32_t* tile_weight; const int32_t* chunk_tab; const int32_t* chunk0; const int32_t* group_beg;
  const int32_t* group_end;
  size_t w_stride; uint32_t sw_stride;
  bool rows128;  // the pull-back runs 128-row x 512-k tiles (the tables are padded to match)
  BwdDxSplit split; uint64_t part; uint32_t part_blocks;  // dense calls
  // group-scaled weights: their format (weight_bits 0: per-channel), A itself and the notes of non-finite operands
  uint32_t weight_bits, group, terms; const float* w_scales;
  const void* lora_a; uint64_t beyond;
  const float* z_rows;  // x @ A[idx] as the forward left it, or null
};

template <bool W4, int TERMS, int NKK>
int launch_gq_bwd_dx_one(const GqBwdDxArgs& a, hipStream_t s) {
  const BwdDxArgs& g = a.g;
  uint32_t want = ((g.direct_tiles + 7u) / 8u) * 8u;
  if (g.sk_wgs > want) want = g.sk_wgs;
  const dim3 grid(want < 256u ? want : 256u), block(256);
  if (hipFuncSetAttribute(reinterpret_cast<const void*>(&gq_bwd_dx_wide_kernel<W4, TERMS, NKK>),
                          hipFuncAttributeMaxDynamicSharedMemorySize, kGqBwdLdsBytes) != hipSuccess)
    return MI355_W8A8_ERR_LAUNCH;
  hipLaunchKernelGGL((gq_bwd_dx_wide_kernel<W4, TERMS, NKK>), grid, block, kGqBwdLdsBytes, s, a);
  if (!g.sk_wgs) return launch_status();
  if (const int st = launch_status()) return st;
  hipLaunchKernelGGL((bwd_dx_finish_kernel<NKK, 1>), dim3((g.tiles_m * g.tiles_k - g.direct_tiles) * 8u), dim3(256), 0, s, g);
  return launch_status();
}
template <int NKK>
int launch_gq_bwd_dx(const GqBwdDxArgs& a, uint32_t bits, uint32_t terms, hipStream_t s) {
  if (bits == 4u) return terms == 2u ? launch_gq_bwd_dx_one<true, 2, NKK>(a, s) : launch_gq_bwd_dx_one<true, 3, NKK>(a, s);
  return terms == 2u ? launch_gq_bwd_dx_one<false, 2, NKK>(a, s) : launch_gq_bwd_dx_one<false, 3, NKK>(a, s);
}

template <class Layout>
int launch_bwd_body(const BwdBody& b, const Layout& w, unsigned char* ws, hipStream_t s) {
  int st;
  uint32_t* const beyond = b.lora && b.weight_bits ? reinterpret_cast<uint32_t*>(ws + b.beyond) : nullptr;
  if (!b.skip_prologue) {  // dy into operand order; the same pass leaves the partial sums of r = dy @ B.T
    BwdPackDyArgs d{};
    d.dy = static_cast<const uint16_t*>(b.dy);
    d.src_row = b.src_row; d.slot_group = b.slot_group; d.blk_range = b.blk_range;
    d.dyp = ws + w.dyp;
    d.lora_b = static_cast<const uint16_t*>(b.lora_b);
    d.rpart = b.lora ? reinterpret_cast<float*>(ws + w.rpart) : nullptr;
    d.M = b.m; d.N = b.n; d.NB = w.NB; d.n_row_blocks = w.slots / 32u; d.n_col_groups = w.N_pad / 128u;
    d.n_slices = w.n_slices; d.groups_per_slice = w.groups_per_slice; d.r = b.rank; d.slots = w.slots;
    const dim3 grid(d.n_row_blocks * d.n_slices), block(256);
    if (b.weight_bits) {
      if (!b.lora) hipLaunchKernelGGL((gq_bwd_pack_dy_kernel<0>), grid, block, 0, s, d);
      else if (w.nkk > 2u) hipLaunchKernelGGL((gq_bwd_pack_dy_kernel<2>), grid, block, 0, s, d);
      else hipLaunchKernelGGL((gq_bwd_pack_dy_kernel<1>), grid, block, 0, s, d);
    } else if (!b.lora) hipLaunchKernelGGL((bwd_pack_dy_kernel<0>), grid, block, 0, s, d);
    else if (w.nkk > 2u) hipLaunchKernelGGL((bwd_pack_dy_kernel<2>), grid, block, 0, s, d);
    else hipLaunchKernelGGL((bwd_pack_dy_kernel<1>), grid, block, 0, s, d);
    if ((st = launch_status())) return st;
  }
  if (b.lora && !b.skip_prologue) {
    BwdRFinishArgs f{};
    f.rpart = reinterpret_cast<const float*>(ws + w.rpart);
    f.zpart = reinterpret_cast<const float*>(ws + w.zpart);
    f.slot_group = b.slot_group;
    f.blk_range = b.skip_range;
    f.lora_scaling = b.lora_scaling;
    f.r_raw = reinterpret_cast<float*>(ws + w.r_raw);
    f.rs = reinterpret_cast<float*>(ws + w.rs);
    f.rp = ws + w.rp;
    f.z = reinterpret_cast<float*>(ws + w.z);
    f.row_dot = reinterpret_cast<double*>(ws + w.row_dot);
    f.r = b.rank;
    f.n_slices = w.n_slices; f.slots = w.slots; f.nkk = w.nkk; f.cols = w.nkk > 2u ? 64u : 32u;
    f.beyond = beyond;
    // z = x @ A, as the forward left it or formed again (and, of a group-scaled call, looked at for x).  Formed again it is a launch over all
    // of x and one for A transposed: 42 us of an MLP's step at 3003 rows, 32 of an expert layer's at 1021 tokens.
    if (b.z_rows && (b.d_lora_b || b.d_lora_scaling)) {
      f.z_rows = b.z_rows; f.src_row = b.src_row; f.M = b.m;
    } else if (b.d_lora_b || b.d_lora_scaling || (beyond && b.d_lora_a)) {
      LoraAArgs lz{};
      lz.xsrc = static_cast<const uint16_t*>(b.x);
      lz.at = reinterpret_cast<const uint16_t*>(ws + w.at);
      lz.src_row = b.x_row ? b.x_row : b.src_row; lz.slot_group = b.slot_group; lz.blk_range = b.blk_range;
      lz.M = b.x_row ? b.x_rows : b.m; lz.K = b.k; lz.r = b.rank;
      lz.n_steps = (b.k + 63u) / 64u;
      lz.n_blocks = w.slots / 32u;
      const uint32_t nks = bwd_z_slices(b.k, w.n_slices);
      lz.n_ksplit = nks;
      lz.steps_per_wave = ((lz.n_steps + nks - 1u) / nks + 15u) / 16u;
      lz.zf = reinterpret_cast<float*>(ws + w.zpart);
      lz.zf_stride = kBwdRankStride;
      lz.zf_slice = w.slots * kBwdRankStride;
      const dim3 grid(lz.n_blocks * nks);
      if ((st = launch_lora_a(lz, w.nkk, grid, s))) return st;
      f.z_slices = nks;
    }
    hipLaunchKernelGGL(bwd_r_finish_kernel, dim3(w.slots / 32u), dim3(256), 0, s, f);
    if ((st = launch_status())) return st;
  }
  if (!b.skip_gemm) {
    BwdDxArgs g{};
    g.dyp = ws + w.dyp;
    g.wp = static_cast<const unsigned char*>(b.w_packed);
    g.swp = reinterpret_cast<const float*>(ws + w.swp);
    g.rp = b.lora ? ws + w.rp : nullptr;
    g.ap = b.lora ? ws + w.ap : nullptr;
    g.src_row = b.src_row; g.slot_group = b.slot_group; g.blk_range = b.blk_range;
    g.dx = static_cast<uint16_t*>(b.dx);
    g.M = b.m; g.K = b.k; g.KB = w.KB; g.NB = w.NB; g.tiles_m = w.tiles_m; g.tiles_k = w.tiles_k;
    g.tile_weight = b.tile_weight; g.w_stride = b.w_stride; g.sw_stride = b.sw_stride;
    g.direct_tiles = b.split.sk_wgs ? b.split.direct_tiles : w.tiles_m * w.tiles_k;
    g.sk_q = b.split.sk_q; g.sk_wgs = b.split.sk_wgs;
    g.part = b.split.sk_wgs ? reinterpret_cast<float*>(ws + b.part) : nullptr;
    g.part_blocks = b.part_blocks;
    if (b.weight_bits) {
      GqBwdDxArgs a{};
      a.g = g;
      a.ws = b.w_scales; a.N = b.n; a.group = b.group; a.weight_nb = (b.n + 31u) / 32u;
      switch (b.lora ? w.nkk : 0u) {
        case 0: st = launch_gq_bwd_dx<0>(a, b.weight_bits, b.terms, s); break;
        case 1: st = launch_gq_bwd_dx<1>(a, b.weight_bits, b.terms, s); break;
        case 2: st = launch_gq_bwd_dx<2>(a, b.weight_bits, b.terms, s); break;
        default: st = launch_gq_bwd_dx<4>(a, b.weight_bits, b.terms, s); break;
      }
    } else switch (b.lora ? w.nkk : 0u) {
      case 0: st = launch_bwd_dx<0>(g, b.rows128, s); break;
      case 1: st = launch_bwd_dx<1>(g, b.rows128, s); break;
      case 2: st = launch_bwd_dx<2>(g, b.rows128, s); break;
      default: st = launch_bwd_dx<4>(g, b.rows128, s); break;
    }
    if (st) return st;
  }
  BwdReduceArgs r{};
  if (b.lora && b.want_grads) {
    BwdDloraArgs d{};
    d.x = static_cast<const uint16_t*>(b.x);
    d.dy = static_cast<const uint16_t*>(b.dy);
    d.rs = reinterpret_cast<const float*>(ws + w.rs);
    d.z = reinterpret_cast<const float*>(ws + w.z);
    d.src_row = b.src_row;
    d.x_row = b.x_row ? b.x_row : b.src_row;
    d.group_off = b.group_off;
    d.chunk_tab = b.chunk_tab;
    d.partA = reinterpret_cast<float*>(ws + w.partA);
    d.partB = reinterpret_cast<float*>(ws + w.partB);
    d.chunk0_tab = b.chunk0;
    d.d_a = static_cast<uint16_t*>(b.d_lora_a); d.d_b = static_cast<uint16_t*>(b.d_lora_b);
    d.lora_scaling = b.lora_scaling;
    d.M = b.m; d.K = b.k; d.N = b.n; d.r = b.rank; d.n_groups = b.n_groups; d.max_chunks = w.max_chunks;
    d.col_tiles_a = b.d_lora_a ? (b.k + 255u) / 256u : 0u;
    d.col_tiles_b = b.d_lora_b ? (b.n + 255u) / 256u : 0u;
    if (d.col_tiles_a + d.col_tiles_b) {
      const dim3 grid(w.max_chunks * (d.col_tiles_a + d.col_tiles_b)), block(256);
      const uint32_t lds_bytes = (kBwdStageRows / 32u) * (w.R / 32u) * 6u * kBlockBytes;
      if (w.R == 32u) {
        hipLaunchKernelGGL((bwd_dlora_kernel<1>), grid, block, lds_bytes, s, d);
      } else {
        if (hipFuncSetAttribute(reinterpret_cast<const void*>(&bwd_dlora_kernel<2>),
                                hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes) != hipSuccess)
          return MI355_W8A8_ERR_LAUNCH;
        hipLaunchKernelGGL((bwd_dlora_kernel<2>), grid, block, lds_bytes, s, d);
      }
      if ((st = launch_status())) return st;
    }
    r.partA = d.partA; r.partB = d.partB;
    r.r_raw = reinterpret_cast<const float*>(ws + w.r_raw);
    r.z = d.z;
    r.row_dot = reinterpret_cast<const double*>(ws + w.row_dot);
    r.lora_scaling = b.lora_scaling;
    r.group_off = b.group_off;
    r.chunk0_tab = b.chunk0; r.group_beg = b.group_beg; r.group_end = b.group_end;
    r.d_a = static_cast<uint16_t*>(b.d_lora_a);
    r.d_b = static_cast<uint16_t*>(b.d_lora_b);
    r.d_s = b.d_lora_scaling;
    r.K = b.k; r.N = b.n; r.r = b.rank; r.R = w.R; r.n_groups = b.n_groups;
    r.blocks_a = b.d_lora_a ? b.n_groups * ((b.k + kBwdReduceCols - 1u) / kBwdReduceCols) : 0u;
    r.blocks_b = b.d_lora_b ? (uint32_t)(((uint64_t)b.n_groups * b.rank * b.n / 4u + 255u) / 256u) : 0u;
  }
  if (b.lora && (b.want_grads || (beyond && !b.skip_gemm))) {
    const uint32_t blocks = r.blocks_a + r.blocks_b + (b.d_lora_scaling ? b.n_groups : 0u);
    if (beyond) {
      GqBwdPlain q{};
      q.beyond = beyond; q.n_beyond = 1u + bwd_ap_blocks(b.n_groups, w.KB, w.nkk);
      q.x = static_cast<const uint16_t*>(b.x); q.dy = static_cast<const uint16_t*>(b.dy);
      q.lora_a = static_cast<const uint16_t*>(b.lora_a); q.lora_b = static_cast<const uint16_t*>(b.lora_b);
      q.rs = reinterpret_cast<const float*>(ws + w.rs);
      q.dx = b.skip_gemm ? nullptr : static_cast<uint16_t*>(b.dx);
      q.wp = static_cast<const unsigned char*>(b.w_packed); q.ws = b.w_scales;
      q.M = b.m; q.K = b.k; q.N = b.n; q.r = b.rank; q.KB = w.KB; q.group = b.group; q.bits = b.weight_bits;
      hipLaunchKernelGGL((bwd_dlora_reduce_kernel<GqBwdPlain>), dim3(blocks + (q.dx ? kGqPlainDxBlocks : 0u)), dim3(256), 0, s, r, q);
    } else {
      hipLaunchKernelGGL((bwd_dlora_reduce_kernel<BwdNoPlain>), dim3(blocks), dim3(256), 0, s, r, BwdNoPlain{});
    }
    if ((st = launch_status())) return st;
  }
  return MI355_W8A8_OK;
}

int run_backward(const mi355_w8a8_bwd_problem* p, hipStream_t s) {
  if (!p) return MI355_W8A8_ERR_NULL;
  const float* z_rows = nullptr;
  if (p->struct_size == sizeof(mi355_w8a8_bwd_problem_z)) z_rows = reinterpret_cast<const mi355_w8a8_bwd_problem_z*>(p)->z;
  else if (p->struct_size != sizeof(mi355_w8a8_bwd_problem)) return MI355_W8A8_ERR_STRUCT;
  int st = validate_bwd_dims(p->m, p->k, p->n, p->n_adapters, p->rank);
  if (st) return st;
  if (p->flags & ~(MI355_W8A8_FLAG_SKIP_PROLOGUE | MI355_W8A8_FLAG_SKIP_GEMM)) return MI355_W8A8_ERR_SHAPE;
  const bool skip_prologue = (p->flags & MI355_W8A8_FLAG_SKIP_PROLOGUE) != 0;  // measurement: the workspace holds a previous call's tables
  const bool skip_gemm = (p->flags & MI355_W8A8_FLAG_SKIP_GEMM) != 0;
  if (!p->dy || !p->w_packed || !p->w_scales || !p->dx) return MI355_W8A8_ERR_NULL;
  const bool lora = p->n_adapters > 0;
  const bool want_grads = p->d_lora_a || p->d_lora_b || p->d_lora_scaling;
  if (lora) {
    if (!p->lora_a || !p->lora_b || !p->lora_scaling) return MI355_W8A8_ERR_NULL;
    if (want_grads && !p->x) return MI355_W8A8_ERR_NULL;
  } else if (p->adapter_indices || want_grads) {
    return MI355_W8A8_ERR_SHAPE;
  }
  if (!aligned16(p->x) || !aligned16(p->dy) || !aligned16(p->w_packed) || !aligned16(p->w_scales) ||
      !aligned16(p->lora_a) || !aligned16(p->lora_b) || !aligned16(p->dx) || !aligned16(p->d_lora_a) ||
      !aligned16(p->d_lora_b) || !aligned16(p->adapter_indices) || !aligned16(z_rows))
    return MI355_W8A8_ERR_ALIGN;
  if (z_rows && !lora) return MI355_W8A8_ERR_SHAPE;
  const uint64_t dx_bytes = (uint64_t)p->m * p->k * 2u, dy_bytes = (uint64_t)p->m * p->n * 2u;
  const uint64_t a_bytes = (uint64_t)p->n_adapters * p->rank * p->k * 2u, b_bytes = (uint64_t)p->n_adapters * p->rank * p->n * 2u;
  if (overlaps(z_rows, (uint64_t)p->m * p->rank * 4u, p->dx, dx_bytes) || overlaps(p->dx, dx_bytes, p->dy, dy_bytes) || overlaps(p->dx, dx_bytes, p->x, dx_bytes) ||
      overlaps(p->dx, dx_bytes, p->workspace, p->workspace_bytes) ||
      overlaps(p->d_lora_a, a_bytes, p->lora_a, a_bytes) || overlaps(p->d_lora_b, b_bytes, p->lora_b, b_bytes) ||
      overlaps(p->d_lora_a, a_bytes, p->workspace, p->workspace_bytes) ||
      overlaps(p->d_lora_b, b_bytes, p->workspace, p->workspace_bytes) ||
      overlaps(p->d_lora_a, a_bytes, p->dx, dx_bytes) || overlaps(p->d_lora_b, b_bytes, p->dx, dx_bytes))
    return MI355_W8A8_ERR_ALIAS;
  const BwdLayout w = make_bwd_layout(p->m, p->k, p->n, p->n_adapters, lora ? p->rank : 0u);
  if (!p->workspace || p->workspace_bytes < w.total) return MI355_W8A8_ERR_WORKSPACE;
  if (reinterpret_cast<uintptr_t>(p->workspace) & 255u) return MI355_W8A8_ERR_ALIGN;
  unsigned char* ws = static_cast<unsigned char*>(p->workspace);
  const bool routed = lora && p->adapter_indices && p->n_adapters > 1;
  int32_t* src_row = reinterpret_cast<int32_t*>(ws + w.src_row);
  int32_t* slot_group = reinterpret_cast<int32_t*>(ws + w.slot_group);
  int32_t* blk_range = reinterpret_cast<int32_t*>(ws + w.blk_range);
  int32_t* group_off = reinterpret_cast<int32_t*>(ws + w.group_off);
  (void)hipGetLastError();

  if (!skip_prologue) {  // tables: routing, A transposed / in operand order, scales in packed column order
    BwdPrepArgs pa{};
    pa.idx = routed ? p->adapter_indices : nullptr;
    pa.src_row = src_row;
    pa.slot_group = slot_group; pa.blk_range = blk_range; pa.group_off = group_off;
    pa.lora_a = static_cast<const uint16_t*>(p->lora_a);
    pa.at = lora ? reinterpret_cast<uint16_t*>(ws + w.at) : nullptr;
    pa.ap = lora ? ws + w.ap : nullptr;
    pa.sw = p->w_scales; pa.swp = reinterpret_cast<float*>(ws + w.swp);
    pa.M = p->m; pa.K = p->k; pa.N = p->n; pa.N_pad = w.N_pad; pa.n_groups = p->n_adapters; pa.r = p->rank;
    pa.nkk = w.nkk; pa.kb32 = w.KB; pa.slots = w.slots;
    pa.route_blocks = lora ? 1u : 0u;
    pa.a_blocks = lora && !z_rows ? (uint32_t)(((uint64_t)p->n_adapters * p->k * ((p->rank + 7u) / 8u) + 1023u) / 1024u) : 0u;
    pa.ap_blocks = lora ? bwd_ap_blocks(p->n_adapters, w.KB, w.nkk) : 0u;
    const uint32_t sw_blocks = (w.N_pad + 1023u) / 1024u;
    hipLaunchKernelGGL(bwd_prep_kernel, dim3(pa.route_blocks + pa.a_blocks + pa.ap_blocks + sw_blocks), dim3(1024), 0, s, pa);
    if ((st = launch_status())) return st;
  }
  BwdBody b{};
  b.m = p->m; b.k = p->k; b.n = p->n; b.n_groups = p->n_adapters; b.rank = p->rank;
  b.x = p->x; b.dy = p->dy; b.w_packed = p->w_packed; b.lora_b = p->lora_b; b.lora_scaling = p->lora_scaling;
  b.dx = p->dx; b.d_lora_a = p->d_lora_a; b.d_lora_b = p->d_lora_b; b.d_lora_scaling = p->d_lora_scaling;
  b.lora = lora; b.want_grads = want_grads; b.skip_prologue = skip_prologue; b.skip_gemm = skip_gemm;
  b.z_rows = z_rows;
  b.src_row = routed ? src_row : nullptr;
  b.slot_group = routed ? slot_group : nullptr;
  b.blk_range = routed ? blk_range : nullptr;
  b.group_off = group_off;
  b.split = w.split; b.part = w.part; b.part_blocks = w.part_blocks;
  return launch_bwd_body(b, w, ws, s);
}

// group-scaled weights: the same stages around the group-scaled pull-back, one adapter
int validate_gq_bwd_dims(uint32_t m, uint32_t k, uint32_t k_pad, uint32_t n, uint32_t group, uint32_t rank) {
  if (m == 0 || k == 0 || n == 0 || k > k_pad) return MI355_W8A8_ERR_SHAPE;
  if (group == 0 || group % 32u || k_pad % group) return MI355_W8A8_ERR_SHAPE;
  if (m > kMaxRows || n > kMaxN || k_pad > kMaxK || k % 8u || n % 8u || rank > (uint32_t)kMaxRank) return MI355_W8A8_ERR_UNSUPPORTED;
  const uint64_t limit = (1ull << 32) - (1ull << 20);  // 32-bit offsets
  if ((uint64_t)m * k >= limit || (uint64_t)m * n >= limit) return MI355_W8A8_ERR_UNSUPPORTED;
  return MI355_W8A8_OK;
}

int run_gq_backward(const mi355_w8a8_gq_bwd_problem* p, hipStream_t s) {
  if (!p) return MI355_W8A8_ERR_NULL;
  if (p->struct_size != sizeof(mi355_w8a8_gq_bwd_problem)) return MI355_W8A8_ERR_STRUCT;
  int st = validate_gq_bwd_dims(p->m, p->k, p->k_pad, p->n, p->group_size, p->rank);
  if (st) return st;
  if (p->flags & ~(MI355_W8A8_FLAG_SKIP_GEMM | MI355_W8A8_FLAG_GQ_BF16_SCALES)) return MI355_W8A8_ERR_SHAPE;
  if (p->weight_bits != 4u && p->weight_bits != 8u) return MI355_W8A8_ERR_SHAPE;
  const bool no_dx = (p->flags & MI355_W8A8_FLAG_SKIP_GEMM) != 0;
  if (!p->dy || !p->w_packed || !p->w_scales || (!p->dx && !no_dx)) return MI355_W8A8_ERR_NULL;
  const bool lora = p->rank > 0;
  const bool want_grads = p->d_lora_a || p->d_lora_b || p->d_lora_scaling;
  if (lora) {
    if (!p->lora_a || !p->lora_b || !p->lora_scaling) return MI355_W8A8_ERR_NULL;
    if (want_grads && !p->x) return MI355_W8A8_ERR_NULL;
  } else if (want_grads) {
    return MI355_W8A8_ERR_SHAPE;
  }
  if (!aligned16(p->x) || !aligned16(p->dy) || !aligned16(p->w_packed) || !aligned16(p->w_scales) ||
      !aligned16(p->lora_a) || !aligned16(p->lora_b) || !aligned16(p->dx) || !aligned16(p->d_lora_a) || !aligned16(p->d_lora_b))
    return MI355_W8A8_ERR_ALIGN;
  const uint64_t dx_bytes = (uint64_t)p->m * p->k * 2u;
  if (!no_dx && (overlaps(p->dx, dx_bytes, p->dy, (uint64_t)p->m * p->n * 2u) || overlaps(p->dx, dx_bytes, p->x, dx_bytes) ||
                 overlaps(p->dx, dx_bytes, p->workspace, p->workspace_bytes)))
    return MI355_W8A8_ERR_ALIAS;
  const BwdLayout w = make_bwd_layout(p->m, p->k, p->n, lora ? 1u : 0u, p->rank, p->k_pad);
  if (!p->workspace || p->workspace_bytes < w.total) return MI355_W8A8_ERR_WORKSPACE;
  if (reinterpret_cast<uintptr_t>(p->workspace) & 255u) return MI355_W8A8_ERR_ALIGN;
  unsigned char* ws = static_cast<unsigned char*>(p->workspace);
  (void)hipGetLastError();
  if (lora) {  // A transposed and in operand order, the group table
    BwdPrepArgs pa{};
    pa.group_off = reinterpret_cast<int32_t*>(ws + w.group_off);
    pa.lora_a = static_cast<const uint16_t*>(p->lora_a);
    pa.at = reinterpret_cast<uint16_t*>(ws + w.at);
    pa.ap = ws + w.ap;
    pa.M = p->m; pa.K = p->k; pa.n_groups = 1u; pa.r = p->rank;
    pa.nkk = w.nkk; pa.kb32 = w.KB; pa.slots = w.slots;
    pa.route_blocks = 1u;
    pa.a_blocks = (uint32_t)(((uint64_t)p->k * ((p->rank + 7u) / 8u) + 1023u) / 1024u);
    pa.ap_blocks = bwd_ap_blocks(1u, w.KB, w.nkk);
    pa.beyond = reinterpret_cast<uint32_t*>(ws + w.beyond);
    hipLaunchKernelGGL(bwd_prep_kernel, dim3(pa.route_blocks + pa.a_blocks + pa.ap_blocks), dim3(1024), 0, s, pa);
    if ((st = launch_status())) return st;
  }
  BwdBody b{};
  b.m = p->m; b.k = p->k; b.n = p->n; b.n_groups = lora ? 1u : 0u; b.rank = p->rank;
  b.x = p->x; b.dy = p->dy; b.w_packed = p->w_packed; b.lora_b = p->lora_b; b.lora_scaling = p->lora_scaling;
  b.dx = p->dx; b.d_lora_a = p->d_lora_a; b.d_lora_b = p->d_lora_b; b.d_lora_scaling = p->d_lora_scaling;
  b.lora = lora; b.want_grads = want_grads; b.skip_gemm = no_dx;
  b.group_off = reinterpret_cast<int32_t*>(ws + w.group_off);
  b.split = w.split; b.part = w.part; b.part_blocks = w.part_blocks;
  b.weight_bits = p->weight_bits; b.group = p->group_size; b.w_scales = p->w_scales;
  b.lora_a = p->lora_a; b.beyond = w.beyond;
  b.terms = (p->flags & MI355_W8A8_FLAG_GQ_BF16_SCALES) ? 2u : 3u;
  return launch_bwd_body(b, w, ws, s);
}

// ---------------------------------------------------------------------------------------
// grouped (per-expert) backward
// ---------------------------------------------------------------------------------------
struct BwdGroupedLayout {
  uint64_t dyp, swp, src_row, slot_group, blk_range, group_beg, group_end, tile_weight, chunk_tab, chunk0,
      at, ap, rp, z, r_raw, rs, rpart, zpart, row_dot, partA, partB, x_row, total;
  uint32_t slots, nkk, K_pad, KB, N_pad, NB, tiles_m, tiles_k, max_chunks, R, n_slices, groups_per_slice, n_weights,
      gpw, sw_stride, tile_rows;
};

BwdGroupedLayout make_bwd_grouped_layout(uint32_t m, uint32_t k, uint32_t n, uint32_t n_groups, uint32_t rank,
                                         uint32_t gpw_in) {
  BwdGroupedLayout w{};
  w.gpw = gpw_in ? gpw_in : 1u;
  w.n_weights = n_groups / w.gpw;
  w.K_pad = k_padded(k); w.KB = w.K_pad / 32u;
  w.N_pad = n_padded(n); w.NB = w.N_pad / 32u;
  // Tile geometry of the pull-back: 256 rows x 256 k, or 128 rows x 512 k (the same area).  The group sizes
  // live on the device, so the choice goes by the average rows per weight: a weight with r rows takes about
  // r / rows + 1/2 row tiles, and the geometry with fewer tiles in total wins (ties keep 256 rows).
  {
    const double avg = (double)m / (double)w.n_weights;
    const double t256 = (avg / 256.0 + 0.5) * (double)((w.KB + 7u) / 8u);
    const double t128 = (avg / 128.0 + 0.5) * (double)((w.KB + 15u) / 16u);
    w.tile_rows = t128 < t256 ? 128u : 256u;
  }
  // every weight with rows pads its slots to a multiple of the tile rows
  const uint32_t with_rows = w.n_weights < m ? w.n_weights : m;
  w.slots = round_up(m + (w.tile_rows - 1u) * with_rows, 256u);
  w.tiles_m = w.slots / w.tile_rows;
  w.tiles_k = w.tile_rows == 128u ? (w.KB + 15u) / 16u : (w.KB + 7u) / 8u;
  w.nkk = rank_chunks(rank);
  w.R = w.nkk > 2u ? 64u : 32u;
  w.max_chunks = (m + kBwdChunkRows - 1u) / kBwdChunkRows + n_groups;
  {
    const uint32_t ng = w.N_pad / 128u;
    w.n_slices = (ng + 3u) / 4u < kBwdMaxSlices ? (ng + 3u) / 4u : kBwdMaxSlices;
    w.groups_per_slice = (ng + w.n_slices - 1u) / w.n_slices;
  }
  w.sw_stride = w.N_pad + kBwdScalePad;
  uint64_t off = 0;
  w.dyp = off; off += align256((uint64_t)w.slots * w.N_pad * 2u);
  w.swp = off; off += align256((uint64_t)w.n_weights * w.sw_stride * 4u);
  w.src_row = off; off += align256((uint64_t)w.slots * 4u);
  w.slot_group = off; off += align256((uint64_t)w.slots * 4u);
  w.blk_range = off; off += align256((uint64_t)(w.slots / 32u) * 4u);
  w.group_beg = off; off += align256((uint64_t)n_groups * 4u);
  w.group_end = off; off += align256((uint64_t)n_groups * 4u);
  w.tile_weight = off; off += align256((uint64_t)w.tiles_m * 4u);
  w.chunk_tab = off; off += align256((uint64_t)w.max_chunks * 12u);
  w.chunk0 = off; off += align256((uint64_t)(n_groups + 1u) * 4u);
  if (rank) {
    w.at = off; off += align256((uint64_t)n_groups * rank * k * 2u);
    w.ap = off; off += align256((uint64_t)n_groups * w.KB * w.nkk * kBlockBytes);
    w.rp = off; off += align256((uint64_t)(w.slots / 32u) * w.nkk * 3u * kBlockBytes);
    w.z = off; off += align256((uint64_t)w.slots * kBwdRankStride * 4u);
    w.r_raw = off; off += align256((uint64_t)w.slots * kBwdRankStride * 4u);
    w.rs = off; off += align256((uint64_t)w.slots * kBwdRankStride * 4u);
    w.rpart = off; off += align256((uint64_t)w.n_slices * w.slots * kBwdRankStride * 4u);
    w.zpart = off; off += align256((uint64_t)bwd_z_slices(k, w.n_slices) * w.slots * kBwdRankStride * 4u);
    w.row_dot = off; off += align256((uint64_t)w.slots * 8u);
    w.partA = off; off += align256((uint64_t)w.max_chunks * w.R * k * 4u);
    w.partB = off; off += align256((uint64_t)w.max_chunks * w.R * n * 4u);
  }
  w.x_row = off; off += rank ? align256((uint64_t)w.slots * 4u) : 0u;
  w.total = off;
  return w;
}

int validate_bwd_grouped_dims(uint32_t m, uint32_t k, uint32_t n, uint32_t n_groups, uint32_t rank, uint32_t gpw) {
  int st = validate_common(m, k, n);
  if (st) return st;
  if (n % 8u) return MI355_W8A8_ERR_UNSUPPORTED;
  if (n_groups == 0) return MI355_W8A8_ERR_SHAPE;
  if (gpw == 0) gpw = 1;
  if (n_groups % gpw) return MI355_W8A8_ERR_SHAPE;
  if (n_groups > (uint32_t)kMaxGroups || rank > (uint32_t)kMaxRank) return MI355_W8A8_ERR_UNSUPPORTED;
  // 32-bit element offsets into dx, and slots that stay below the row limit
  if ((uint64_t)m * k >= (1ull << 32) - (1ull << 20)) return MI355_W8A8_ERR_UNSUPPORTED;
  if ((uint64_t)m + 255ull * (n_groups / gpw) + 256ull > (uint64_t)kMaxRows) return MI355_W8A8_ERR_UNSUPPORTED;
  return MI355_W8A8_OK;
}

int run_grouped_backward(const mi355_w8a8_grouped_bwd_problem* given, hipStream_t s) {
  if (!given) return MI355_W8A8_ERR_NULL;
  constexpr uint32_t kWithoutMap = offsetof(mi355_w8a8_grouped_bwd_problem, x_row_map);
  const bool with_z = given->struct_size == sizeof(mi355_w8a8_grouped_bwd_problem_z);
  if (!with_z && given->struct_size != sizeof(mi355_w8a8_grouped_bwd_problem) && given->struct_size != kWithoutMap) return MI355_W8A8_ERR_STRUCT;
  const float* const z_rows = with_z ? reinterpret_cast<const mi355_w8a8_grouped_bwd_problem_z*>(given)->z : nullptr;
  mi355_w8a8_grouped_bwd_problem problem{};
  memcpy(&problem, given, with_z ? sizeof(problem) : given->struct_size);
  const mi355_w8a8_grouped_bwd_problem* const p = &problem;
  if (p->flags) return MI355_W8A8_ERR_SHAPE;
  int st = validate_bwd_grouped_dims(p->m, p->k, p->n, p->n_groups, p->rank, p->groups_per_weight);
  if (st) return st;
  if (!p->dy || !p->w_packed || !p->w_scales || !p->dx || !p->group_sizes) return MI355_W8A8_ERR_NULL;
  const bool lora = p->rank > 0;
  const bool want_grads = p->d_lora_a || p->d_lora_b || p->d_lora_scaling;
  if (lora) {
    if (!p->lora_a || !p->lora_b || !p->lora_scaling) return MI355_W8A8_ERR_NULL;
    if (want_grads && !p->x) return MI355_W8A8_ERR_NULL;
  } else if (p->lora_a || p->lora_b || want_grads) {
    return MI355_W8A8_ERR_SHAPE;
  }
  if (!aligned16(p->x) || !aligned16(p->dy) || !aligned16(p->w_packed) || !aligned16(p->w_scales) ||
      !aligned16(p->lora_a) || !aligned16(p->lora_b) || !aligned16(p->dx) || !aligned16(p->d_lora_a) ||
      !aligned16(p->d_lora_b) || !aligned16(z_rows) || (reinterpret_cast<uintptr_t>(p->group_sizes) & 3u))
    return MI355_W8A8_ERR_ALIGN;
  if (z_rows && !lora) return MI355_W8A8_ERR_SHAPE;
  const uint32_t x_repeat = p->x_row_map ? p->x_row_repeat : 1u;
  if (p->x_row_map && (x_repeat == 0 || (reinterpret_cast<uintptr_t>(p->x_row_map) & 3u))) return MI355_W8A8_ERR_SHAPE;
  const uint32_t x_rows = (p->x_row_map && p->x_rows) ? p->x_rows : (p->m + x_repeat - 1u) / x_repeat;
  if ((uint64_t)x_rows * p->k >= (1ull << 32) - (1ull << 20)) return MI355_W8A8_ERR_UNSUPPORTED;
  const uint64_t dx_bytes = (uint64_t)p->m * p->k * 2u, dy_bytes = (uint64_t)p->m * p->n * 2u, x_bytes = (uint64_t)x_rows * p->k * 2u;
  const uint64_t a_bytes = (uint64_t)p->n_groups * p->rank * p->k * 2u, b_bytes = (uint64_t)p->n_groups * p->rank * p->n * 2u;
  if (overlaps(z_rows, (uint64_t)p->m * p->rank * 4u, p->dx, dx_bytes) ||
      overlaps(p->dx, dx_bytes, p->dy, dy_bytes) || overlaps(p->dx, dx_bytes, p->x, x_bytes) ||
      overlaps(p->dx, dx_bytes, p->x_row_map, (uint64_t)p->m * 4u) ||
      overlaps(p->dx, dx_bytes, p->workspace, p->workspace_bytes) ||
      overlaps(p->d_lora_a, a_bytes, p->lora_a, a_bytes) || overlaps(p->d_lora_b, b_bytes, p->lora_b, b_bytes) ||
      overlaps(p->d_lora_a, a_bytes, p->workspace, p->workspace_bytes) ||
      overlaps(p->d_lora_b, b_bytes, p->workspace, p->workspace_bytes) ||
      overlaps(p->d_lora_a, a_bytes, p->dx, dx_bytes) || overlaps(p->d_lora_b, b_bytes, p->dx, dx_bytes))
    return MI355_W8A8_ERR_ALIAS;
  const BwdGroupedLayout w = make_bwd_grouped_layout(p->m, p->k, p->n, p->n_groups, p->rank, p->groups_per_weight);
  // (the table of gathered rows lies at the end: a call without a map does without it)
  if (!p->workspace || p->workspace_bytes < (p->x_row_map ? w.total : w.x_row)) return MI355_W8A8_ERR_WORKSPACE;
  if (reinterpret_cast<uintptr_t>(p->workspace) & 255u) return MI355_W8A8_ERR_ALIGN;
  unsigned char* ws = static_cast<unsigned char*>(p->workspace);
  BwdGroupTables tab{};
  if (p->x_row_map && lora) {
    tab.x_row = reinterpret_cast<int32_t*>(ws + w.x_row);
    tab.x_map = p->x_row_map; tab.x_div = x_repeat; tab.x_rows = x_rows;
  }
  tab.src_row = reinterpret_cast<int32_t*>(ws + w.src_row);
  tab.slot_group = reinterpret_cast<int32_t*>(ws + w.slot_group);
  tab.blk_range = reinterpret_cast<int32_t*>(ws + w.blk_range);
  tab.group_beg = reinterpret_cast<int32_t*>(ws + w.group_beg);
  tab.group_end = reinterpret_cast<int32_t*>(ws + w.group_end);
  tab.tile_weight = reinterpret_cast<int32_t*>(ws + w.tile_weight);
  tab.chunk_tab = reinterpret_cast<int32_t*>(ws + w.chunk_tab);
  tab.chunk0 = reinterpret_cast<int32_t*>(ws + w.chunk0);
  (void)hipGetLastError();

  {  // tables: routing, A transposed / in operand order, every weight's scales in packed column order
    BwdGroupedPrepArgs pa{};
    pa.group_sizes = p->group_sizes;
    pa.tab = tab;
    pa.lora_a = static_cast<const uint16_t*>(p->lora_a);
    pa.at = lora ? reinterpret_cast<uint16_t*>(ws + w.at) : nullptr;
    pa.ap = lora ? ws + w.ap : nullptr;
    pa.sw = p->w_scales; pa.swp = reinterpret_cast<float*>(ws + w.swp);
    pa.dx = static_cast<uint16_t*>(p->dx);
    pa.M = p->m; pa.K = p->k; pa.N = p->n; pa.N_pad = w.N_pad; pa.n_groups = p->n_groups; pa.gpw = w.gpw;
    pa.n_weights = w.n_weights; pa.r = p->rank; pa.nkk = w.nkk; pa.kb32 = w.KB; pa.slots = w.slots;
    pa.max_chunks = w.max_chunks; pa.sw_stride = w.sw_stride; pa.tile_rows = w.tile_rows;
    pa.a_blocks = lora && !z_rows ? (uint32_t)(((uint64_t)p->n_groups * p->k * ((p->rank + 7u) / 8u) + 1023u) / 1024u) : 0u;
    pa.ap_blocks = lora ? bwd_ap_blocks(p->n_groups, w.KB, w.nkk) : 0u;
    pa.sw_blocks_per_weight = (w.N_pad + 1023u) / 1024u;
    // (the tables are filled slot by slot: a few workgroups, each with the prefix sums of its own)
    pa.route_blocks = (w.slots + 2047u) / 2048u < 16u ? (w.slots + 2047u) / 2048u : 16u;
    hipLaunchKernelGGL(bwd_grouped_prep_kernel,
                       dim3(pa.route_blocks + pa.a_blocks + pa.ap_blocks + pa.sw_blocks_per_weight * w.n_weights), dim3(1024), 0, s, pa);
    if ((st = launch_status())) return st;
  }
  BwdBody b{};
  b.m = p->m; b.k = p->k; b.n = p->n; b.n_groups = p->n_groups; b.rank = p->rank;
  b.x = p->x; b.dy = p->dy; b.w_packed = p->w_packed; b.lora_b = p->lora_b; b.lora_scaling = p->lora_scaling;
  b.dx = p->dx; b.d_lora_a = p->d_lora_a; b.d_lora_b = p->d_lora_b; b.d_lora_scaling = p->d_lora_scaling;
  b.lora = lora; b.want_grads = want_grads;
  b.src_row = tab.src_row; b.slot_group = tab.slot_group; b.blk_range = tab.blk_range; b.skip_range = tab.blk_range;
  b.x_row = tab.x_row; b.x_rows = x_rows; b.z_rows = z_rows;
  b.tile_weight = tab.tile_weight; b.chunk_tab = tab.chunk_tab; b.chunk0 = tab.chunk0;
  b.group_beg = tab.group_beg; b.group_end = tab.group_end;
  b.w_stride = (size_t)mi355_w8a8_packed_weight_bytes(p->k, p->n);
  b.sw_stride = w.sw_stride;
  b.rows128 = w.tile_rows == 128u;
  return launch_bwd_body(b, w, ws, s);
}

int run_qkv_post(const mi355_w8a8_qkv_post_problem* p, hipStream_t s) {
  if (!p) return MI355_W8A8_ERR_NULL;
  if (p->struct_size != sizeof(mi355_w8a8_qkv_post_problem)) return MI355_W8A8_ERR_STRUCT;
  if (p->flags & ~MI355_W8A8_FLAG_QKV_WEIGHTS_BF16) return MI355_W8A8_ERR_SHAPE;
  if (p->m == 0 || p->num_query_heads == 0 || p->num_kv_heads == 0 || p->head_dim == 0) return MI355_W8A8_ERR_SHAPE;
  if (p->num_query_heads % p->num_kv_heads) return MI355_W8A8_ERR_SHAPE;
  if ((p->head_dim & 1u) || (p->rotary_dim & 1u) || p->rotary_dim > p->head_dim) return MI355_W8A8_ERR_SHAPE;
  if (!(p->rope_theta > 0.0f) || !(p->rms_eps > 0.0f)) return MI355_W8A8_ERR_SHAPE;
  if (p->head_dim > kQkvMaxHeadDim || p->m > kMaxRows || p->num_query_heads > 1024u) return MI355_W8A8_ERR_UNSUPPORTED;
  const uint64_t width = ((uint64_t)p->num_query_heads * 2u + 2u * p->num_kv_heads) * p->head_dim;
  if (width * p->m >= (1ull << 32)) return MI355_W8A8_ERR_UNSUPPORTED;
  if (!p->fused || !p->q_norm_weight || !p->k_norm_weight || !p->positions || !p->q || !p->k || !p->v || !p->gate)
    return MI355_W8A8_ERR_NULL;
  if (!aligned16(p->fused) || !aligned16(p->q) || !aligned16(p->k) || !aligned16(p->v) || !aligned16(p->gate) ||
      !aligned16(p->q_norm_weight) || !aligned16(p->k_norm_weight) || (reinterpret_cast<uintptr_t>(p->positions) & 3u))
    return MI355_W8A8_ERR_ALIGN;
  const uint64_t fused_bytes = width * p->m * 2u;
  const uint64_t q_bytes = (uint64_t)p->m * p->num_query_heads * p->head_dim * 2u;
  const uint64_t kv_bytes = (uint64_t)p->m * p->num_kv_heads * p->head_dim * 2u;
  if (overlaps(p->fused, fused_bytes, p->q, q_bytes) || overlaps(p->fused, fused_bytes, p->gate, q_bytes) ||
      overlaps(p->fused, fused_bytes, p->k, kv_bytes) || overlaps(p->fused, fused_bytes, p->v, kv_bytes) ||
      overlaps(p->q, q_bytes, p->gate, q_bytes) || overlaps(p->k, kv_bytes, p->v, kv_bytes) ||
      overlaps(p->q, q_bytes, p->k, kv_bytes) || overlaps(p->q, q_bytes, p->v, kv_bytes) ||
      overlaps(p->gate, q_bytes, p->k, kv_bytes) || overlaps(p->gate, q_bytes, p->v, kv_bytes))
    return MI355_W8A8_ERR_ALIAS;
  QkvPostArgs a{};
  a.fused = static_cast<const uint16_t*>(p->fused);
  a.q_w = p->q_norm_weight; a.k_w = p->k_norm_weight; a.pos = p->positions;
  a.w_bf16 = p->flags & MI355_W8A8_FLAG_QKV_WEIGHTS_BF16 ? 1u : 0u;
  a.q = static_cast<uint16_t*>(p->q); a.k = static_cast<uint16_t*>(p->k);
  a.v = static_cast<uint16_t*>(p->v); a.gate = static_cast<uint16_t*>(p->gate);
  a.M = p->m; a.Hq = p->num_query_heads; a.Hkv = p->num_kv_heads; a.D = p->head_dim; a.rot = p->rotary_dim;
  a.width = (uint32_t)width; a.theta = p->rope_theta; a.eps = p->rms_eps;
  (void)hipGetLastError();
  if (p->head_dim <= 256u) hipLaunchKernelGGL((qkv_post_kernel<1>), dim3(p->m), dim3(256), 0, s, a);
  else hipLaunchKernelGGL((qkv_post_kernel<2>), dim3(p->m), dim3(256), 0, s, a);
  return launch_status();
}

// Workgroups of the QKV pull-back when the head-norm weights get cotangents: each leaves one partial.
inline uint32_t qkv_bwd_parts(uint32_t m) { return m < 1024u ? m : 1024u; }
inline uint64_t qkv_bwd_workspace_bytes(uint32_t m, uint32_t head_dim) {
  return (uint64_t)qkv_bwd_parts(m) * 2u * head_dim * 4u;
}

int run_qkv_post_bwd(const mi355_w8a8_qkv_post_bwd_problem* p, hipStream_t s) {
  if (!p) return MI355_W8A8_ERR_NULL;
  if (p->struct_size != sizeof(mi355_w8a8_qkv_post_bwd_problem)) return MI355_W8A8_ERR_STRUCT;
  if (p->flags & ~MI355_W8A8_FLAG_QKV_WEIGHTS_BF16) return MI355_W8A8_ERR_SHAPE;
  if (p->m == 0 || p->num_query_heads == 0 || p->num_kv_heads == 0 || p->head_dim == 0) return MI355_W8A8_ERR_SHAPE;
  if (p->num_query_heads % p->num_kv_heads) return MI355_W8A8_ERR_SHAPE;
  if ((p->head_dim & 1u) || (p->rotary_dim & 1u) || p->rotary_dim > p->head_dim) return MI355_W8A8_ERR_SHAPE;
  if (!(p->rope_theta > 0.0f) || !(p->rms_eps > 0.0f)) return MI355_W8A8_ERR_SHAPE;
  if (p->head_dim > kQkvMaxHeadDim || p->m > kMaxRows || p->num_query_heads > 1024u) return MI355_W8A8_ERR_UNSUPPORTED;
  const uint64_t width = ((uint64_t)p->num_query_heads * 2u + 2u * p->num_kv_heads) * p->head_dim;
  if (width * p->m >= (1ull << 32)) return MI355_W8A8_ERR_UNSUPPORTED;
  if (!p->fused || !p->q_norm_weight || !p->k_norm_weight || !p->positions || !p->d_q || !p->d_k || !p->d_v ||
      !p->d_gate || !p->d_fused)
    return MI355_W8A8_ERR_NULL;
  const bool wgrad = p->d_q_norm_weight != nullptr;
  if (wgrad != (p->d_k_norm_weight != nullptr)) return MI355_W8A8_ERR_NULL;
  if (!aligned16(p->fused) || !aligned16(p->d_q) || !aligned16(p->d_k) || !aligned16(p->d_v) || !aligned16(p->d_gate) ||
      !aligned16(p->d_fused) || !aligned16(p->q_norm_weight) || !aligned16(p->k_norm_weight) ||
      (reinterpret_cast<uintptr_t>(p->positions) & 3u))
    return MI355_W8A8_ERR_ALIGN;
  const uint64_t fused_bytes = width * p->m * 2u;
  const uint64_t q_bytes = (uint64_t)p->m * p->num_query_heads * p->head_dim * 2u;
  const uint64_t kv_bytes = (uint64_t)p->m * p->num_kv_heads * p->head_dim * 2u;
  if (overlaps(p->d_fused, fused_bytes, p->fused, fused_bytes) || overlaps(p->d_fused, fused_bytes, p->d_q, q_bytes) ||
      overlaps(p->d_fused, fused_bytes, p->d_gate, q_bytes) || overlaps(p->d_fused, fused_bytes, p->d_k, kv_bytes) ||
      overlaps(p->d_fused, fused_bytes, p->d_v, kv_bytes))
    return MI355_W8A8_ERR_ALIAS;
  const uint32_t parts = qkv_bwd_parts(p->m);
  if (wgrad) {
    const uint64_t need = qkv_bwd_workspace_bytes(p->m, p->head_dim);
    if (!p->workspace) return MI355_W8A8_ERR_NULL;
    if (p->workspace_bytes < need) return MI355_W8A8_ERR_WORKSPACE;
    if (!aligned16(p->workspace) || (reinterpret_cast<uintptr_t>(p->d_q_norm_weight) & 3u) ||
        (reinterpret_cast<uintptr_t>(p->d_k_norm_weight) & 3u))
      return MI355_W8A8_ERR_ALIGN;
    if (overlaps(p->workspace, need, p->d_fused, fused_bytes) || overlaps(p->workspace, need, p->fused, fused_bytes) ||
        overlaps(p->d_q_norm_weight, p->head_dim * 4ull, p->d_k_norm_weight, p->head_dim * 4ull))
      return MI355_W8A8_ERR_ALIAS;
  }
  QkvPostBwdArgs a{};
  a.fused = static_cast<const uint16_t*>(p->fused);
  a.q_w = p->q_norm_weight; a.k_w = p->k_norm_weight; a.pos = p->positions;
  a.w_bf16 = p->flags & MI355_W8A8_FLAG_QKV_WEIGHTS_BF16 ? 1u : 0u;
  a.dq = static_cast<const uint16_t*>(p->d_q); a.dk = static_cast<const uint16_t*>(p->d_k);
  a.dv = static_cast<const uint16_t*>(p->d_v); a.dgate = static_cast<const uint16_t*>(p->d_gate);
  a.dfused = static_cast<uint16_t*>(p->d_fused);
  a.partial = wgrad ? static_cast<float*>(p->workspace) : nullptr;
  a.M = p->m; a.Hq = p->num_query_heads; a.Hkv = p->num_kv_heads; a.D = p->head_dim; a.rot = p->rotary_dim;
  a.width = (uint32_t)width; a.theta = p->rope_theta; a.eps = p->rms_eps;
  const bool vec4 = (p->head_dim & 3u) == 0;
  (void)hipGetLastError();
  if (wgrad) {
    if (vec4 && p->head_dim <= 256u) hipLaunchKernelGGL((qkv_post_bwd_kernel<4, true, 1>), dim3(parts), dim3(256), 0, s, a);
    else if (vec4) hipLaunchKernelGGL((qkv_post_bwd_kernel<4, true>), dim3(parts), dim3(256), 0, s, a);
    else hipLaunchKernelGGL((qkv_post_bwd_kernel<1, true>), dim3(parts), dim3(256), 0, s, a);
    int st;
    if ((st = launch_status())) return st;
    ColumnSumArgs c{};
    c.partial = a.partial; c.n_parts = parts; c.stride = 2u * p->head_dim; c.cols = p->head_dim;
    c.out = p->d_q_norm_weight; c.col0 = 0;
    hipLaunchKernelGGL(column_sum_kernel, dim3((p->head_dim + 15u) / 16u), dim3(256), 0, s, c);
    c.out = p->d_k_norm_weight; c.col0 = p->head_dim;
    hipLaunchKernelGGL(column_sum_kernel, dim3((p->head_dim + 15u) / 16u), dim3(256), 0, s, c);
  } else {
    if (vec4 && p->head_dim <= 256u) hipLaunchKernelGGL((qkv_post_bwd_kernel<4, false, 1>), dim3(p->m), dim3(256), 0, s, a);
    else if (vec4) hipLaunchKernelGGL((qkv_post_bwd_kernel<4, false>), dim3(p->m), dim3(256), 0, s, a);
    else hipLaunchKernelGGL((qkv_post_bwd_kernel<1, false>), dim3(p->m), dim3(256), 0, s, a);
  }
  return launch_status();
}

// Row slices of the decoder-norm weight cotangent: each leaves one partial row.
inline uint32_t rms_dgamma_slices(uint32_t m) { return m < 256u ? m : 256u; }
inline uint64_t delta_rms_bwd_workspace_bytes(uint32_t m, uint32_t k) {
  return (uint64_t)round_up(m, 64u) * 4u + (uint64_t)rms_dgamma_slices(m) * k * 4u;
}

int run_delta_rms_norm_bwd(const void* x, const float* gamma, const void* d_normalized, void* d_x, float* d_gamma,
                           void* workspace, uint64_t workspace_bytes, uint32_t m, uint32_t k, float eps,
                           hipStream_t s) {
  if (!x || !gamma || !d_normalized || !d_x) return MI355_W8A8_ERR_NULL;
  if (m == 0 || k == 0 || !(eps > 0.0f)) return MI355_W8A8_ERR_SHAPE;
  if (m > kMaxRows) return MI355_W8A8_ERR_UNSUPPORTED;
  if (!aligned16(x) || !aligned16(d_normalized) || !aligned16(d_x) || !aligned16(gamma)) return MI355_W8A8_ERR_ALIGN;
  const uint64_t bytes = (uint64_t)m * k * 2u;
  if (overlaps(d_x, bytes, x, bytes) || overlaps(d_x, bytes, gamma, (uint64_t)k * 4u)) return MI355_W8A8_ERR_ALIAS;
  const uint64_t need = delta_rms_bwd_workspace_bytes(m, k);
  if (d_gamma) {
    // the weight cotangent reads d_normalized after the row pull-back has written d_x
    if (overlaps(d_x, bytes, d_normalized, bytes)) return MI355_W8A8_ERR_ALIAS;
    if (!workspace) return MI355_W8A8_ERR_NULL;
    if (workspace_bytes < need) return MI355_W8A8_ERR_WORKSPACE;
    if (!aligned16(workspace) || (reinterpret_cast<uintptr_t>(d_gamma) & 3u)) return MI355_W8A8_ERR_ALIGN;
    if (overlaps(workspace, need, d_x, bytes) || overlaps(workspace, need, x, bytes) ||
        overlaps(workspace, need, d_normalized, bytes) || overlaps(d_gamma, (uint64_t)k * 4u, d_x, bytes))
      return MI355_W8A8_ERR_ALIAS;
  } else if (d_x != d_normalized && overlaps(d_x, bytes, d_normalized, bytes)) {
    return MI355_W8A8_ERR_ALIAS;
  }
  DeltaRmsBwdArgs a{};
  a.x = static_cast<const uint16_t*>(x);
  a.gamma = gamma;
  a.dn = static_cast<const uint16_t*>(d_normalized);
  a.dx = static_cast<uint16_t*>(d_x);
  a.inv_out = d_gamma ? static_cast<float*>(workspace) : nullptr;
  a.M = m; a.K = k; a.eps = eps;
  (void)hipGetLastError();
  if ((k & 7u) == 0) hipLaunchKernelGGL((delta_rms_norm_bwd_kernel<true>), dim3(m), dim3(256), 0, s, a);
  else hipLaunchKernelGGL((delta_rms_norm_bwd_kernel<false>), dim3(m), dim3(256), 0, s, a);
  int st;
  if ((st = launch_status())) return st;
  if (d_gamma) {
    const uint32_t slices = rms_dgamma_slices(m);
    RmsDgammaArgs g{};
    g.x = a.x; g.dn = a.dn; g.inv = a.inv_out;
    g.partial = reinterpret_cast<float*>(static_cast<uint8_t*>(workspace) + (uint64_t)round_up(m, 64u) * 4u);
    g.M = m; g.K = k;
    hipLaunchKernelGGL(rms_dgamma_partial_kernel, dim3((k + 255u) / 256u, slices), dim3(256), 0, s, g);
    if ((st = launch_status())) return st;
    ColumnSumArgs c{};
    c.partial = g.partial; c.n_parts = slices; c.stride = k; c.cols = k; c.col0 = 0; c.out = d_gamma;
    hipLaunchKernelGGL(column_sum_kernel, dim3((k + 15u) / 16u), dim3(256), 0, s, c);
    return launch_status();
  }
  return MI355_W8A8_OK;
}

int run_swiglu_bwd(const void* fused, const void* d_product, void* d_fused, uint32_t m, uint32_t n, hipStream_t s) {
  if (!fused || !d_product || !d_fused) return MI355_W8A8_ERR_NULL;
  if (m == 0 || n == 0 || (n & 7u)) return MI355_W8A8_ERR_SHAPE;
  if (m > kMaxRows) return MI355_W8A8_ERR_UNSUPPORTED;
  if (!aligned16(fused) || !aligned16(d_fused) || (reinterpret_cast<uintptr_t>(d_product) & 7u))
    return MI355_W8A8_ERR_ALIGN;
  const uint64_t fused_bytes = (uint64_t)m * n * 2u;
  // d_fused may be fused itself (element i is read and written by the same thread), nothing else
  if (d_fused != fused && overlaps(d_fused, fused_bytes, fused, fused_bytes)) return MI355_W8A8_ERR_ALIAS;
  if (overlaps(d_fused, fused_bytes, d_product, fused_bytes / 2u)) return MI355_W8A8_ERR_ALIAS;
  SwigluBwdArgs a{};
  a.fused = static_cast<const uint16_t*>(fused);
  a.dprod = static_cast<const uint16_t*>(d_product);
  a.dfused = static_cast<uint16_t*>(d_fused);
  a.n_chunks = (uint64_t)m * n / 8u;
  const uint64_t blocks = (a.n_chunks + 255u) / 256u;
  (void)hipGetLastError();
  hipLaunchKernelGGL(swiglu_bwd_kernel, dim3((uint32_t)(blocks < 16384u ? blocks : 16384u)), dim3(256), 0, s, a);
  return launch_status();
}

int run_swiglu_fwd(const void* fused, void* product, uint32_t m, uint32_t n, hipStream_t s) {
  if (!fused || !product) return MI355_W8A8_ERR_NULL;
  if (m == 0 || n == 0 || (n & 7u)) return MI355_W8A8_ERR_SHAPE;
  if (m > kMaxRows) return MI355_W8A8_ERR_UNSUPPORTED;
  if (!aligned16(fused) || (reinterpret_cast<uintptr_t>(product) & 7u)) return MI355_W8A8_ERR_ALIGN;
  if (overlaps(product, (uint64_t)m * n, fused, (uint64_t)m * n * 2u)) return MI355_W8A8_ERR_ALIAS;
  SwigluFwdArgs a{};
  a.fused = static_cast<const uint16_t*>(fused);
  a.product = static_cast<uint16_t*>(product);
  a.n_chunks = (uint64_t)m * n / 8u;
  const uint64_t blocks = (a.n_chunks + 255u) / 256u;
  (void)hipGetLastError();
  hipLaunchKernelGGL(swiglu_fwd_kernel, dim3((uint32_t)(blocks < 16384u ? blocks : 16384u)), dim3(256), 0, s, a);
  return launch_status();
}

int run_rms_norm_bwd(const void* x, const float* gamma, const void* d_normalized, void* d_x, uint32_t m, uint32_t k,
                     float eps, hipStream_t s) {
  if (!x || !gamma || !d_normalized || !d_x) return MI355_W8A8_ERR_NULL;
  if (m == 0 || k == 0 || !(eps > 0.0f)) return MI355_W8A8_ERR_SHAPE;
  if (m > kMaxRows) return MI355_W8A8_ERR_UNSUPPORTED;
  if (!aligned16(x) || !aligned16(d_normalized) || !aligned16(d_x) || !aligned16(gamma)) return MI355_W8A8_ERR_ALIGN;
  const uint64_t bytes = (uint64_t)m * k * 2u;
  // d_x may be d_normalized itself (a row is reduced before any of it is rewritten, element i by
  // the thread that reads it), nothing else
  if (d_x != d_normalized && overlaps(d_x, bytes, d_normalized, bytes)) return MI355_W8A8_ERR_ALIAS;
  if (overlaps(d_x, bytes, x, bytes) || overlaps(d_x, bytes, gamma, (uint64_t)k * 4u)) return MI355_W8A8_ERR_ALIAS;
  RmsNormBwdArgs a{};
  a.x = static_cast<const uint16_t*>(x);
  a.gamma = gamma;
  a.dn = static_cast<const uint16_t*>(d_normalized);
  a.dx = static_cast<uint16_t*>(d_x);
  a.M = m; a.K = k; a.eps = eps;
  (void)hipGetLastError();
  if ((k & 7u) == 0) hipLaunchKernelGGL((rms_norm_bwd_kernel<true>), dim3(m), dim3(256), 0, s, a);
  else hipLaunchKernelGGL((rms_norm_bwd_kernel<false>), dim3(m), dim3(256), 0, s, a);
  return launch_status();
}


int run_moe_route(const float* logits, uint32_t t, uint32_t e, uint32_t top_k, uint32_t norm, float* weights,
                  int32_t* selected, hipStream_t s) {
  if (!logits || !weights || !selected) return MI355_W8A8_ERR_NULL;
  if (t == 0 || e == 0 || top_k == 0 || top_k > e || norm > 1u) return MI355_W8A8_ERR_SHAPE;
  if (e > kMoeMaxExperts || top_k > kMoeMaxTopK || t > kMaxRows) return MI355_W8A8_ERR_UNSUPPORTED;
  if ((reinterpret_cast<uintptr_t>(logits) | reinterpret_cast<uintptr_t>(weights) |
       reinterpret_cast<uintptr_t>(selected)) & 3u)
    return MI355_W8A8_ERR_ALIGN;
  const uint64_t out_bytes = (uint64_t)t * top_k * 4u;
  if (overlaps(weights, out_bytes, logits, (uint64_t)t * e * 4u) ||
      overlaps(selected, out_bytes, logits, (uint64_t)t * e * 4u) || overlaps(weights, out_bytes, selected, out_bytes))
    return MI355_W8A8_ERR_ALIAS;
  MoeRouteArgs a{};
  a.logits = logits; a.weights = weights; a.selected = selected;
  a.T = t; a.E = e; a.top_k = top_k; a.norm = norm;
  (void)hipGetLastError();
  const dim3 grid((t + 3u) / 4u), block(256);
  if (e <= 64u) hipLaunchKernelGGL((moe_route_kernel<1>), grid, block, 0, s, a);
  else if (e <= 128u) hipLaunchKernelGGL((moe_route_kernel<2>), grid, block, 0, s, a);
  else if (e <= 256u) hipLaunchKernelGGL((moe_route_kernel<4>), grid, block, 0, s, a);
  else if (e <= 512u) hipLaunchKernelGGL((moe_route_kernel<8>), grid, block, 0, s, a);
  else hipLaunchKernelGGL((moe_route_kernel<16>), grid, block, 0, s, a);
  return launch_status();
}

int run_moe_route_bwd(const float* logits, const int32_t* selected, const float* d_weights, uint32_t t, uint32_t e,
                      uint32_t top_k, uint32_t norm, float* d_logits, hipStream_t s) {
  if (!logits || !selected || !d_weights || !d_logits) return MI355_W8A8_ERR_NULL;
  if (t == 0 || e == 0 || top_k == 0 || top_k > e || norm > 1u) return MI355_W8A8_ERR_SHAPE;
  if (e > kMoeMaxExperts || top_k > kMoeMaxTopK || t > kMaxRows) return MI355_W8A8_ERR_UNSUPPORTED;
  if ((reinterpret_cast<uintptr_t>(logits) | reinterpret_cast<uintptr_t>(selected) |
       reinterpret_cast<uintptr_t>(d_weights) | reinterpret_cast<uintptr_t>(d_logits)) & 3u)
    return MI355_W8A8_ERR_ALIGN;
  const uint64_t tab_bytes = (uint64_t)t * top_k * 4u, row_bytes = (uint64_t)t * e * 4u;
  // d_logits may be the logits buffer itself (a token's row is read whole before it is rewritten), nothing else
  if (d_logits != logits && overlaps(d_logits, row_bytes, logits, row_bytes)) return MI355_W8A8_ERR_ALIAS;
  if (overlaps(d_logits, row_bytes, selected, tab_bytes) || overlaps(d_logits, row_bytes, d_weights, tab_bytes))
    return MI355_W8A8_ERR_ALIAS;
  MoeRouteBwdArgs a{};
  a.logits = logits; a.selected = selected; a.d_weights = d_weights; a.d_logits = d_logits;
  a.T = t; a.E = e; a.top_k = top_k; a.norm = norm;
  (void)hipGetLastError();
  const dim3 grid((t + 3u) / 4u), block(256);
  if (e <= 64u) hipLaunchKernelGGL((moe_route_bwd_kernel<1>), grid, block, 0, s, a);
  else if (e <= 128u) hipLaunchKernelGGL((moe_route_bwd_kernel<2>), grid, block, 0, s, a);
  else if (e <= 256u) hipLaunchKernelGGL((moe_route_bwd_kernel<4>), grid, block, 0, s, a);
  else if (e <= 512u) hipLaunchKernelGGL((moe_route_bwd_kernel<8>), grid, block, 0, s, a);
  else hipLaunchKernelGGL((moe_route_bwd_kernel<16>), grid, block, 0, s, a);
  return launch_status();
}

struct MoeSortLayout { uint64_t chunk_cnt, group_start, total; uint32_t n_chunks; };

MoeSortLayout make_moe_sort_layout(uint32_t n_pairs, uint32_t n_groups) {
  MoeSortLayout L{};
  L.n_chunks = (n_pairs + kMoeChunk - 1u) / kMoeChunk;
  L.chunk_cnt = 0;
  L.group_start = ((uint64_t)L.n_chunks * n_groups * 4u + 255u) & ~255ull;
  L.total = L.group_start + (((uint64_t)n_groups * 4u + 255u) & ~255ull);
  return L;
}

int validate_moe_sort_dims(uint32_t n_pairs, uint32_t n_groups) {
  if (n_pairs == 0 || n_groups == 0) return MI355_W8A8_ERR_SHAPE;
  if (n_groups > kMoeMaxExperts || n_pairs > (1u << 30)) return MI355_W8A8_ERR_UNSUPPORTED;
  return MI355_W8A8_OK;
}

int run_moe_dispatch(const mi355_w8a8_moe_dispatch_problem* p, hipStream_t s) {
  if (!p) return MI355_W8A8_ERR_NULL;
  if (p->struct_size != sizeof(mi355_w8a8_moe_dispatch_problem)) return MI355_W8A8_ERR_STRUCT;
  if (p->flags) return MI355_W8A8_ERR_SHAPE;
  int st = validate_moe_sort_dims(p->n_pairs, p->n_groups);
  if (st) return st;
  if (p->repeat == 0 || p->n_pairs % p->repeat) return MI355_W8A8_ERR_SHAPE;
  if (!p->indices || !p->group_sizes || !p->sort_indices || !p->unsort_indices) return MI355_W8A8_ERR_NULL;
  if ((p->adapter_indices != nullptr) != (p->sorted_adapters != nullptr)) return MI355_W8A8_ERR_NULL;
  if ((p->tokens != nullptr) != (p->sorted_tokens != nullptr)) return MI355_W8A8_ERR_NULL;
  if (p->tokens && (p->width == 0 || (p->width & 7u))) return MI355_W8A8_ERR_SHAPE;
  if (!aligned16(p->tokens) || !aligned16(p->sorted_tokens)) return MI355_W8A8_ERR_ALIGN;
  if ((reinterpret_cast<uintptr_t>(p->indices) | reinterpret_cast<uintptr_t>(p->group_sizes) |
       reinterpret_cast<uintptr_t>(p->sort_indices) | reinterpret_cast<uintptr_t>(p->unsort_indices) |
       reinterpret_cast<uintptr_t>(p->adapter_indices) | reinterpret_cast<uintptr_t>(p->sorted_adapters)) & 3u)
    return MI355_W8A8_ERR_ALIGN;
  const uint64_t idx_bytes = (uint64_t)p->n_pairs * 4u;
  if (p->tokens) {
    const uint64_t out_bytes = (uint64_t)p->n_pairs * p->width * 2u;
    if (overlaps(p->sorted_tokens, out_bytes, p->tokens, out_bytes / p->repeat) ||
        overlaps(p->sorted_tokens, out_bytes, p->indices, idx_bytes) ||
        overlaps(p->sorted_tokens, out_bytes, p->sort_indices, idx_bytes) ||
        overlaps(p->sorted_tokens, out_bytes, p->unsort_indices, idx_bytes))
      return MI355_W8A8_ERR_ALIAS;
  }
  if (overlaps(p->sort_indices, idx_bytes, p->indices, idx_bytes) ||
      overlaps(p->unsort_indices, idx_bytes, p->indices, idx_bytes) ||
      overlaps(p->sort_indices, idx_bytes, p->unsort_indices, idx_bytes))
    return MI355_W8A8_ERR_ALIAS;
  const MoeSortLayout L = make_moe_sort_layout(p->n_pairs, p->n_groups);
  if (!p->workspace || p->workspace_bytes < L.total) return MI355_W8A8_ERR_WORKSPACE;
  if (reinterpret_cast<uintptr_t>(p->workspace) & 255u) return MI355_W8A8_ERR_ALIGN;
  unsigned char* ws = static_cast<unsigned char*>(p->workspace);
  MoeSortArgs a{};
  a.indices = p->indices;
  a.tokens = static_cast<const uint16_t*>(p->tokens);
  a.adapters = p->adapter_indices;
  a.sorted_tokens = static_cast<uint16_t*>(p->sorted_tokens);
  a.group_sizes = p->group_sizes;
  a.sort_indices = p->sort_indices;
  a.unsort_indices = p->unsort_indices;
  a.sorted_adapters = p->sorted_adapters;
  a.chunk_cnt = reinterpret_cast<int32_t*>(ws + L.chunk_cnt);
  a.group_start = reinterpret_cast<int32_t*>(ws + L.group_start);
  a.P = p->n_pairs; a.G = p->n_groups; a.repeat = p->repeat; a.width = p->width; a.n_chunks = L.n_chunks;
  (void)hipGetLastError();
  if (L.n_chunks <= kMoeSortChunks) {
    hipLaunchKernelGGL(moe_sort_kernel, dim3(L.n_chunks), dim3(1024), 0, s, a);
  } else {
    hipLaunchKernelGGL(moe_hist_kernel, dim3(L.n_chunks), dim3(1024), 0, s, a);
    if ((st = launch_status())) return st;
    hipLaunchKernelGGL(moe_scan_kernel, dim3(1), dim3(1024), 0, s, a);
    if ((st = launch_status())) return st;
    hipLaunchKernelGGL(moe_scatter_kernel, dim3(L.n_chunks), dim3(1024), 0, s, a);
  }
  if ((st = launch_status()) || !a.tokens) return st;
  if (p->repeat > 1u)
    hipLaunchKernelGGL(moe_spread_kernel, dim3((p->n_pairs / p->repeat + 3u) / 4u), dim3(256), 0, s, a);
  else
    hipLaunchKernelGGL(moe_gather_kernel, dim3((p->n_pairs + 7u) / 8u), dim3(256), 0, s, a);
  return launch_status();
}

int run_moe_combine(const void* expert_out, const int32_t* unsort, const float* weights, void* out, uint32_t t,
                    uint32_t top_k, uint32_t width, hipStream_t s) {
  if (!expert_out || !unsort || !weights || !out) return MI355_W8A8_ERR_NULL;
  if (t == 0 || top_k == 0 || width == 0 || (width & 7u)) return MI355_W8A8_ERR_SHAPE;
  if (top_k > kMoeMaxTopK || t > kMaxRows || (uint64_t)t * top_k > (1ull << 30)) return MI355_W8A8_ERR_UNSUPPORTED;
  if (!aligned16(expert_out) || !aligned16(out)) return MI355_W8A8_ERR_ALIGN;
  if ((reinterpret_cast<uintptr_t>(unsort) | reinterpret_cast<uintptr_t>(weights)) & 3u) return MI355_W8A8_ERR_ALIGN;
  const uint64_t out_bytes = (uint64_t)t * width * 2u;
  if (overlaps(out, out_bytes, expert_out, out_bytes * top_k) || overlaps(out, out_bytes, unsort, (uint64_t)t * top_k * 4u) ||
      overlaps(out, out_bytes, weights, (uint64_t)t * top_k * 4u))
    return MI355_W8A8_ERR_ALIAS;
  MoeCombineArgs a{};
  a.expert_out = static_cast<const uint16_t*>(expert_out);
  a.unsort = unsort; a.weights = weights;
  a.out = static_cast<uint16_t*>(out);
  a.T = t; a.top_k = top_k; a.width = width;
  (void)hipGetLastError();
  hipLaunchKernelGGL(moe_combine_kernel, dim3(t), dim3(256), 0, s, a);
  return launch_status();
}

int run_moe_combine_bwd(const void* d_out, const void* expert_out, const int32_t* sort, const float* weights,
                        void* d_expert_out, float* d_weights, uint32_t t, uint32_t top_k, uint32_t width, hipStream_t s) {
  if (!d_out || !sort || !weights || !d_expert_out) return MI355_W8A8_ERR_NULL;
  if (d_weights && !expert_out) return MI355_W8A8_ERR_NULL;
  if (t == 0 || top_k == 0 || width == 0 || (width & 7u)) return MI355_W8A8_ERR_SHAPE;
  if (top_k > kMoeMaxTopK || t > kMaxRows || (uint64_t)t * top_k > (1ull << 30)) return MI355_W8A8_ERR_UNSUPPORTED;
  if (!aligned16(d_out) || !aligned16(expert_out) || !aligned16(d_expert_out)) return MI355_W8A8_ERR_ALIGN;
  if ((reinterpret_cast<uintptr_t>(sort) | reinterpret_cast<uintptr_t>(weights) | reinterpret_cast<uintptr_t>(d_weights)) & 3u)
    return MI355_W8A8_ERR_ALIGN;
  const uint64_t tok_bytes = (uint64_t)t * width * 2u, pair_bytes = tok_bytes * top_k, tab_bytes = (uint64_t)t * top_k * 4u;
  if (overlaps(d_expert_out, pair_bytes, d_out, tok_bytes) || overlaps(d_expert_out, pair_bytes, expert_out, pair_bytes) ||
      overlaps(d_expert_out, pair_bytes, sort, tab_bytes) || overlaps(d_expert_out, pair_bytes, weights, tab_bytes) ||
      overlaps(d_weights, tab_bytes, weights, tab_bytes) || overlaps(d_weights, tab_bytes, d_expert_out, pair_bytes) ||
      overlaps(d_weights, tab_bytes, sort, tab_bytes))
    return MI355_W8A8_ERR_ALIAS;
  MoeCombineBwdArgs a{};
  a.d_out = static_cast<const uint16_t*>(d_out);
  a.expert_out = d_weights ? static_cast<const uint16_t*>(expert_out) : nullptr;
  a.sort = sort; a.weights = weights;
  a.d_expert_out = static_cast<uint16_t*>(d_expert_out);
  a.d_weights = d_weights;
  a.P = t * top_k; a.top_k = top_k; a.width = width;
  (void)hipGetLastError();
  hipLaunchKernelGGL(moe_combine_bwd_kernel, dim3((a.P + 7u) / 8u), dim3(256), 0, s, a);
  return launch_status();
}

constexpr uint32_t kGqZSlices = 32;
// K slices of the routed LoRA-A projection: one workgroup per 32-row block and slice, so that calls with
// fewer row blocks than the chip has CUs still fill it (the consumer adds the slices in order)
inline uint32_t gq_z_ksplit(uint32_t m_pad, uint32_t k) {
  const uint32_t n_blocks = m_pad / 32u, n_steps = (k + 63u) / 64u;
  uint32_t ks = n_blocks >= 192u ? 1u : (256u + n_blocks - 1u) / n_blocks;
  if (ks > 4u) ks = 4u;
  while (ks > 1u && n_steps / ks < 16u) --ks;  // every wave of a slice keeps at least one step
  return ks;
}
struct GqLayout { uint64_t codes, scales, z, src_row, dst_pos, slot_group, blk_range, at, total; uint32_t m_pad, G; };

GqLayout make_gq_layout(uint32_t m, uint32_t k_pad, uint32_t group, uint32_t n_adapters, uint32_t rank) {
  GqLayout L{};
  L.m_pad = round_up(m, 32u);
  L.G = k_pad / group;
  uint64_t off = 0;
  L.codes = off; off += align256((uint64_t)L.m_pad * k_pad);
  L.scales = off; off += align256((uint64_t)L.m_pad * L.G * 4u);
  // decode (one row block): LoRA-A arrives as up to kGqZSlices slices over K
  L.z = off; off += rank ? align256((uint64_t)L.m_pad * 64u * 4u * (L.m_pad == 32u ? kGqZSlices : 4u)) : 0u;
  L.src_row = off; off += rank ? align256((uint64_t)L.m_pad * 4u) : 0u;
  L.dst_pos = off; off += rank ? align256((uint64_t)L.m_pad * 4u) : 0u;
  L.slot_group = off; off += rank ? align256((uint64_t)L.m_pad * 4u) : 0u;
  L.blk_range = off; off += rank ? align256((uint64_t)(L.m_pad / 32u) * 4u) : 0u;
  // LoRA A in lora_a_kernel's operand order: per adapter and 64-wide k step 4 KiB per 32 rank columns
  L.at = off; off += (rank && n_adapters <= (uint32_t)kMaxAdapters)
                         ? align256((uint64_t)n_adapters * ((k_pad + 63u) / 64u) * (rank_chunks(rank) > 2u ? 2u : 1u) * 4u * kBlockBytes)
                         : 0u;
  L.total = off;
  return L;
}

int validate_gq_dims(uint32_t m, uint32_t k_pad, uint32_t group, uint32_t rank) {
  if (m == 0 || k_pad == 0 || group == 0) return MI355_W8A8_ERR_SHAPE;
  if ((group & 31u) || k_pad % group) return MI355_W8A8_ERR_UNSUPPORTED;
  if (m > kMaxRows || k_pad > kMaxK || rank > (uint32_t)kMaxRank) return MI355_W8A8_ERR_UNSUPPORTED;
  return MI355_W8A8_OK;
}

int run_gq_pack(const void* codes, void* packed, uint32_t k_pad, uint32_t n, uint32_t bits, hipStream_t s) {
  if (!codes || !packed) return MI355_W8A8_ERR_NULL;
  if (k_pad == 0 || n == 0 || (bits != 4u && bits != 8u)) return MI355_W8A8_ERR_SHAPE;
  if ((k_pad & 31u) || k_pad > kMaxK || n > kMaxN) return MI355_W8A8_ERR_UNSUPPORTED;
  if (!aligned16(packed)) return MI355_W8A8_ERR_ALIGN;
  const uint64_t src_bytes = (uint64_t)k_pad * n / (bits == 4u ? 2u : 1u);
  if (overlaps(packed, gq_packed_bytes(k_pad, n, bits), codes, src_bytes)) return MI355_W8A8_ERR_ALIAS;
  GqPackArgs a{};
  a.codes = static_cast<const unsigned char*>(codes);
  a.packed = static_cast<unsigned char*>(packed);
  a.k_pad = k_pad; a.n = n; a.bits = bits;
  a.n_items = (uint64_t)((n + 31u) / 32u) * (k_pad / 32u) * 64u;
  (void)hipGetLastError();
  hipLaunchKernelGGL(gq_pack_weight_kernel, dim3((uint32_t)((a.n_items + 255u) / 256u)), dim3(256), 0, s, a);
  return launch_status();
}

// Whether the staged group-scaled product of 8-bit codes in groups beyond kGqSmallGroup takes 128 x 128 tiles (512 places) instead of
// 64 x 128 (1024): with little scaling between the MFMAs the operands' way from the L2 counts, 17 KiB a stage for twice
// the outputs instead of 13, and a long K repays the taller tile's longer fill and end.  Where the places of a first round are nearly all taken,
// or beyond one and a half.  Whole call, 64 x 128 / 128 x 128, one adapter of rank 32: 12288 -> 4096, groups of 1024: 1536 rows (768 tiles of 64 x 128) 141 us / 138,
// 2048 180 / 163, 2560 228 / 251, 3072 269 / 267, 4096 338 / 307, 8192 686 / 629, groups of 512 347 / 322 and 697 / 651; 12288 -> 2560, 3072 rows
// (960) 200 / 181, 4096 (1280) 247 / 267; 8192 -> 2048, 4096 rows 153 / 143; 6144 -> 4096, 4096 rows 184 / 173; 4096 -> 12288, groups of 512, 3072 rows
// 262 / 272; 2048 -> 8192, 4096 rows 137 / 145.  Groups of 256 7 % better at 12288 and 1 to 5 % worse at 4096 and below, of 128 level or worse.
constexpr uint32_t kGqTallMinK = 6144u;
inline bool gq_tall_tiles_pay(uint32_t m, uint32_t k_pad, uint32_t n) {
  const uint64_t tiles = (uint64_t)((m + 63u) / 64u) * ((n + kGqTileCols - 1u) / kGqTileCols);
  return k_pad >= kGqTallMinK && ((tiles > 896u && tiles <= 1024u) || tiles > 1600u);
}

int run_gq_linear(const mi355_w8a8_gq_problem* p, hipStream_t s) {
  if (!p) return MI355_W8A8_ERR_NULL;
  if (p->struct_size != sizeof(mi355_w8a8_gq_problem)) return MI355_W8A8_ERR_STRUCT;
  if (p->flags & ~MI355_W8A8_FLAG_GQ_DIRECT) return MI355_W8A8_ERR_SHAPE;
  int st = validate_gq_dims(p->m, p->k_pad, p->group_size, p->rank);
  if (st) return st;
  if (p->n == 0 || p->k == 0 || p->k > p->k_pad) return MI355_W8A8_ERR_SHAPE;
  if ((p->weight_bits != 4u && p->weight_bits != 8u) || (p->activation_bits != 4u && p->activation_bits != 8u))
    return MI355_W8A8_ERR_SHAPE;
  if (p->n > kMaxN || (uint64_t)p->m * p->n >= (1ull << 32)) return MI355_W8A8_ERR_UNSUPPORTED;
  if (!p->x || !p->w_packed || !p->w_scales || !p->out) return MI355_W8A8_ERR_NULL;
  const bool lora = p->n_adapters > 0;
  if (lora) {
    if (!p->lora_a || !p->lora_b || !p->lora_scaling) return MI355_W8A8_ERR_NULL;
    if (p->rank == 0 || p->n_adapters > (uint32_t)kMaxGroups) return MI355_W8A8_ERR_UNSUPPORTED;
  } else if (p->adapter_indices) {
    return MI355_W8A8_ERR_SHAPE;
  }
  if (!aligned16(p->w_packed) || (reinterpret_cast<uintptr_t>(p->x) & 1u) || (reinterpret_cast<uintptr_t>(p->out) & 1u) ||
      (reinterpret_cast<uintptr_t>(p->w_scales) & 3u) || (reinterpret_cast<uintptr_t>(p->adapter_indices) & 3u))
    return MI355_W8A8_ERR_ALIGN;
  const uint64_t out_bytes = (uint64_t)p->m * p->n * 2u;
  if (overlaps(p->out, out_bytes, p->x, (uint64_t)p->m * p->k * 2u) ||
      overlaps(p->out, out_bytes, p->w_packed, gq_packed_bytes(p->k_pad, p->n, p->weight_bits)) ||
      overlaps(p->out, out_bytes, p->workspace, p->workspace_bytes))
    return MI355_W8A8_ERR_ALIAS;
  const GqLayout L = make_gq_layout(p->m, p->k_pad, p->group_size, p->n_adapters, lora ? p->rank : 0u);
  if (!p->workspace || p->workspace_bytes < L.total) return MI355_W8A8_ERR_WORKSPACE;
  if (reinterpret_cast<uintptr_t>(p->workspace) & 255u) return MI355_W8A8_ERR_ALIGN;
  unsigned char* ws = static_cast<unsigned char*>(p->workspace);
  (void)hipGetLastError();

  GqQuantArgs q{};
  q.x = static_cast<const uint16_t*>(p->x);
  q.codes = reinterpret_cast<int8_t*>(ws + L.codes);
  q.scales = reinterpret_cast<float*>(ws + L.scales);
  q.codes_rm = p->aux_x_codes; q.scales_rm = p->aux_x_scales;
  q.M = p->m; q.M_pad = L.m_pad; q.K = p->k; q.K_pad = p->k_pad; q.group = p->group_size; q.G = L.G;
  q.qmax = p->activation_bits == 4u ? 7.0f : 127.0f;
  // gq_quant_kernel (groups that gq_quant_tile_kernel does not take, and decode): a row's groups are dealt to several
  // waves, with few rows so that the launch fills the chip (2816 waves), with many so that a wave that waits for its 3072
  // values has others beside it.  More waves than that only find less to do each.
  uint32_t q_slices = 2816u / L.m_pad;
  if (q_slices < (p->k + 3071u) / 3072u) q_slices = (p->k + 3071u) / 3072u;
  if (q_slices > 16u) q_slices = 16u;
  if (q_slices > L.G) q_slices = L.G;
  q.groups_per_slice = (L.G + q_slices - 1u) / q_slices;
  const uint32_t q_grid_y = (L.G + q.groups_per_slice - 1u) / q.groups_per_slice;
  const bool decode = L.m_pad == 32u;  // few rows: z in K slices instead of row blocks
  // one adapter's z shares the quantizer's launch (rows of 16-byte pieces; several adapters: a wave per row)
  const bool decode_z = decode && p->n_adapters == 1u && (p->k & 7u) == 0 && aligned16(p->x);
  // z = x @ A[idx]: rows routed by adapter and multiplied on the matrix core (the kernels of the
  // per-channel path) when the adapter count and K allow it, else one wave per row
  const bool fast_z = lora && !decode && p->n_adapters <= (uint32_t)kMaxAdapters && (p->k & 7u) == 0 &&
                      aligned16(p->x) && aligned16(p->lora_a);
  const bool routed = fast_z && p->adapter_indices && p->n_adapters > 1u;
  // A in lora_a_kernel's operand order
  const uint32_t a_steps = (p->k + 63u) / 64u, a_rb = rank_chunks(p->rank) > 2u ? 2u : 1u;
  const uint64_t a_items = (uint64_t)p->n_adapters * a_steps * a_rb * 256u;
  uint16_t* const at = reinterpret_cast<uint16_t*>(ws + L.at);
  // the quantizer's launch packs it where there is no routing launch to do it beside
  const bool quant_tiles = !decode && (p->k & 7u) == 0 && (p->group_size == 32u || p->group_size == 64u || p->group_size == 128u);
  const bool quant_packs = quant_tiles && fast_z && !routed;
  if (!decode_z) {
    if (quant_tiles) {
      const uint32_t halves = L.m_pad / 16u;
      GqQuantTileArgs t{};
      t.q = q;
      if (quant_packs) {
        t.lora_a = static_cast<const uint16_t*>(p->lora_a); t.at = at;
        t.n_groups = p->n_adapters; t.r = p->rank; t.steps = a_steps; t.rb = a_rb;
        t.pack_y = (uint32_t)((a_items / 256u + halves - 1u) / halves);
      }
      const dim3 qgrid(halves, t.pack_y + (p->k_pad + 511u) / 512u);
      if (p->group_size == 32u) hipLaunchKernelGGL((gq_quant_tile_kernel<1>), qgrid, dim3(256), 0, s, t);
      else if (p->group_size == 64u) hipLaunchKernelGGL((gq_quant_tile_kernel<2>), qgrid, dim3(256), 0, s, t);
      else hipLaunchKernelGGL((gq_quant_tile_kernel<4>), qgrid, dim3(256), 0, s, t);
    } else {
      hipLaunchKernelGGL(gq_quant_kernel, dim3(L.m_pad / 4u, q_grid_y), dim3(256), 0, s, q);
    }
    if ((st = launch_status())) return st;
  }

  int32_t* dst_pos = reinterpret_cast<int32_t*>(ws + L.dst_pos);
  uint32_t z_slices = 1u, z_slice_stride = p->m * 64u;
  if (fast_z) {
    int32_t* src_row = reinterpret_cast<int32_t*>(ws + L.src_row);
    int32_t* slot_group = reinterpret_cast<int32_t*>(ws + L.slot_group);
    int32_t* blk_range = reinterpret_cast<int32_t*>(ws + L.blk_range);
    LoraPrepArgs pa{};
    pa.idx = routed ? p->adapter_indices : nullptr;
    pa.src_row = src_row; pa.dst_pos = dst_pos; pa.slot_group = slot_group; pa.blk_range = blk_range;
    pa.lora_a = static_cast<const uint16_t*>(p->lora_a);
    pa.at = at;
    pa.M = p->m; pa.K = p->k; pa.N = p->n; pa.n_groups = p->n_adapters; pa.r = p->rank;
    pa.slots = L.m_pad;
    pa.route_blocks = routed ? 1u : 0u;
    pa.a_operand_steps = a_steps; pa.a_operand_rb = a_rb;
    pa.a_blocks = (uint32_t)((a_items + 1023u) / 1024u);
    if (!quant_packs) {
      hipLaunchKernelGGL((lora_prep_kernel<0>), dim3(pa.route_blocks + pa.a_blocks), dim3(1024), 0, s, pa);
      if ((st = launch_status())) return st;
    }
    LoraAArgs la{};
    la.xsrc = q.x;
    la.at = at;
    la.at_operand = 1u;
    la.src_row = routed ? src_row : nullptr;
    la.slot_group = routed ? slot_group : nullptr;
    la.blk_range = routed ? blk_range : nullptr;
    la.zf = reinterpret_cast<float*>(ws + L.z);
    la.zf_stride = 64u;
    la.M = p->m; la.K = p->k; la.r = p->rank;
    const uint32_t nks = gq_z_ksplit(L.m_pad, p->k);
    la.n_steps = (p->k + 63u) / 64u; la.steps_per_wave = ((la.n_steps + nks - 1u) / nks + 15u) / 16u;
    la.n_ksplit = nks; la.zf_slice = L.m_pad * 64u;
    z_slices = nks; z_slice_stride = L.m_pad * 64u;
    la.n_blocks = L.m_pad / 32u;
    const dim3 zgrid(L.m_pad / 32u * nks);
    if ((st = launch_lora_a(la, rank_chunks(p->rank), zgrid, s))) return st;
  } else if (lora) {
    GqLoraZArgs z{};
    z.x = q.x;
    z.lora_a = static_cast<const uint16_t*>(p->lora_a);
    z.idx = p->adapter_indices;
    z.z = reinterpret_cast<float*>(ws + L.z);
    z.M = p->m; z.K = p->k; z.r = p->rank; z.n_adapters = p->n_adapters;
    const uint32_t most = decode_z ? kGqDecodeZSlices : kGqZSlices, per = decode_z ? kGqDecodeZChunk : 256u;
    z.k_split = decode ? (p->k + per - 1u) / per : 1u;
    if (z.k_split > most) z.k_split = most;
    z.k_chunk = round_up((p->k + z.k_split - 1u) / z.k_split, decode_z ? 128u : 64u);
    z_slices = z.k_split;
    if (decode_z) {
      GqDecodePrologueArgs d{};
      d.q = q; d.z = z;
      d.z_units = z.k_split * ((p->rank + 15u) / 16u) * ((p->m + 15u) / 16u);
      d.row_quads = L.m_pad / 4u;
      hipLaunchKernelGGL(gq_decode_prologue_kernel, dim3(d.z_units + d.row_quads * q_grid_y), dim3(256), 0, s, d);
    } else {
      const dim3 zgrid((p->m + 3u) / 4u, z.k_split), zblock(256);
      if (p->rank <= 8u) hipLaunchKernelGGL((gq_lora_z_kernel<1>), zgrid, zblock, 0, s, z);
      else if (p->rank <= 16u) hipLaunchKernelGGL((gq_lora_z_kernel<2>), zgrid, zblock, 0, s, z);
      else if (p->rank <= 32u) hipLaunchKernelGGL((gq_lora_z_kernel<4>), zgrid, zblock, 0, s, z);
      else hipLaunchKernelGGL((gq_lora_z_kernel<8>), zgrid, zblock, 0, s, z);
    }
    if ((st = launch_status())) return st;
  }

  GqGemmArgs g{};
  g.codes = q.codes; g.xs = q.scales;
  g.wp = static_cast<const unsigned char*>(p->w_packed);
  g.ws = p->w_scales;
  g.z = lora ? reinterpret_cast<const float*>(ws + L.z) : nullptr;
  g.z_slot = routed ? dst_pos : nullptr;
  g.z_slices = z_slices; g.z_slice_stride = z_slice_stride;
  g.lora_b = static_cast<const uint16_t*>(p->lora_b);
  g.lora_scaling = p->lora_scaling;
  g.idx = p->adapter_indices;
  g.out = static_cast<uint16_t*>(p->out);
  g.aux_base = p->aux_base;
  g.M = p->m; g.M_pad = L.m_pad; g.N = p->n; g.K_pad = p->k_pad; g.group = p->group_size; g.G = L.G;
  g.bits = p->weight_bits;
  g.r = p->rank; g.n_adapters = p->n_adapters;
  g.n_col_blocks = (p->n + 31u) / 32u;
  if (decode && p->group_size % 64u == 0) {  // the groups split over the waves of a workgroup per 16 columns
    const dim3 sgrid((p->n + 15u) / 16u), sblock(1024);
    if (p->weight_bits == 4u) {
      if (p->m <= 16u) hipLaunchKernelGGL((gq_stream_kernel<true, 1>), sgrid, sblock, 0, s, g);
      else hipLaunchKernelGGL((gq_stream_kernel<true, 2>), sgrid, sblock, 0, s, g);
    } else {
      if (p->m <= 16u) hipLaunchKernelGGL((gq_stream_kernel<false, 1>), sgrid, sblock, 0, s, g);
      else hipLaunchKernelGGL((gq_stream_kernel<false, 2>), sgrid, sblock, 0, s, g);
    }
    return launch_status();
  }
  if (decode) {  // groups that are no multiple of 64: per 32-column block
    const dim3 sgrid(g.n_col_blocks), sblock(kGqSkinnyWaves * 64u);
    if (p->weight_bits == 4u) hipLaunchKernelGGL((gq_skinny_kernel<true>), sgrid, sblock, 0, s, g);
    else hipLaunchKernelGGL((gq_skinny_kernel<false>), sgrid, sblock, 0, s, g);
    return launch_status();
  }
  if (p->group_size % 64u == 0 && !(p->flags & MI355_W8A8_FLAG_GQ_DIRECT)) {
    // groups of whole 64-wide k steps: tiles of 64 or 128 rows x 128 columns staged through the LDS
    const bool w4 = p->weight_bits == 4u, small = p->group_size <= kGqSmallGroup;
    const bool tall = !w4 && !small && gq_tall_tiles_pay(p->m, p->k_pad, p->n);
    const uint32_t rb = tall ? 4u : 2u;
    const dim3 grid((p->n + kGqTileCols - 1u) / kGqTileCols, (L.m_pad + rb * 32u - 1u) / (rb * 32u)), block(256);
    const auto kernel = tall ? &gq_gemm_lds_kernel<false, false, 4>
                        : w4 ? (small ? &gq_gemm_lds_kernel<true, true, 2> : &gq_gemm_lds_kernel<true, false, 2>)
                             : (small ? &gq_gemm_lds_kernel<false, true, 2> : &gq_gemm_lds_kernel<false, false, 2>);
    const uint32_t lds_bytes = gq_lds_bytes(w4, rb);
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes) != hipSuccess)
      return MI355_W8A8_ERR_LAUNCH;
    hipLaunchKernelGGL(kernel, grid, block, lds_bytes, s, g);
    return launch_status();
  }
  const dim3 grid((g.n_col_blocks + 7u) / 8u, (L.m_pad / 32u + 1u) / 2u), block(256);
  if (p->weight_bits == 4u) hipLaunchKernelGGL((gq_gemm_kernel<true>), grid, block, 0, s, g);
  else hipLaunchKernelGGL((gq_gemm_kernel<false>), grid, block, 0, s, g);
  return launch_status();
}

}  // namespace

extern "C" {

int mi355_w8a8_abi_version(void) { return MI355_W8A8_ABI_VERSION; }

const char* mi355_w8a8_status_string(int status) {
  switch (status) {
    case MI355_W8A8_OK: return "ok";
    case MI355_W8A8_ERR_NULL: return "a required pointer is NULL";
    case MI355_W8A8_ERR_SHAPE: return "a dimension or flag combination is invalid";
    case MI355_W8A8_ERR_ALIGN: return "a pointer is not sufficiently aligned";
    case MI355_W8A8_ERR_ALIAS: return "the output overlaps an input or the workspace";
    case MI355_W8A8_ERR_WORKSPACE: return "workspace missing or too small";
    case MI355_W8A8_ERR_LAUNCH: return "the HIP runtime refused a launch";
    case MI355_W8A8_ERR_UNSUPPORTED: return "request outside the supported geometry";
    case MI355_W8A8_ERR_STRUCT: return "struct_size does not match this library";
    default: return "unknown status";
  }
}

uint64_t mi355_w8a8_packed_weight_bytes(uint32_t k, uint32_t n) {
  if (k == 0 || n == 0) return 0;
  return (uint64_t)k_padded(k) * n_padded(n);
}

int mi355_w8a8_pack_weight_v1(const int8_t* codes_kn, void* packed, uint32_t k, uint32_t n, void* stream) {
  if (!codes_kn || !packed) return MI355_W8A8_ERR_NULL;
  if (k == 0 || n == 0) return MI355_W8A8_ERR_SHAPE;
  if (n > kMaxN || k > (1u << 20)) return MI355_W8A8_ERR_UNSUPPORTED;
  if (!aligned16(packed)) return MI355_W8A8_ERR_ALIGN;
  const uint64_t bytes = mi355_w8a8_packed_weight_bytes(k, n);
  if (overlaps(codes_kn, (uint64_t)k * n, packed, bytes)) return MI355_W8A8_ERR_ALIAS;
  const uint64_t chunks = bytes / 16u;
  (void)hipGetLastError();
  hipLaunchKernelGGL(pack_weight_kernel, dim3((uint32_t)((chunks + 255u) / 256u)), dim3(256), 0,
                     static_cast<hipStream_t>(stream), codes_kn, static_cast<unsigned char*>(packed), k, n,
                     k_padded(k) / 32u, chunks);
  return launch_status();
}

int mi355_w8a8_unpack_weight_v1(const void* packed, int8_t* codes_kn, uint32_t k, uint32_t n, void* stream) {
  if (!codes_kn || !packed) return MI355_W8A8_ERR_NULL;
  if (k == 0 || n == 0) return MI355_W8A8_ERR_SHAPE;
  if (n > kMaxN || k > (1u << 20)) return MI355_W8A8_ERR_UNSUPPORTED;
  if (overlaps(codes_kn, (uint64_t)k * n, packed, mi355_w8a8_packed_weight_bytes(k, n)))
    return MI355_W8A8_ERR_ALIAS;
  const uint64_t total = (uint64_t)k * n;
  (void)hipGetLastError();
  hipLaunchKernelGGL(unpack_weight_kernel, dim3((uint32_t)((total + 255u) / 256u)), dim3(256), 0,
                     static_cast<hipStream_t>(stream), static_cast<const unsigned char*>(packed), codes_kn, k, n,
                     k_padded(k) / 32u);
  return launch_status();
}

int mi355_w8a8_quantize_rows_v1(const void* x_bf16, int8_t* codes, float* scales, uint32_t m, uint32_t k,
                                void* stream) {
  if (!x_bf16 || !codes || !scales) return MI355_W8A8_ERR_NULL;
  int st = validate_common(m, k, 1);
  if (st) return st;
  if (!aligned16(x_bf16) || (reinterpret_cast<uintptr_t>(codes) & 7u) || (reinterpret_cast<uintptr_t>(scales) & 3u))
    return MI355_W8A8_ERR_ALIGN;
  if (overlaps(x_bf16, (uint64_t)m * k * 2u, codes, (uint64_t)m * k) ||
      overlaps(x_bf16, (uint64_t)m * k * 2u, scales, (uint64_t)m * 4u) ||
      overlaps(codes, (uint64_t)m * k, scales, (uint64_t)m * 4u))
    return MI355_W8A8_ERR_ALIAS;
  QuantArgs q{};
  q.x = static_cast<const uint16_t*>(x_bf16);
  q.M = m; q.K = k;
  q.codes_rm = codes;
  q.scales_rm = scales;
  (void)hipGetLastError();
  return launch_quant(q, static_cast<hipStream_t>(stream));
}

uint64_t mi355_w8a8_workspace_bytes(uint32_t m, uint32_t k, uint32_t n, uint32_t n_adapters, uint32_t rank,
                                    uint32_t flags) {
  if (validate_common(m, k, n)) return 0;
  if (n_adapters > (uint32_t)kMaxAdapters || rank > (uint32_t)kMaxRank) return 0;
  // (sized for groups on block boundaries wherever a call of these dimensions may lay them out so)
  const bool keep_b = (flags & (MI355_W8A8_FLAG_DECODE_B_WRITE | MI355_W8A8_FLAG_DECODE_B_KEPT)) && n_adapters &&
                      skinny_b_can_be_kept(m, n, rank, (flags & MI355_W8A8_FLAG_SWIGLU) != 0);
  return make_layout(m, k, n, n_adapters, n_adapters ? rank : 0u, n_adapters > 1,
                     padded_groups_fit(m, n, n_adapters) || padded_groups_fit(m, n, n_adapters, true), keep_b).total;
}

int mi355_w8a8_lora_linear_v1(const mi355_w8a8_problem* p, void* stream) {
  return run_forward(p, static_cast<hipStream_t>(stream), kReqLinear);
}
int mi355_w8a8_rms_gateup_swiglu_v1(const mi355_w8a8_problem* p, void* stream) {
  return run_forward(p, static_cast<hipStream_t>(stream), kReqGateUp);
}
int mi355_w8a8_lora_residual_v1(const mi355_w8a8_problem* p, void* stream) {
  return run_forward(p, static_cast<hipStream_t>(stream), kReqResidual);
}
int mi355_w8a8_forward_keeps_z(uint32_t m, uint32_t k, uint32_t n, uint32_t n_adapters, uint32_t rank, uint32_t flags) {
  return forward_keeps_z(m, k, n, n_adapters, rank, flags) ? 1 : 0;
}
int mi355_w8a8_forward_v1(const mi355_w8a8_problem* p, void* stream) {
  return run_forward(p, static_cast<hipStream_t>(stream), kReqNone);
}

int mi355_w8a8_forward_static_ws_v1(const mi355_w8a8_problem* p, void* stream) {
  if (!p) return MI355_W8A8_ERR_NULL;
  if (p->struct_size != sizeof(mi355_w8a8_problem)) return MI355_W8A8_ERR_STRUCT;
  const int st = validate_common(p->m, p->k, p->n);
  if (st) return st;
  // Every caller in the process shares the array: what an earlier call left in it may be another layer's,
  // so a call must not be told to keep it.
  if (p->flags & (MI355_W8A8_FLAG_LORA_PACK_VALID | MI355_W8A8_FLAG_SKIP_PROLOGUE | MI355_W8A8_FLAG_DECODE_B_KEPT))
    return MI355_W8A8_ERR_UNSUPPORTED;
  const uint64_t full = mi355_w8a8_workspace_bytes(p->m, p->k, p->n, p->n_adapters, p->rank, p->flags);
  const uint64_t need = full ? full - split_z_bytes(p->m, p->n, p->n_adapters, p->n_adapters ? p->rank : 0u) : 0u;
  if (need == 0 || need > MI355_W8A8_STATIC_WORKSPACE_BYTES) return MI355_W8A8_ERR_WORKSPACE;
  void* ws = static_workspace();
  if (!ws) return MI355_W8A8_ERR_LAUNCH;
  // Nothing in the workspace has to start at zero: every table a kernel reads is written by an earlier
  // kernel of the same call (the tile counters are cleared by the quantizer launch), so the contents a
  // previous call left behind are never read.
  mi355_w8a8_problem q = *p;
  q.workspace = ws;
  q.workspace_bytes = MI355_W8A8_STATIC_WORKSPACE_BYTES;
  return run_forward(&q, static_cast<hipStream_t>(stream), kReqNone);
}

uint64_t mi355_w8a8_grouped_workspace_bytes(uint32_t m, uint32_t k, uint32_t n, uint32_t n_groups, uint32_t rank,
                                            uint32_t flags) {
  if (validate_common(m, k, n)) return 0;
  if (n_groups == 0 || n_groups > (uint32_t)kMaxGroups || rank > (uint32_t)kMaxRank) return 0;
  return make_grouped_layout(m, k, n, n_groups, rank, flags).total;
}

int mi355_w8a8_grouped_v1(const mi355_w8a8_grouped_problem* p, void* stream) {
  return run_grouped(p, static_cast<hipStream_t>(stream));
}

uint64_t mi355_w8a8_bwd_workspace_bytes(uint32_t m, uint32_t k, uint32_t n, uint32_t n_adapters, uint32_t rank,
                                        uint32_t flags) {
  (void)flags;
  if (validate_bwd_dims(m, k, n, n_adapters, rank)) return 0;
  return make_bwd_layout(m, k, n, n_adapters, n_adapters ? rank : 0u).total;
}

int mi355_w8a8_lora_linear_bwd_v1(const mi355_w8a8_bwd_problem* p, void* stream) {
  return run_backward(p, static_cast<hipStream_t>(stream));
}

uint64_t mi355_w8a8_grouped_bwd_workspace_bytes(uint32_t m, uint32_t k, uint32_t n, uint32_t n_groups, uint32_t rank,
                                                uint32_t groups_per_weight) {
  if (validate_bwd_grouped_dims(m, k, n, n_groups, rank, groups_per_weight)) return 0;
  return make_bwd_grouped_layout(m, k, n, n_groups, rank, groups_per_weight).total;
}

int mi355_w8a8_grouped_bwd_v1(const mi355_w8a8_grouped_bwd_problem* p, void* stream) {
  return run_grouped_backward(p, static_cast<hipStream_t>(stream));
}

int mi355_w8a8_qkv_split_norm_rope_v1(const mi355_w8a8_qkv_post_problem* p, void* stream) {
  return run_qkv_post(p, static_cast<hipStream_t>(stream));
}

uint64_t mi355_w8a8_qkv_bwd_workspace_bytes(uint32_t m, uint32_t head_dim) { return qkv_bwd_workspace_bytes(m, head_dim); }

int mi355_w8a8_qkv_split_norm_rope_bwd_v1(const mi355_w8a8_qkv_post_bwd_problem* p, void* stream) {
  return run_qkv_post_bwd(p, static_cast<hipStream_t>(stream));
}

uint64_t mi355_w8a8_delta_rms_norm_bwd_workspace_bytes(uint32_t m, uint32_t k) {
  return delta_rms_bwd_workspace_bytes(m, k);
}

int mi355_w8a8_delta_rms_norm_bwd_v1(const void* x, const float* gamma, const void* d_normalized, void* d_x,
                                     float* d_gamma, void* workspace, uint64_t workspace_bytes, uint32_t m,
                                     uint32_t k, float eps, void* stream) {
  return run_delta_rms_norm_bwd(x, gamma, d_normalized, d_x, d_gamma, workspace, workspace_bytes, m, k, eps,
                                static_cast<hipStream_t>(stream));
}

int mi355_w8a8_swiglu_v1(const void* fused, void* product, uint32_t m, uint32_t n, void* stream) {
  return run_swiglu_fwd(fused, product, m, n, static_cast<hipStream_t>(stream));
}

int mi355_w8a8_swiglu_bwd_v1(const void* fused, const void* d_product, void* d_fused, uint32_t m, uint32_t n,
                             void* stream) {
  return run_swiglu_bwd(fused, d_product, d_fused, m, n, static_cast<hipStream_t>(stream));
}

int mi355_w8a8_rms_norm_bwd_v1(const void* x, const float* gamma, const void* d_normalized, void* d_x, uint32_t m,
                               uint32_t k, float eps, void* stream) {
  return run_rms_norm_bwd(x, gamma, d_normalized, d_x, m, k, eps, static_cast<hipStream_t>(stream));
}

int mi355_w8a8_moe_route_v1(const float* router_logits, uint32_t n_tokens, uint32_t n_experts, uint32_t top_k,
                            uint32_t norm_topk_prob, float* weights, int32_t* selected, void* stream) {
  return run_moe_route(router_logits, n_tokens, n_experts, top_k, norm_topk_prob, weights, selected,
                       static_cast<hipStream_t>(stream));
}

int mi355_w8a8_moe_route_bwd_v1(const float* router_logits, const int32_t* selected, const float* d_weights,
                                uint32_t n_tokens, uint32_t n_experts, uint32_t top_k, uint32_t norm_topk_prob,
                                float* d_router_logits, void* stream) {
  return run_moe_route_bwd(router_logits, selected, d_weights, n_tokens, n_experts, top_k, norm_topk_prob,
                           d_router_logits, static_cast<hipStream_t>(stream));
}

uint64_t mi355_w8a8_moe_dispatch_workspace_bytes(uint32_t n_pairs, uint32_t n_groups) {
  if (validate_moe_sort_dims(n_pairs, n_groups)) return 0;
  return make_moe_sort_layout(n_pairs, n_groups).total;
}

int mi355_w8a8_moe_dispatch_v1(const mi355_w8a8_moe_dispatch_problem* p, void* stream) {
  return run_moe_dispatch(p, static_cast<hipStream_t>(stream));
}

int mi355_w8a8_moe_combine_v1(const void* expert_out, const int32_t* unsort_indices, const float* weights, void* out,
                              uint32_t n_tokens, uint32_t top_k, uint32_t width, void* stream) {
  return run_moe_combine(expert_out, unsort_indices, weights, out, n_tokens, top_k, width,
                         static_cast<hipStream_t>(stream));
}

int mi355_w8a8_moe_combine_bwd_v1(const void* d_out, const void* expert_out, const int32_t* sort_indices,
                                  const float* weights, void* d_expert_out, float* d_weights, uint32_t n_tokens,
                                  uint32_t top_k, uint32_t width, void* stream) {
  return run_moe_combine_bwd(d_out, expert_out, sort_indices, weights, d_expert_out, d_weights, n_tokens, top_k, width,
                             static_cast<hipStream_t>(stream));
}

uint64_t mi355_w8a8_gq_packed_weight_bytes(uint32_t k_pad, uint32_t n, uint32_t weight_bits) {
  if (k_pad == 0 || (k_pad & 31u) || n == 0 || (weight_bits != 4u && weight_bits != 8u)) return 0;
  return gq_packed_bytes(k_pad, n, weight_bits);
}

int mi355_w8a8_gq_pack_weight_v1(const void* codes, void* packed, uint32_t k_pad, uint32_t n, uint32_t weight_bits,
                                 void* stream) {
  return run_gq_pack(codes, packed, k_pad, n, weight_bits, static_cast<hipStream_t>(stream));
}

uint64_t mi355_w8a8_gq_workspace_bytes(uint32_t m, uint32_t k_pad, uint32_t group_size, uint32_t n_adapters,
                                       uint32_t rank) {
  if (validate_gq_dims(m, k_pad, group_size, rank)) return 0;
  return make_gq_layout(m, k_pad, group_size, n_adapters, n_adapters ? rank : 0u).total;
}

int mi355_w8a8_gq_linear_v1(const mi355_w8a8_gq_problem* p, void* stream) {
  return run_gq_linear(p, static_cast<hipStream_t>(stream));
}

uint64_t mi355_w8a8_gq_bwd_workspace_bytes(uint32_t m, uint32_t k, uint32_t k_pad, uint32_t n, uint32_t group_size,
                                           uint32_t rank) {
  if (validate_gq_bwd_dims(m, k, k_pad, n, group_size, rank)) return 0;
  return make_bwd_layout(m, k, n, rank ? 1u : 0u, rank, k_pad).total;
}

int mi355_w8a8_gq_linear_bwd_v1(const mi355_w8a8_gq_bwd_problem* p, void* stream) {
  return run_gq_backward(p, static_cast<hipStream_t>(stream));
}

int mi355_w8a8_forward_path(uint32_t m, uint32_t k, uint32_t n, uint32_t flags) {
  const int st = validate_common(m, k, n);
  if (st) return st;
  if ((flags & MI355_W8A8_FLAG_FORCE_TILED) && (flags & MI355_W8A8_FLAG_FORCE_SKINNY)) return MI355_W8A8_ERR_SHAPE;
  return choose_forward_path(m, k, n, flags);
}

uint64_t mi355_w8a8_calibrate_operand_bytes(void) { return kCalOperandBytes; }

uint64_t mi355_w8a8_calibrate_mfma_ops(uint32_t shape, uint32_t iters) {
  // per wave and round: 16 x (2 x 32 x 32 x 32) or 64 x (2 x 16 x 16 x 64) operations; 4 waves x 256 workgroups
  if (shape > 1u) return 0;
  return (shape == 1u ? 64ull * 32768ull : 16ull * 65536ull) * 4ull * kCalGrid * iters;
}

int mi355_w8a8_calibrate_mfma_v1(uint32_t shape, const void* operands, uint32_t iters, uint64_t* clocks,
                                 int32_t* sink, void* stream) {
  if (!operands || !clocks || !sink) return MI355_W8A8_ERR_NULL;
  if (shape > 1u || iters == 0 || iters > (1u << 18)) return MI355_W8A8_ERR_SHAPE;  // (2^18 rounds keep a launch under half a second)
  if (reinterpret_cast<uintptr_t>(operands) & 15u) return MI355_W8A8_ERR_ALIGN;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const unsigned char* src = static_cast<const unsigned char*>(operands);
  if (shape == 1u) hipLaunchKernelGGL(cal_mfma_kernel<1>, dim3(kCalGrid), dim3(256), 0, s, src, iters, clocks, sink);
  else hipLaunchKernelGGL(cal_mfma_kernel<0>, dim3(kCalGrid), dim3(256), 0, s, src, iters, clocks, sink);
  return launch_status();
}

int mi355_w8a8_calibrate_read_v1(const void* src, uint64_t bytes, uint32_t* sink, void* stream) {
  if (!src || !sink) return MI355_W8A8_ERR_NULL;
  if (bytes == 0 || (bytes & 32767u)) return MI355_W8A8_ERR_SHAPE;
  if (reinterpret_cast<uintptr_t>(src) & 15u) return MI355_W8A8_ERR_ALIGN;
  hipLaunchKernelGGL(cal_read_kernel, dim3(2048), dim3(256), 0, static_cast<hipStream_t>(stream),
                     static_cast<const v4i*>(src), bytes / 16u, sink);
  return launch_status();
}

int mi355_w8a8_calibrate_copy_v1(const void* src, void* dst, uint64_t bytes, void* stream) {
  if (!src || !dst) return MI355_W8A8_ERR_NULL;
  if (bytes == 0 || (bytes & 15u)) return MI355_W8A8_ERR_SHAPE;
  if (!aligned16(src) || !aligned16(dst)) return MI355_W8A8_ERR_ALIGN;
  if (overlaps(src, bytes, dst, bytes)) return MI355_W8A8_ERR_ALIAS;
  hipLaunchKernelGGL(cal_copy_kernel, dim3(4096), dim3(256), 0, static_cast<hipStream_t>(stream),
                     static_cast<const v4i*>(src), static_cast<v4i*>(dst), bytes / 16u);
  return launch_status();
}

}  // extern "C"
