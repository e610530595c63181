// C ABI of libawq_mi355x.so: host-side validation and launch of the gfx950 kernels.
// Every entry point checks its arguments before touching the device, launches on the
// caller's stream and returns; nothing here allocates, synchronises or keeps state apart
// from the thread-local last HIP error and the one-time kernel attribute set-up.  Launch
// shapes assume the MI355X's 256 CUs in 8 XCDs.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstdint>
#include <type_traits>
#include <utility>

#include "../../include/awq_mi355x.h"
#include "../../include/awq_mi355x_dev.h"
#include "awq_dequant.hpp"
#include "awq_gemm_dense.hpp"
#include "awq_gemm_mid.hpp"
#include "awq_gemm_tile.hpp"
#include "awq_gemv.hpp"
#include "awq_moe.hpp"
#include "awq_probes.hpp"

using namespace awqmi;

// Scratch of the allocation-free entry point (awqmi_gemm_f16_noalloc): split-K arrival counters
// (the first AWQMI_WS_COUNTER_BYTES) and fp32 partial tiles.  Every GPU the library runs on
// holds its own copy of this array at its own address until the process ends.  The name below
// is a host-side stand-in, not a device address: host code only ever uses the pointer that
// hipGetSymbolAddress returned for the current device (static_scratch_ptr).
static __device__ __align__(256) unsigned char scratch[AWQMI_STATIC_SCRATCH_BYTES];

namespace {

thread_local int t_last_hip_error = 0;
// which kernel family the last awqmi_gemm_* call on this thread launched (awqmi_dev_last_gemm_form)
thread_local int t_last_gemm_form = 0;
// time-stamp buffer of the call in progress (awqmi_dev_gemm_timeline_f16 only; null otherwise)
thread_local unsigned long long* t_trace = nullptr;

// Launch-rule variant of the call in progress on this thread: -1 (every default) for the whole
// public C ABI; the awqmi_dev_* entry points set it for the duration of their own call only, so
// no call can change what another call, on this thread or any other, launches.
thread_local int t_variant = -1;
struct VariantScope {
  int prev;
  explicit VariantScope(int v) : prev(t_variant) { t_variant = v; }
  ~VariantScope() { t_variant = prev; }
};

// Bits of the `variant` argument of the awqmi_dev_* entry points: each turns one launch choice
// off, or forces one, so that two forms can be compared and timed in one process.
enum : int {
  VAR_WPL1 = 1,               // one packed word per lane for every shape
  VAR_MOE_RING4 = 2,          // MoE launches with the dense kernel's register ring of four steps
  VAR_XCD_RUN_SHIFT = 2,      // bits 2..4 = v: force runs of 1 << (v - 1) blocks per XCD
  VAR_NO_PAIR_COLS = 64,      // never two column blocks per workgroup
  VAR_MOE_RUNS = 512,         // the one-call MoE block takes its 16-slot blocks in tiles of up to four, whatever the shape
  VAR_NO_FUSED_ACT = 1024,    // the one-call MoE block always runs the separate activation kernel
  VAR_MOE_TILE16 = 2048,      // the one-call MoE block always uses the skinny kernel's 16-row blocks
  VAR_NO_LDS_RING = 4096,     // every launch keeps the weight ring in registers
  VAR_ALIGN_ONE_WG = 16384,   // the one-call MoE block aligns batches of more than one routing launch in one workgroup
  VAR_MOE_TILE_SHIFT = 16,    // bits 16..17 = v: the one-call MoE block uses 64 / 128 / 256-row blocks (v = 1 / 2 / 3)
  VAR_MID_M_SKINNY = 1 << 18, // awq_gemm with 17..64 rows: skinny passes wherever they can run
  VAR_MID_M_MFMA = 1 << 19,   // awq_gemm with 17..64 rows: the tile kernel wherever it can run
  VAR_MFMA_ROWS_SHIFT = 20,   // bits 20..22 = v: fused tiles of 64 v rows (v = 1..4) or 16 v rows (v = 5..7) whatever M is
  VAR_NO_TAIL_STEP = 1 << 23, // dense skinny launches never share left-over chunks step by step
  VAR_NO_FOLDED_ROUTE = 1 << 24, // the one-call MoE block always routes in a launch of its own
  VAR_NO_DENSE = 1 << 25,        // awq_gemm never takes the dequantise-once form
  VAR_DENSE = 1 << 26,           // awq_gemm takes the dequantise-once form from 257 rows on (workspace permitting)
  VAR_MOE_T32_WIDE = 1 << 27,    // 32-row MoE blocks in the two-words-per-lane form (one workgroup per CU)
  VAR_TILE_ROWS_SHIFT = 29,      // bits 29..30 = v: fused tiles of 160 / 208 / 224 rows (v = 1 / 2 / 3) whatever M is
  VAR_MID = 1 << 28,             // awq_gemm with 33 .. 64 rows: the one-pass mid kernel on layers of any size
};
inline bool variant_on(int bit) {
  return t_variant >= 0 && (t_variant & bit);
}

// height of the fused kernel's tile that the variant forces, in 16-row steps (0: none)
inline int forced_tile() {
  if (t_variant < 0) return 0;
  constexpr int hi[4] = {0, 10, 13, 14};
  const int v = (t_variant >> VAR_MFMA_ROWS_SHIFT) & 7, h = (t_variant >> VAR_TILE_ROWS_SHIFT) & 3;
  return h ? hi[h] : v <= 4 ? 4 * v : v;
}

inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

// Device address of `scratch` on the current GPU, looked up once per device.
constexpr int MAX_DEVICES = 64;
std::atomic<void*> g_scratch_ptr[MAX_DEVICES];
int static_scratch_ptr(void** out, bool* first_use) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) { t_last_hip_error = (int)e; return AWQMI_LAUNCH_FAILED; }
  if (dev < 0 || dev >= MAX_DEVICES) return AWQMI_BAD_ARGUMENT;
  void* ptr = g_scratch_ptr[dev].load(std::memory_order_acquire);
  *first_use = ptr == nullptr;
  if (!ptr) {
    e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !ptr) { t_last_hip_error = (int)e; return AWQMI_LAUNCH_FAILED; }
    g_scratch_ptr[dev].store(ptr, std::memory_order_release);
  }
  *out = ptr;
  return AWQMI_OK;
}

inline int launch_status() {
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    t_last_hip_error = (int)e;
    return AWQMI_LAUNCH_FAILED;
  }
  return AWQMI_OK;
}

inline int norm_group(int K, int group) { return group <= 0 ? K : group; }

int check_awq_shape(int K, int N, int G) {
  if (K <= 0 || N <= 0 || G <= 0) return AWQMI_BAD_SHAPE;
  if (N % 8 != 0 || K % G != 0) return AWQMI_BAD_SHAPE;
  return AWQMI_OK;
}

// tiled skinny kernel covers: K a multiple of 128 and G in {32, 64, 128 * i}
inline bool gemv_tiled_ok(int K, int G) { return K % 128 == 0 && (G == 32 || G == 64 || G % 128 == 0); }

inline int gemv_wpl(int N) {
  return (variant_on(VAR_WPL1) || (N / 8) % 2 != 0) ? 1 : 2;
}

// Split-K choice.  The skinny kernel runs one workgroup (one wave per SIMD, 16 KiB of loads
// in flight per wave) per CU and that saturates HBM; a second round of workgroups costs a
// drain and refill of the memory pipeline.  So: split K just far enough that the launch is
// one round of at most 256 workgroups, preferring a split whose 4 x split wave ranges
// divide the 128-row chunks evenly, never below one chunk per wave.
// Left-over chunks shared one 32-row step per wave (the kernel's TAIL form): every wave gets
// nchunks / parts whole chunks, and the L chunks left are 4 L steps for the first 4 L waves.
// Used for the split already chosen (down_proj of the 72B shapes, 231 chunks over 32 waves:
// 29 steps on the busiest wave instead of 32, 1.2 - 1.9 us of 30 - 36); letting the split
// choice count on it picked five parts for a 8192 x 10240 layer, which measured 4 % slower
// than six without tail steps.
inline bool gemv_tail_ok(int nchunks, int split) {
  const int parts = 4 * split, base = nchunks / parts, left = nchunks - base * parts;
  return base >= 1 && left > 0 && 4 * left <= parts;
}

// dense launches of up to 16 rows with two words per lane and G = 128 can take the TAIL form
inline bool gemv_tail_shape(int M, int N, int G) {
  return M <= 16 && G == 128 && gemv_wpl(N) == 2 && !variant_on(VAR_NO_TAIL_STEP);
}

// dense: a dense launch (blocks_z = 1), which takes the TAIL form where its shape and the split
// allow; the busiest wave is then counted in 32-row steps (on 21 layer shapes of eight model
// sizes at 1 and 16 rows, every split forced in turn: the pick is the best split or within 2 % of
// it on all 42 points; counting whole chunks was 6 - 8 % behind on the 5120-wide layers).
int pick_split_k(int rows, int K, int N, int G, long long blocks_z, bool dense = false) {
  const bool tail_form = dense && blocks_z == 1 && gemv_tail_shape(rows, N, G);
  const int nchunks = K / 128;
  const long long ncb = (N + 255) / 256;
  const long long wg = ncb * blocks_z;            // workgroups at split 1
  long long smax = 256 / wg;                      // largest split that stays within one round
  if (smax > nchunks / 4) smax = nchunks / 4;
  if (smax > AWQMI_MAX_SPLIT_K) smax = AWQMI_MAX_SPLIT_K;
  if (smax < 1) smax = 1;
  // among splits >= smax / 2 take the one with the best balance (work of the busiest wave)
  long long best = smax;
  double best_cost = 1e300;
  for (long long s = smax; s >= 1 && 2 * s >= smax; --s) {
    const long long parts = 4 * s;
    const double fill = (double)(wg * s) / 256.0;            // fraction of the round used
    double cost;
    if (tail_form) {
      const long long steps = gemv_tail_ok(nchunks, (int)s) ? 4 * (nchunks / parts) + 1
                                                            : 4 * ((nchunks + parts - 1) / parts);
      // the finishing workgroup reads the parts eight at a time: every further batch is one more
      // dependent trip to memory, over partial tiles that grow with the split
      const double batches = (double)((s + 7) / 8 - 1);
      cost = (double)steps * (double)parts / (4.0 * nchunks) / (0.4 + 0.6 * fill) * (1.0 + 0.15 * batches * batches);
      if (cost <= best_cost + 1e-9) { best_cost = cost; best = s; }     // ties go to the smaller split
      continue;
    }
    const long long busiest = (nchunks + parts - 1) / parts;
    cost = (double)busiest * (double)parts / (double)nchunks / (0.5 + 0.5 * fill);
    if (cost < best_cost - 1e-9) { best_cost = cost; best = s; }
  }
  return (int)best;
}

inline size_t gemv_partial_bytes(int N, int split, long long blocks_z, int tile_m = 16) {
  if (split <= 1) return 0;
  const size_t npad = ((size_t)N + 255) / 256 * 256;
  return (size_t)split * (size_t)blocks_z * tile_m * npad * sizeof(float);
}

template <int WPL, int MB, bool MOE, int RING = 4, int KW = 4, bool ACT = false, bool LDSQ = false>
void launch_gemv(const GemvParams& p, dim3 grid, hipStream_t st) {
  if (p.G == 32) hipLaunchKernelGGL((awq_gemv_kernel<WPL, 0, MB, MOE, RING, KW, ACT, LDSQ>), grid, dim3(256), 0, st, p);
  else if (p.G == 64) hipLaunchKernelGGL((awq_gemv_kernel<WPL, 1, MB, MOE, RING, KW, ACT, LDSQ>), grid, dim3(256), 0, st, p);
  else if (p.G == 128) hipLaunchKernelGGL((awq_gemv_kernel<WPL, 2, MB, MOE, RING, KW, ACT, LDSQ>), grid, dim3(256), 0, st, p);
  else hipLaunchKernelGGL((awq_gemv_kernel<WPL, 3, MB, MOE, RING, KW, ACT, LDSQ>), grid, dim3(256), 0, st, p);
}

// rows the skinny kernel takes in one awq_gemm call (passes of up to 32 rows)
constexpr int SKINNY_MAX_M = 64;

// Up to 32 rows one skinny pass (two row blocks share every unpacked operand; see low_tile_pays for the calls of more
// than 16 rows that take a tile instead); from 33 rows on a tile or the one-pass kernel, which two skinny passes
// never beat (nine shapes from 2048 x 5120 to 8192 x 59136, weights read from HBM).
inline bool skinny_rows(int M, int /*N*/) { return M <= 32; }

inline size_t mid_partial_bytes(int N, int split) {
  return split <= 1 ? 0 : (size_t)split * ((N + 255) / 256) * MID_SLOT_FLOATS * sizeof(float);
}
// K split of the mid kernel, within one round of workgroups: a 128-row chunk takes a wave about 4 us,
// the second launch 3 us and a partial tile 64 KiB of traffic each way (the pick is within 3 % of the
// best split on 18 layer shapes at 64 rows).
int mid_pick_split(int K, int N) {
  const int nchunks = K / 128, ncb = (N + 255) / 256;
  int best = 1;
  double best_t = 1e300;
  for (int s = 1; s <= AWQMI_MAX_SPLIT_K && (s == 1 || (4 * s <= nchunks && ncb * s <= 256)); ++s) {
    const double t = 4.0 * ((nchunks + 4 * s - 1) / (4 * s)) + (s > 1 ? 3.0 + 0.033 * ncb * s : 0.0);
    if (t < best_t) { best_t = t; best = s; }
  }
  return best;
}

// From 33 to 64 rows: awq_gemm_mid_kernel on the largest layers, where it beats awq_gemm_tile_kernel, whose tiles of 48 and 64 rows hold
// all rows of the call too.  Both, mid / tile, at 40, 48 and 64 rows (us, weights from HBM, rows as the layer
// method keeps them): 16512 x 43904 (691 Mi weights, G = 32) 148, 149, 152 / 150, 149, 215; 8192 x 59136 (462 Mi) 81, 78, 80 / 79, 78,
// 85; 15360 x 22848 (334 Mi) 78, 76, 77 / 75, 76, 79; 7936 x 41792 (316 Mi) 75, 74, 75 / 67, 67, 70; 29568 x 8192 49, 48, 49 / 44,
// 44, 49; 8192 x 10240 26.4, 26.1, 27.6 / 22, 22, 23; 8320 x 5120 23, 23, 24 / 17.9, 17.8, 18.4; 13312 x 5632 28, 27, 28 / 22, 22, 23.
// On 34 layers of 40 Mi weights and more below the line the tile is 14 % faster on average and 0.3 % slower at worst.  Its column
// blocks run in whole rounds of workgroups: above 256 of them only multiples of 256.
constexpr long long MID_MIN_WEIGHTS = 320LL << 20;
inline bool mid_shape(int M, int K, int N) {
  const int ncb = (N + 255) / 256;
  return M > 32 && M <= MID_MAX_ROWS && K % 128 == 0 && N % 16 == 0 && K >= 2048 &&
         (long long)K * N >= MID_MIN_WEIGHTS && (ncb <= 256 || ncb % 256 == 0);
}
inline bool mid_rows(int M, int K, int N, int G, int ldw) {
  return (mid_shape(M, K, N) || (variant_on(VAR_MID) && M > 32 && M <= MID_MAX_ROWS && N % 16 == 0)) &&
         gemv_tiled_ok(K, G) && (size_t)M * K * 2 < (1ull << 31) && (size_t)K * ldw * 4 < (1ull << 31) &&
         !variant_on(VAR_MID_M_SKINNY) && !variant_on(VAR_MID_M_MFMA);
}

// Work split of the dense kernel (and of a forced height of the tile kernel): whole rounds of 256 tiles run one workgroup per tile; a
// last round of fewer than 129 tiles (and any launch that small) is split in K over
// floor(256 / tiles) workgroups per tile (at most 8, at least 4 k-tiles each).
// The MFMA kernels address X through 32-bit buffer offsets: calls with more than 4 GiB of
// activations run as consecutive row slabs (multiples of 256 rows).
inline int mfma_slab_rows(int M, int K) {
  const long long fit = ((1LL << 32) - 1) / ((long long)K * 2);
  const long long rows = fit / 256 * 256;
  return rows <= 0 ? 0 : (int)(rows < M ? rows : M);
}

struct MfmaPlan { int dp_tiles, sk_tiles, sk_split; size_t part_bytes; };
MfmaPlan plan_mfma(int M, int K, int N, int bm) {
  const int mt = (M + bm - 1) / bm, nt = (N + PF_BN - 1) / PF_BN;
  const int tiles = mt * nt, KT = K / DG_BK;
  MfmaPlan pl{tiles, 0, 1, 0};
  const int rem = tiles % 256;
  if (rem == 0) return pl;
  int c = 256 / rem;
  if (c > 8) c = 8;
  while (c > 1 && KT / c < 4) --c;
  if (c < 2) return pl;
  pl.dp_tiles = tiles - rem;
  pl.sk_tiles = rem;
  pl.sk_split = c;
  pl.part_bytes = (size_t)rem * c * PF_SK_SLOT_FLOATS * sizeof(float);
  return pl;
}

// Dequantise-once form (awq_gemm_dense.hpp): the weights go through awq_dequant_panel_kernel into
// an fp16 panel in the workspace, then awq_gemm_dense_kernel.  The tile kernel unpacks every weight again
// for each 256 rows, which the panel pass pays for once, but runs faster below some 6000 rows.  Both, panel / tile (us, timed in
// turn, 15 layers at 2048 ... 8192 rows):
//   rows             2048          3072          4096          5000          6144          8192
//   8192 x 59136     1586 / 1438   2279 / 2164   2941 / 2868   3617 / 3606   4355 / 4402   5588 / 5743
//   29568 x 8192     800 / 730     1199 / 1126   1488 / 1472   1880 / 1870   2245 / 2229   2932 / 3005
//   3584 x 37888     506 / 465     706 / 662     936 / 906     1139 / 1124   1352 / 1324   1762 / 1770
//   4096 x 2048      55 / 42       65 / 52       79 / 64       84 / 75       93 / 86       107 / 112
//   1024 x 12288     80 / 56       102 / 78      105 / 98      131 / 127     179 / 156     201 / 193
//   512 x 8192       28 / 22       63 / 36       50 / 43       82 / 56       68 / 63       89 / 82
// At 6144 rows the tile is within 2.3 % either way from 2048 weight rows on; with fewer it stays ahead at any size, as the panel is as
// much traffic as the products.  One row count keeps the panel where the tile is 8 - 11 % faster: 2048 on layers of 64 Mi weights and
// more with three quarters of a round of 256 x 256 tiles, whose prefill record and its test name the form.  Narrower ones run the tile
// there (18944 x 3584 260 / 229, 13824 x 5120, G = 32, 283 / 261).  Layers of fewer than 512 weight rows, which no model here has, keep the
// lines that were drawn for all: from 4096 rows on, from 2048 with those three quarters of a round.  K % 64 == 0 and G % 8 == 0 (both
// implied by mfma_ok).
constexpr int DENSE_MIN_ROWS = 6144;
// One rule for the call and for the workspace query: a call never takes the panel in room that another one's query asked for, and no
// room is asked for that the call leaves unused.
inline bool dense_default(int M, int K, int N) {
  const bool wide = M >= 2048 && (long long)((M + 255) / 256) * ((N + 255) / 256) >= 192;
  if (K < 512) return M >= 4096 || wide;
  return (K >= 2048 && M >= DENSE_MIN_ROWS) || (M == 2048 && wide && (long long)K * N >= 64LL << 20);
}
inline bool dense_rows(int M, int K, int N) {
  if (variant_on(VAR_NO_DENSE)) return false;
  if (variant_on(VAR_DENSE)) return M > 256;
  return dense_default(M, K, N);
}
// workspace of the dequantise-once form: counters, K-split partial tiles, then the panel
inline size_t dense_panel_offset(size_t part_bytes) {
  return (AWQMI_WS_COUNTER_BYTES + part_bytes + 1023) / 1024 * 1024;
}

// Fused kernel: height of its tile in 16-row steps and the K split of one launch.  Whole rounds of 256
// tiles run one workgroup per tile; a last round that leaves CUs idle (and any launch that small) may be split
// in K over `split` workgroups per tile, at least four stages of 64 k each.
constexpr int TILE_RT[] = {3, 4, 5, 6, 7, 8, 10, 12, 13, 14, 16};
struct TilePlan { int rt, dp_tiles, sk_tiles, sk_split; size_t part_bytes; };
TilePlan tile_plan(int M, int K, int N, int rt, int split) {
  const int tiles = ((M + 16 * rt - 1) / (16 * rt)) * ((N + TG_COLS - 1) / TG_COLS), rem = tiles % 256;
  if (rem == 0 || split < 2) return TilePlan{rt, tiles, 0, 1, 0};
  return TilePlan{rt, tiles - rem, rem, split, (size_t)rem * split * tg_part_floats(rt) * sizeof(float)};
}
// The cheapest plan whose partial tiles fit into `room` bytes, by price (us): a stage of 64 k costs 0.28 + 0.0746 rt
// on a full chip and down to 0.79 of it on a nearly idle one (the clock), a tile 3.8 stages beside its own, a partial
// last round counts as at least 0.88 of one, a K split 4.3 + 0.22 per part for its sum launch and 0.003 rt per
// partial tile.  Fitted on 7800 timed launches (16 layer shapes from 1024 x 12288 to 8192 x 59136, 33 ... 2047 rows,
// every height of 64 rows and more, up to five splits each): 0.6 % behind the best of them on average, 15 % at worst.  The same
// price on 56 layers at 40, 48 and 64 rows with tiles of 48 as well: 1 % behind the best split of either height.  A price with
// terms for two workgroups on a CU (and splits over 512) is no better: 1.3 % behind on average, 11 % slower than this pick at worst.
double tile_price(const TilePlan& pl, int KT) {
  const double stage = 0.28 + 0.0746 * pl.rt;
  double t = 0.0;
  if (pl.dp_tiles > 0) {
    const double part = (pl.dp_tiles % 256) / 256.0;
    const double rounds = pl.dp_tiles < 256 ? 0.79 + 0.21 * part : pl.dp_tiles / 256 + (part > 0 ? std::max(part, 0.88) : 0.0);
    t += rounds * (KT + 3.8) * stage;
  }
  if (pl.sk_tiles > 0) {
    const int wgs = pl.sk_tiles * pl.sk_split;
    t += ((KT + pl.sk_split - 1) / pl.sk_split + 3.8) * stage * (0.79 + 0.21 * wgs / 256.0) + 4.3 +
         0.22 * pl.sk_split + 0.003 * wgs * pl.rt;
  }
  return t;
}
TilePlan pick_tile(int M, int K, int N, size_t room) {
  const int KT = K / 64;
  TilePlan best{};
  double best_t = 1e300;
  for (const int rt : TILE_RT) {
    const TilePlan one = tile_plan(M, K, N, rt, 1);
    const int tiles = one.dp_tiles, rem = tiles % 256;
    auto take = [&](const TilePlan& pl) {
      const double t = tile_price(pl, KT);
      if (t < best_t) { best_t = t; best = pl; }
    };
    take(one);
    for (int c = 2; rem > 0 && c <= 16 && c * rem <= 256 && KT / c >= 4; ++c) {
      const TilePlan pl = tile_plan(M, K, N, rt, c);
      if (pl.part_bytes <= room) take(pl);
    }
    if (16 * rt >= M) break;        // one tile holds every row: a higher one multiplies more padding
  }
  return best;
}
// 17 .. 32 rows on a tile of 32 whose weights are the integers w - z and whose group sums are scaled in fp32 (SCALE32): as
// exact as the skinny kernel, which multiplies a lane's weights by two row blocks in turn.  Both, skinny / tile, at 17 and 32 rows (us,
// weights from HBM, rows as the layer method keeps them): 2048 x 2048 13.1, 16.2 / 10.0, 10.0; 5120 x 5120 17.8, 23.1 / 14.4, 14.3;
// 4096 x 12288, G = 64, 21.8, 25.1 / 16.7, 16.7; 8192 x 10240 21.2, 25.0 / 20.4, 20.3; 13824 x 5120 24.0, 29.7 / 19.1, 19.1; 5120 x
// 20480 27.3, 31.6 / 21.8, 21.8; 28672 x 4096 28.3, 33.8 / 26.9, 26.6.  Below 128 Mi weights no point of 35 layers is slower; from there
// on the unsplit skinny launch streams better and only 25 rows and more, or groups of 64, gain (16384 x 8192 25.5, 29.1 / 26.0, 25.8;
// 29568 x 8192 37.5, 41.0 / 38.9, 38.9, G = 64 41.6, 45.1 / 41.6, 41.4), and above 256 Mi neither (8192 x 59136 64, 60 / 68, 69).  Up to 16 rows the
// skinny kernel stays: at 16 it is 5 - 29 % faster on 12 of 16 layers, 7 % slower at worst (1024 x 12288 10.8 / 10.0), at 4 rows 15 - 49 %
// faster.
// Groups of 32 and of more than 128, and ragged columns, stay too: a tile scales its sums after one or two whole stages of 64 k, and
// with weights rounded to fp16 as on higher tiles it would be less exact than the skinny kernel.
bool low_tile_pays(int M, int K, int N, int G) {
  return M > 16 && M <= 32 && (G == 64 || G == 128) && N % 32 == 0 && K % 128 == 0 &&
         (long long)K * N < (M > 24 || G == 64 ? 256LL << 20 : 128LL << 20);
}
// its K split, in whole pairs of stages
TilePlan pick_low_tile(int K, int N) {
  const int KT = K / 64, rem = (N + TG_COLS - 1) / TG_COLS % 256;
  TilePlan best = tile_plan(32, K, N, 2, 1);
  double best_t = tile_price(best, KT);
  for (int c = 2; rem > 0 && c <= 16 && c * rem <= 256 && KT / c >= 4; ++c) {
    const TilePlan pl = tile_plan(32, K, N, 2, c);
    const double t = tile_price(pl, 2 * ((KT / 2 + c - 1) / c) * c);
    if (t < best_t) { best_t = t; best = pl; }
  }
  return best;
}
// Launch of a tile height with the least of three kernels that holds the layer's groups and columns (see awq_tile).
template <int RT>
void launch_tile(const TileGemmParams& p, hipStream_t st) {
  const dim3 grid(p.per_xcd * 8 + p.sk_tiles * p.sk_split);
  if (p.G % 64 == 0 && p.N % 32 == 0) hipLaunchKernelGGL((awq_gemm_tile_kernel<RT, 0>), grid, dim3(256), 0, st, p);
  else if (p.G >= 32) hipLaunchKernelGGL((awq_gemm_tile_kernel<RT, 2>), grid, dim3(256), 0, st, p);
  else hipLaunchKernelGGL((awq_gemm_tile_kernel<RT, 8>), grid, dim3(256), 0, st, p);
  if (p.sk_tiles > 0) hipLaunchKernelGGL((awq_gemm_tile_reduce_kernel<RT>), dim3(p.sk_tiles * RT), dim3(1024), 0, st, p);
}
void launch_tile(int rt, const TileGemmParams& p, hipStream_t st) {
  switch (rt) {
    case 2: {
      const dim3 grid(p.per_xcd * 8 + p.sk_tiles * p.sk_split);
      if (p.G == 64) hipLaunchKernelGGL((awq_gemm_tile_kernel<2, 0, 1>), grid, dim3(256), 0, st, p);
      else hipLaunchKernelGGL((awq_gemm_tile_kernel<2, 0, 2>), grid, dim3(256), 0, st, p);
      if (p.sk_tiles > 0) hipLaunchKernelGGL((awq_gemm_tile_reduce_kernel<2>), dim3(p.sk_tiles * 2), dim3(1024), 0, st, p);
      return;
    }
    case 3: return launch_tile<3>(p, st);
    case 4: return launch_tile<4>(p, st);
    case 5: return launch_tile<5>(p, st);
    case 6: return launch_tile<6>(p, st);
    case 7: return launch_tile<7>(p, st);
    case 8: return launch_tile<8>(p, st);
    case 10: return launch_tile<10>(p, st);
    case 12: return launch_tile<12>(p, st);
    case 13: return launch_tile<13>(p, st);
    case 14: return launch_tile<14>(p, st);
    default: return launch_tile<16>(p, st);
  }
}

}  // namespace

// The routing kernels come for 16 or 64 lanes per token, 4, 8 or 16 resp. 1 to 16 experts per lane, and both scorings:
// f(lanes, experts per lane, sigmoid) for all of them ...
template <class F>
static void moe_topk_forms(F&& f) {
  using std::integral_constant;
  auto both = [&](auto L, auto P) {
    f(L, P, std::false_type{});
    f(L, P, std::true_type{});
  };
  both(integral_constant<int, 16>{}, integral_constant<int, 4>{});
  both(integral_constant<int, 16>{}, integral_constant<int, 8>{});
  both(integral_constant<int, 16>{}, integral_constant<int, 16>{});
  both(integral_constant<int, 64>{}, integral_constant<int, 1>{});
  both(integral_constant<int, 64>{}, integral_constant<int, 2>{});
  both(integral_constant<int, 64>{}, integral_constant<int, 4>{});
  both(integral_constant<int, 64>{}, integral_constant<int, 8>{});
  both(integral_constant<int, 64>{}, integral_constant<int, 16>{});
}
// ... and for the one that E experts, topk of them a token, take: a row of 16 lanes holds 16 picks and 16 keys a lane.
static int moe_topk_lanes(int E, int topk) { return E <= 256 && topk <= 16 ? 16 : 64; }
template <class F>
static void moe_topk_form(int E, int topk, int scoring, F&& f) {
  const int lanes = moe_topk_lanes(E, topk);
  int per = lanes == 16 ? 4 : 1;
  while (lanes * per < E) per *= 2;
  moe_topk_forms([&](auto L, auto P, auto S) {
    if (decltype(L)::value == lanes && decltype(P)::value == per && decltype(S)::value == (scoring == 1)) f(L, P, S);
  });
}

// Kernels that use more dynamic LDS than the default limit need a function attribute; it is
// set once per device for all of them (by awqmi_init, or by the first call on that device that
// needs one).
static int ensure_kernel_attributes() {
  static std::atomic<bool> done[MAX_DEVICES];
  int dev = -1;
  const hipError_t ge = hipGetDevice(&dev);
  if (ge != hipSuccess) { t_last_hip_error = (int)ge; return AWQMI_LAUNCH_FAILED; }
  if (dev < 0 || dev >= MAX_DEVICES) return AWQMI_BAD_ARGUMENT;
  if (done[dev].load(std::memory_order_acquire)) return AWQMI_OK;
  auto allow = [](const void* fn, int bytes) {
    const hipError_t e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    if (e != hipSuccess) t_last_hip_error = (int)e;
    return e == hipSuccess;
  };
  constexpr int align_lds = (MOE_ALIGN_WAVES + 2) * AWQMI_MAX_EXPERTS * (int)sizeof(int);
  bool ok = allow(reinterpret_cast<const void*>(moe_align_kernel), align_lds) &&
            allow(reinterpret_cast<const void*>(moe_align_parts_kernel), moe_parts_lds(AWQMI_MAX_EXPERTS));
  moe_topk_forms([&](auto L, auto P, auto S) {
    ok = ok && allow(reinterpret_cast<const void*>(moe_route_align_kernel<decltype(L)::value, decltype(P)::value, decltype(S)::value>), align_lds);
  });
  if (!ok) return AWQMI_LAUNCH_FAILED;
  done[dev].store(true, std::memory_order_release);
  return AWQMI_OK;
}

// Routing of one MoE block: inputs and the five lists it produces.
struct MoeRoute {
  const float* logits;
  const float* bias;
  int T, E, topk, scoring, renorm;
  float scale;
  int32_t* ids;
  float* wts;
  int32_t* sorted;
  int32_t* experts;
  int32_t* npp;
  int32_t* runs;     // tiles of several 16-slot blocks, or null
  int32_t* tab;      // expert counts of the parts of a longer batch, [MOE_PARTS_MAX][E]
};

static int moe_align_launch(const int32_t* topk_ids, int n_slots, int E, int tile_m, int32_t* sorted, int32_t* experts,
                            int32_t* npp, int32_t* runs, void* stream) {
  const int cap = (int)awqmi_moe_align_capacity(n_slots, E, tile_m);
  if (const int rc = ensure_kernel_attributes()) return rc;
  hipLaunchKernelGGL(moe_align_kernel, dim3(1), dim3(1024), (size_t)(MOE_ALIGN_WAVES + 2) * E * sizeof(int),
                     (hipStream_t)stream, topk_ids, n_slots, E, tile_m, cap, sorted, experts, npp, runs);
  return launch_status();
}
// Routing + align of a block as launches of their own.  Up to 32 tokens (16 with a token a wave): one launch of one workgroup.  Up to 3584
// slots (11264 with a token a wave): top-k over many, then one workgroup for the align.  More: two launches over up to MOE_PARTS_MAX
// workgroups, each with at least sixteen tokens; with a token a wave three, the picks having one of their own.  Whole block, 128 experts of 2048 x 768, top-8, us, as it was before / one launch / top-k and one workgroup / two
// launches of parts: 16 tokens 62.2 / 59.3 / - / -; 32 72.2 / 70.5 / - / -; 48 73.3 / 72.9 / 72.5 / -; 64 75.3 / 75.3 / 74.5 / -; 128 80.6 / - /
// 80.1 / 81.2; 256 98 / - / 97.5 / 97.3; 1500 172 / - / - / 166; 8192 696 / - / - / 688.
// Four tokens a wave, blocks of 256 x 128, align in one workgroup / in parts at 2064, 3200, 4096, 6500 slots: 256 experts, top-8 31.9, 33.9, 34.8, 44.2 / 32.7,
// 34.7, 35.2, 44.1; 256, top-2 30.0, 32.3, 33.2, 43.0 / 30.9, 34.6, 33.5, 43.2; 128, top-8 27.5, 29.5, 32.2, 35.8 / 28.0, 29.5, 31.7, 34.3; 128, top-2
// 26.2, 28.6, 30.8, 34.8 / 28.1, 31.0, 30.7, 35.2; 64, top-6 26.6, 27.6, 30.9, 34.5 / 26.7, 27.3, 30.3, 32.8; 8, top-2 25.7, 27.3, 30.3, 35.5 / 26.5, 27.3, 29.6, 33.0.
// A token a wave, the same block, us, align in one workgroup / in parts: 4096, 8192, 12000, 16000, 24000 slots of 512 experts, top-10 49.3,
// 54.8, 62.4, 73.5, 94.2 / 51.9, 54.0, 58.8, 67.6, 82.0; of 257, top-8 38.2, 50.1, 58.5, 69.1, 89.7 / 40.8, 49.5, 56.9, 64.7, 80.2; of 1024, top-2 56.1, 69.1,
// 76.8, 88.5, 116 / 60.2, 71.8, 78.7, 87.0, 107.7; of 64, top-17 35.1, 47.8, 53.8, 62.6, 76.7 / 35.8, 45.9, 50.9, 57.7, 66.1.
constexpr int MOE_ONE_WG_SLOTS = 3584, MOE_ONE_WG_SLOTS_WAVE = 11264;
struct MoeParts { int part, parts; };     // tokens of a part, parts
static MoeParts moe_parts(int T) {
  const int part = (T + 16 * MOE_PARTS_MAX - 1) / (16 * MOE_PARTS_MAX) * 16;
  return {part, (T + part - 1) / part};
}
// The table of counts has room of its own for 64 parts, the rest lies where the activation goes later: a block in parts has more
// than MOE_ONE_WG_SLOTS rows of that, each of 128 columns or more (K of the second expert GEMM).
constexpr int MOE_TAB_PARTS = 64;
static_assert((MOE_ONE_WG_SLOTS + 1) * 128 * sizeof(half_t) >=
                  (size_t)(MOE_PARTS_MAX - MOE_TAB_PARTS) * AWQMI_MAX_EXPERTS * sizeof(int32_t),
              "every part's counts lie inside the workspace");
static int moe_route_launches(const MoeRoute& r, int tile, void* stream) {
  if (const int rc = ensure_kernel_attributes()) return rc;
  const int n_slots = r.T * r.topk, cap = (int)awqmi_moe_align_capacity(n_slots, r.E, tile);
  hipStream_t st = (hipStream_t)stream;
  const int wave_tokens = 64 / moe_topk_lanes(r.E, r.topk);
  if (r.T <= MOE_ALIGN_WAVES * std::min(wave_tokens, 2)) {
    moe_topk_form(r.E, r.topk, r.scoring, [&](auto L, auto P, auto S) {
      hipLaunchKernelGGL((moe_route_align_kernel<decltype(L)::value, decltype(P)::value, decltype(S)::value>), dim3(1), dim3(1024),
                         (size_t)(MOE_ALIGN_WAVES + 2) * r.E * sizeof(int), st, r.logits, r.bias, r.T, r.E, r.topk, r.renorm,
                         r.scale, r.ids, r.wts, tile, cap, r.sorted, r.experts, r.npp, r.runs);
    });
    return launch_status();
  }
  if (n_slots <= (wave_tokens > 1 ? MOE_ONE_WG_SLOTS : MOE_ONE_WG_SLOTS_WAVE) || variant_on(VAR_ALIGN_ONE_WG)) {
    if (const int rc = awqmi_moe_topk_f32(r.logits, r.bias, r.T, r.E, r.topk, r.scoring, r.renorm, r.scale, r.ids, r.wts, stream))
      return rc;
    return moe_align_launch(r.ids, n_slots, r.E, tile, r.sorted, r.experts, r.npp, r.runs, stream);
  }
  const MoeParts pt = moe_parts(r.T);
  if (wave_tokens > 1) {
    const int waves = std::min(16, pt.part / wave_tokens);
    moe_topk_form(r.E, r.topk, r.scoring, [&](auto L, auto P, auto S) {
      if constexpr (decltype(L)::value == 16)
        hipLaunchKernelGGL((moe_route_count_kernel<decltype(P)::value, decltype(S)::value>), dim3(pt.parts), dim3(64 * waves), 0, st,
                           r.logits, r.bias, r.T, r.E, r.topk, r.renorm, r.scale, r.ids, r.wts, pt.part, r.tab);
    });
  } else {
    if (const int rc = awqmi_moe_topk_f32(r.logits, r.bias, r.T, r.E, r.topk, r.scoring, r.renorm, r.scale, r.ids, r.wts, stream))
      return rc;
    hipLaunchKernelGGL(moe_count_kernel, dim3(pt.parts), dim3(1024), 0, st, r.ids, n_slots, r.E, pt.part * r.topk, r.tab);
  }
  hipLaunchKernelGGL(moe_align_parts_kernel, dim3(pt.parts), dim3(1024), (size_t)moe_parts_lds(r.E), st, r.ids, n_slots, r.E,
                     pt.part * r.topk, tile, cap, r.tab, r.sorted, r.experts, r.npp, r.runs);
  return launch_status();
}

// Folded routing: no more tokens than the four waves of a workgroup pick for at once (16, or 4 with a token a wave), 64 slots (one lane
// each), 256 experts.  Routed apart /
// folded, us, weights from HBM: 128 experts of 2048 x 768, top-8, at 1, 4, 5, 6, 8 tokens 28.7, 36.7, 38.8, 40.5, 47.4 / 25.0, 31.9, 34.9, 36.6,
// 43.5; 64 of 2048 x 1408, top-6, at 10 53.9 / 50.1; 64 of 5120 x 1024, top-4, at 8, 12, 16 62.2, 84.2, 88.8 / 58.3, 80.0, 84.7; 8 of 4096 x
// 14336, top-2, at 8, 16 142.6, 151.4 / 138.5, 148.5; 256 of 3072 x 1536, top-4, at 16 89.2 / 89.0.
constexpr int MOE_FOLD_EXPERTS = 256;
static bool moe_route_foldable(int T, int E, int topk, int tile) {
  return T <= 4 * (64 / moe_topk_lanes(E, topk)) && T * topk <= 64 && E <= MOE_FOLD_EXPERTS && tile == 16 &&
         !variant_on(VAR_NO_FOLDED_ROUTE);
}

extern "C" {

int awqmi_init(void) {
  if (const int rc = ensure_kernel_attributes()) return rc;
  // the current device's static scratch array: look its address up and put its arrival counters
  // at zero (they are zero when the code object is loaded and every completed call leaves them
  // so; calling this again is the way back after a call that was cut short)
  void* ptr = nullptr;
  bool first = false;
  if (const int rc = static_scratch_ptr(&ptr, &first)) return rc;
  hipLaunchKernelGGL(awq_zero_words_kernel, dim3(AWQMI_WS_COUNTER_BYTES / 16 / 256), dim3(256), 0, (hipStream_t) nullptr,
                     reinterpret_cast<u4v*>(ptr), AWQMI_WS_COUNTER_BYTES / 16);
  if (const int rc = launch_status()) return rc;
  const hipError_t e = hipStreamSynchronize(nullptr);
  if (e != hipSuccess) { t_last_hip_error = (int)e; return AWQMI_LAUNCH_FAILED; }
  return AWQMI_OK;
}

int awqmi_version(void) { return AWQMI_VERSION; }

const char* awqmi_status_string(int s) {
  switch (s) {
    case AWQMI_OK: return "ok";
    case AWQMI_BAD_SHAPE: return "bad shape (need N % 8 == 0, K % group == 0, positive sizes)";
    case AWQMI_BAD_ALIGN: return "pointer not 16-byte aligned";
    case AWQMI_WORKSPACE_TOO_SMALL: return "workspace too small";
    case AWQMI_UNSUPPORTED_GROUP: return "unsupported group size";
    case AWQMI_LAUNCH_FAILED: return "kernel launch failed";
    case AWQMI_NULL_POINTER: return "null pointer";
    case AWQMI_BAD_ARGUMENT: return "bad argument";
    case AWQMI_SCRATCH_LIMIT:
      return "call needs more scratch than the static array holds (AWQMI_STATIC_SCRATCH_BYTES); "
             "use awqmi_gemm_f16 with a caller-owned workspace";
    default: return "unknown status";
  }
}

int awqmi_last_hip_error(void) { return t_last_hip_error; }

int awqmi_dequantize_f16(const int32_t* qweight, const void* scales, const int32_t* qzeros,
                         void* out, int K, int N, int group, void* stream) {
  return awqmi_dequantize_ld_f16(qweight, N / 8, scales, qzeros, out, K, N, group, stream);
}

int awqmi_dequantize_ld_f16(const int32_t* qweight, int ldw, const void* scales, const int32_t* qzeros,
                            void* out, int K, int N, int group, void* stream) {
  if (!qweight || !scales || !qzeros || !out) return AWQMI_NULL_POINTER;
  const int G = norm_group(K, group);
  if (const int rc = check_awq_shape(K, N, G)) return rc;
  if (ldw < N / 8 || (ldw != N / 8 && ldw % 4 != 0)) return AWQMI_BAD_ARGUMENT;
  if (!aligned16(scales) || !aligned16(out) || !aligned16(qweight) || !aligned16(qzeros))
    return AWQMI_BAD_ALIGN;
  const int NW = N / 8;
  hipStream_t st = (hipStream_t)stream;
  const uint32_t* qw = reinterpret_cast<const uint32_t*>(qweight);
  const uint32_t* qz = reinterpret_cast<const uint32_t*>(qzeros);
  const half_t* sc = reinterpret_cast<const half_t*>(scales);
  half_t* o = reinterpret_cast<half_t*>(out);
  const unsigned gx = (NW + 255) / 256;
#define AWQMI_DQ(R)                                                                              \
  for (int k0 = 0; k0 < K; k0 += 65535 * R) {                                                    \
    const int slabs = (K - k0) / R < 65535 ? (K - k0) / R : 65535;                               \
    hipLaunchKernelGGL((awq_dequant_kernel<R>), dim3(gx, slabs), dim3(256), 0, st, qw, sc, qz, o, k0, \
                       NW, G, ldw);                                                              \
  }
  if (G % 16 == 0) AWQMI_DQ(16)
  else if (G % 8 == 0) AWQMI_DQ(8)
  else if (G % 4 == 0) AWQMI_DQ(4)
  else if (G % 2 == 0) AWQMI_DQ(2)
  else AWQMI_DQ(1)
#undef AWQMI_DQ
  return launch_status();
}

int awqmi_gemm_auto_split_k(int M, int K, int N, int group) {
  const int G = norm_group(K, group);
  if (check_awq_shape(K, N, G) != AWQMI_OK || M <= 0) return 1;
  if (!skinny_rows(M, N) || !gemv_tiled_ok(K, G)) return 1;
  return pick_split_k(M, K, N, G, 1, true);
}

size_t awqmi_gemm_workspace_bytes(int M, int K, int N, int split_k) {
  if (M <= 0 || K <= 0 || N <= 0) return 0;
  // the group size decides between the kernels for some shapes, so cover both
  size_t mfma = 0, skinny = 0;
  if (M > 16 && K % DG_BK == 0) {
    const int slab = mfma_slab_rows(M, K);
    if (slab > 0) {
      // the plan the call will pick, and room for the K split of 256-row tiles at least (any forced size
      // that needs more runs unsplit)
      for (const int m : {slab, M % slab})
        if (m > 0)
          mfma = std::max({mfma, pick_tile(m, K, N, SIZE_MAX).part_bytes, plan_mfma(m, K, N, 256).part_bytes});
      // the dequantise-once form of many-row calls: 256-row tiles, and the fp16 panel behind the
      // partial tiles (a call with a smaller workspace runs the fused kernel instead)
      if (dense_default(M, K, N)) {
        size_t part = plan_mfma(slab, K, N, 256).part_bytes;
        if (M % slab) part = std::max(part, plan_mfma(M % slab, K, N, 256).part_bytes);
        const size_t dense = dense_panel_offset(part) + dg_panel_bytes(K, N) - AWQMI_WS_COUNTER_BYTES;
        mfma = std::max(mfma, dense);
      }
    }
  }
  if (M <= SKINNY_MAX_M) {
    int s = split_k;
    // the pick depends on the group size (TAIL form only at G = 128): cover both
    if (s <= 0) s = (K % 128 == 0) ? std::max(pick_split_k(M, K, N, 128, 1, true), pick_split_k(M, K, N, 64, 1, true)) : 1;
    skinny = gemv_partial_bytes(N, s, 1, 32);
  }
  if (mid_shape(M, K, N))
    skinny = std::max(skinny, mid_partial_bytes(N, mid_pick_split(K, N)));
  return AWQMI_WS_COUNTER_BYTES + (mfma > skinny ? mfma : skinny);
}

int awqmi_gemm_f16(const void* x, const int32_t* qweight, const void* scales, const int32_t* qzeros,
                   void* y, void* workspace, size_t workspace_bytes, int M, int K, int N, int group,
                   int split_k, void* stream) {
  return awqmi_gemm_ld_f16(x, qweight, N / 8, scales, qzeros, y, workspace, workspace_bytes, M, K, N, group, split_k,
                           stream);
}

int awqmi_gemm_ld_f16(const void* x, const int32_t* qweight, int ldw, const void* scales, const int32_t* qzeros,
                      void* y, void* workspace, size_t workspace_bytes, int M, int K, int N, int group,
                      int split_k, void* stream) {
  if (!x || !qweight || !scales || !qzeros || !y) return AWQMI_NULL_POINTER;
  const int G = norm_group(K, group);
  if (const int rc = check_awq_shape(K, N, G)) return rc;
  if (M <= 0) return AWQMI_BAD_SHAPE;
  if (split_k < 0 || split_k > AWQMI_MAX_SPLIT_K) return AWQMI_BAD_ARGUMENT;
  if (ldw < N / 8 || (ldw != N / 8 && ldw % 4 != 0)) return AWQMI_BAD_ARGUMENT;
  if (!aligned16(x) || !aligned16(scales) || !aligned16(qweight) || !aligned16(qzeros) ||
      !aligned16(y))
    return AWQMI_BAD_ALIGN;
  hipStream_t st = (hipStream_t)stream;
  const int NW = N / 8;
  const uint32_t* qw = reinterpret_cast<const uint32_t*>(qweight);
  const uint32_t* qz = reinterpret_cast<const uint32_t*>(qzeros);
  const half_t* sc = reinterpret_cast<const half_t*>(scales);
  const half_t* xx = reinterpret_cast<const half_t*>(x);
  half_t* yy = reinterpret_cast<half_t*>(y);

  const int wpl = gemv_wpl(N);
  const bool mfma_ok = K % DG_BK == 0 && (((G & (G - 1)) == 0 && G >= 8) || G % 64 == 0) &&
                       mfma_slab_rows(M, K) > 0 && (size_t)K * ldw * 4 < (1ull << 32) &&
                       (size_t)(K / G) * N * 2 < (1ull << 32);
  // room for the partial tiles of a K split; without a workspace every tile runs on one workgroup
  const size_t room = workspace && aligned16(workspace) && workspace_bytes > AWQMI_WS_COUNTER_BYTES
                          ? workspace_bytes - AWQMI_WS_COUNTER_BYTES : 0;
  // rows r0 .. r0 + Ms - 1 on the tile kernel
  auto run_tile = [&](const TilePlan& pl, int r0, int Ms) {
    TileGemmParams p{};
    p.x = xx + (size_t)r0 * K; p.qw = qw; p.sc = sc; p.qz = qz; p.y = yy + (size_t)r0 * N;
    p.M = Ms; p.K = K; p.N = N; p.NW = NW; p.ldw = ldw; p.G = G;
    while ((2 << p.gshift) <= G) ++p.gshift;
    p.mt = (Ms + 16 * pl.rt - 1) / (16 * pl.rt); p.nt = (N + TG_COLS - 1) / TG_COLS;
    p.dp_tiles = pl.dp_tiles; p.sk_tiles = pl.sk_tiles; p.sk_split = pl.sk_split;
    p.per_xcd = (pl.dp_tiles + 7) / 8;
    p.sk_part = room ? reinterpret_cast<float*>(static_cast<char*>(workspace) + AWQMI_WS_COUNTER_BYTES) : nullptr;
    launch_tile(pl.rt, p, st);
  };
  if (mid_rows(M, K, N, G, ldw)) {
    t_last_gemm_form = AWQMI_FORM_MID;
    MidGemmParams p{};
    p.x = xx; p.qw = qw; p.sc = sc; p.qz = qz; p.y = yy;
    p.M = M; p.K = K; p.N = N; p.NW = NW; p.G = G; p.ldw = ldw;
    p.ncb = (NW + 31) / 32;
    // split_k is the skinny kernel's; only the development variant lets it set this one's split
    p.split_k = split_k > 0 && variant_on(VAR_MID) ? std::min(split_k, K / 128) : mid_pick_split(K, N);
    // the K split needs the caller's workspace; without it a workgroup takes all of K
    if (p.split_k > 1 && (!workspace || !aligned16(workspace) ||
                          workspace_bytes < AWQMI_WS_COUNTER_BYTES + mid_partial_bytes(N, p.split_k)))
      p.split_k = 1;
    p.part = workspace ? reinterpret_cast<float*>(static_cast<char*>(workspace) + AWQMI_WS_COUNTER_BYTES) : nullptr;
    const dim3 grid(p.ncb, p.split_k);
    if (G == 32) hipLaunchKernelGGL(awq_gemm_mid_kernel<4>, grid, dim3(256), 0, st, p);
    else if (G == 64) hipLaunchKernelGGL(awq_gemm_mid_kernel<2>, grid, dim3(256), 0, st, p);
    else hipLaunchKernelGGL(awq_gemm_mid_kernel<1>, grid, dim3(256), 0, st, p);
    if (p.split_k > 1)
      hipLaunchKernelGGL(awq_gemm_mid_reduce_kernel, dim3(p.ncb, (M + 15) / 16), dim3(256), 0, st, p);
    return launch_status();
  }
  bool mid_skinny = skinny_rows(M, N);
  if (variant_on(VAR_MID_M_SKINNY)) mid_skinny = true;
  if (variant_on(VAR_MID_M_MFMA)) mid_skinny = false;
  if (gemv_tiled_ok(K, G) &&
      (M <= 16 || (M <= SKINNY_MAX_M && wpl == 2 && (mid_skinny || !mfma_ok)))) {
    int split = split_k > 0 ? split_k : pick_split_k(M, K, N, G, 1, true);
    const int nchunks = K / 128;
    if (split > nchunks) split = nchunks;
    const int ncb = (NW + 16 * wpl - 1) / (16 * wpl);
    if (split > 1) {
      if (!workspace) return AWQMI_NULL_POINTER;
      if (!aligned16(workspace)) return AWQMI_BAD_ALIGN;
      if ((size_t)ncb * sizeof(int) > AWQMI_WS_COUNTER_BYTES) return AWQMI_BAD_SHAPE;
      if (workspace_bytes < AWQMI_WS_COUNTER_BYTES + gemv_partial_bytes(N, split, 1, M > 16 ? 32 : 16))
        return AWQMI_WORKSPACE_TOO_SMALL;
    }
    if (split_k == 0 && mfma_ok && !t_trace && !variant_on(VAR_MID_M_SKINNY) && low_tile_pays(M, K, N, G)) {
      const TilePlan pl = pick_low_tile(K, N);
      if (pl.part_bytes <= room) {
        t_last_gemm_form = AWQMI_FORM_FUSED;
        run_tile(pl, 0, M);
        return launch_status();
      }
    }
    t_last_gemm_form = AWQMI_FORM_SKINNY;
    GemvParams p{};
    p.qw = qw; p.sc = sc; p.qz = qz;
    p.cnt = reinterpret_cast<int*>(workspace);
    p.part = workspace ? reinterpret_cast<float*>(static_cast<char*>(workspace) + AWQMI_WS_COUNTER_BYTES)
                       : nullptr;
    p.K = K; p.N = N; p.NW = NW; p.ldw = ldw; p.G = G; p.ldy = N;
    p.split_k = split; p.ncb = ncb;
    p.trace = t_trace;
    const dim3 grid(ncb, split, 1);
    // passes of up to 32 rows; each pass streams the weights once
    for (int r0 = 0; r0 < M; r0 += 32) {
      p.x = xx + (size_t)r0 * K;
      p.y = yy + (size_t)r0 * N;
      p.M = M - r0 < 32 ? M - r0 : 32;
      // 17 .. 32 rows with long wave ranges (six chunks or more): the weight ring in LDS leaves the
      // register file to the two accumulator sets (gate_up / down_proj of the 72B shapes 3 - 11 %
      // faster, bit-identical; short ranges measured equal or 1 - 2 % slower)
      const bool lds32 = nchunks >= 24 * split && (size_t)K * ldw * 4 < (1ull << 31) && !variant_on(VAR_NO_LDS_RING);
      if (p.M > 16 && lds32) launch_gemv<2, 2, false, 4, 4, false, true>(p, grid, st);
      else if (p.M > 16) launch_gemv<2, 2, false>(p, grid, st);
      else if (gemv_tail_shape(p.M, N, G) && gemv_tail_ok(nchunks, split))
        hipLaunchKernelGGL((awq_gemv_tail_kernel<2, 1>), grid, dim3(256), 0, st, p);
      else if (wpl == 2) launch_gemv<2, 1, false>(p, grid, st);
      else launch_gemv<1, 1, false>(p, grid, st);
    }
    return launch_status();
  }

  // MFMA kernels: K % 64 == 0, G a power of two >= 8 or a multiple of 64; buffer offsets are
  // 32-bit, so every operand must stay below 4 GiB
  if (mfma_ok) {
    const int slab = mfma_slab_rows(M, K);
    // many rows: dequantise once into the workspace, then the dense kernel (the tile kernel's products, added in the
    // same order where both split K alike); needs the workspace to hold the panel
    if (dense_rows(M, K, N) && workspace && aligned16(workspace)) {
      size_t part = plan_mfma(slab < M ? slab : M, K, N, 256).part_bytes;
      if (M % slab) part = std::max(part, plan_mfma(M % slab, K, N, 256).part_bytes);
      const size_t panel_off = dense_panel_offset(part);
      if (workspace_bytes >= panel_off + dg_panel_bytes(K, N)) {
        t_last_gemm_form = AWQMI_FORM_DENSE;
        unsigned char* const panel = static_cast<unsigned char*>(workspace) + panel_off;
        const int nt = (N + 255) / 256;
        hipLaunchKernelGGL(awq_dequant_panel_kernel, dim3(nt, K / 64), dim3(256), 0, st, qw, sc, qz, panel, K, N, NW, G,
                           ldw);
        for (int r0 = 0; r0 < M; r0 += slab) {
          const int Ms = M - r0 < slab ? M - r0 : slab;
          const MfmaPlan pl = plan_mfma(Ms, K, N, 256);
          DenseGemmParams d{};
          d.x = xx + (size_t)r0 * K; d.panel = panel; d.y = yy + (size_t)r0 * N;
          d.M = Ms; d.K = K; d.N = N;
          d.mt = (Ms + 255) / 256; d.nt = nt;
          d.dp_tiles = pl.dp_tiles; d.sk_tiles = pl.sk_tiles; d.sk_split = pl.sk_split;
          d.per_xcd = (pl.dp_tiles + 7) / 8;
          d.sk_part = reinterpret_cast<float*>(static_cast<char*>(workspace) + AWQMI_WS_COUNTER_BYTES);
          hipLaunchKernelGGL(awq_gemm_dense_kernel, dim3(d.per_xcd * 8 + d.sk_tiles * d.sk_split), dim3(256), 0, st, d);
          if (d.sk_tiles > 0)
            hipLaunchKernelGGL(awq_gemm_dense_reduce_kernel, dim3(d.sk_tiles * 8), dim3(256), 0, st, d);
        }
        return launch_status();
      }
    }
    t_last_gemm_form = AWQMI_FORM_FUSED;
    const int forced = forced_tile();
    for (int r0 = 0; r0 < M; r0 += slab) {
      const int Ms = M - r0 < slab ? M - r0 : slab;
      TilePlan pl;
      if (forced) {
        // a forced height takes the dense kernel's split rule
        pl = tile_plan(Ms, K, N, forced, plan_mfma(Ms, K, N, 16 * forced).sk_split);
        if (pl.part_bytes > room) pl = tile_plan(Ms, K, N, forced, 1);
      } else {
        pl = pick_tile(Ms, K, N, room);
      }
      run_tile(pl, r0, Ms);
    }
    return launch_status();
  }

  // any other shape: one thread per packed word and row; the row index is the grid's second
  // dimension (at most 65535), so more rows run as consecutive slabs
  t_last_gemm_form = AWQMI_FORM_GENERIC;
  for (int r0 = 0; r0 < M; r0 += 32768) {
    const int Ms = M - r0 < 32768 ? M - r0 : 32768;
    hipLaunchKernelGGL(awq_gemm_generic_kernel, dim3((NW + 255) / 256, Ms), dim3(256), 0, st,
                       xx + (size_t)r0 * K, qw, sc, qz, yy + (size_t)r0 * N, Ms, K, NW, G, ldw);
  }
  return launch_status();
}

int awqmi_gemm_f16_noalloc(const void* x, const int32_t* qweight, int ldw, const void* scales, const int32_t* qzeros,
                           void* y, int M, int K, int N, int group, int split_k, void* stream) {
  void* ptr = nullptr;
  bool first = false;
  if (const int rc = static_scratch_ptr(&ptr, &first)) return rc;
  // exactly awqmi_gemm_ld_f16 with this GPU's static array as the workspace (it validates before
  // it launches, so a skinny call whose split-K partial tiles do not fit launches nothing)
  const int rc = awqmi_gemm_ld_f16(x, qweight, ldw == 0 ? N / 8 : ldw, scales, qzeros, y, ptr, AWQMI_STATIC_SCRATCH_BYTES,
                                   M, K, N, group, split_k, stream);
  return rc == AWQMI_WORKSPACE_TOO_SMALL ? AWQMI_SCRATCH_LIMIT : rc;
}

int awqmi_moe_topk_f32(const float* logits, const float* score_bias, int T, int E, int topk, int scoring,
                       int renormalize, float scale, int32_t* topk_ids, float* topk_weights, void* stream) {
  if (!logits || !topk_ids || !topk_weights) return AWQMI_NULL_POINTER;
  if (T <= 0 || E <= 0) return AWQMI_BAD_SHAPE;
  if (E > AWQMI_MAX_EXPERTS || topk <= 0 || topk > E || topk > 64 || (scoring != 0 && scoring != 1))
    return AWQMI_BAD_ARGUMENT;
  if (scoring == 0 && score_bias) return AWQMI_BAD_ARGUMENT;   // the bias belongs to sigmoid scoring
  const int tokens = 4 * 64 / moe_topk_lanes(E, topk);      // of a workgroup
  moe_topk_form(E, topk, scoring, [&](auto L, auto P, auto S) {
    hipLaunchKernelGGL((moe_topk_kernel<decltype(L)::value, decltype(P)::value, decltype(S)::value>), dim3((T + tokens - 1) / tokens),
                       dim3(256), 0, (hipStream_t)stream, logits, score_bias, T, E, topk, renormalize, scale, topk_ids, topk_weights);
  });
  return launch_status();
}

int awqmi_moe_topk_softmax_f32(const float* logits, int T, int E, int topk, int renormalize,
                               int32_t* topk_ids, float* topk_weights, void* stream) {
  return awqmi_moe_topk_f32(logits, nullptr, T, E, topk, 0, renormalize, 1.f, topk_ids, topk_weights, stream);
}

size_t awqmi_moe_align_capacity(int n_slots, int E, int tile_m) {
  if (n_slots < 0 || E <= 0 || tile_m <= 0) return 0;
  const size_t worst = (size_t)n_slots + (size_t)E * (tile_m - 1);
  return (worst + tile_m - 1) / tile_m * tile_m;
}

int awqmi_moe_align(const int32_t* topk_ids, int n_slots, int E, int tile_m, int32_t* sorted_token_ids,
                    int32_t* expert_ids, int32_t* num_tokens_post_padded, void* stream) {
  if (!topk_ids || !sorted_token_ids || !expert_ids || !num_tokens_post_padded)
    return AWQMI_NULL_POINTER;
  if (n_slots <= 0 || E <= 0) return AWQMI_BAD_SHAPE;
  if (E > AWQMI_MAX_EXPERTS || tile_m <= 0 || tile_m > 4096) return AWQMI_BAD_ARGUMENT;
  return moe_align_launch(topk_ids, n_slots, E, tile_m, sorted_token_ids, expert_ids, num_tokens_post_padded, nullptr, stream);
}

// sorted-token blocks a grouped launch covers: the align capacity, rounded up to whole groups
static int moe_launch_blocks(int n_slots, int E, int tile_m) {
  int nblk = (int)(awqmi_moe_align_capacity(n_slots, E, tile_m) / tile_m);
  // a block that runs holds at least one real slot: a handful of tokens never fills more blocks
  // than it has slots, whatever the expert count (one token with 8 picks of 128 experts: 8
  // blocks, not 121 -- the rest would be workgroups that start, read the padded count and leave)
  if (nblk > n_slots) nblk = n_slots;
  return (nblk + MOE_BLOCK_GROUP_MAX - 1) / MOE_BLOCK_GROUP_MAX * MOE_BLOCK_GROUP_MAX;
}

// Launch shape of a grouped GEMM, shared by the workspace query and the launch itself.
struct MoePlan { int wpl, ncb, nblk, split; };
static MoePlan moe_plan(int n_slots, int E, int K, int N, int tile_m, int split_req) {
  MoePlan pl{};
  const int NW = N / 8;
  pl.wpl = gemv_wpl(N);
  pl.ncb = (NW + 16 * pl.wpl - 1) / (16 * pl.wpl);
  pl.nblk = moe_launch_blocks(n_slots, E, tile_m);
  const int nchunks = K / 128;
  // blocks that will actually run: at most one per tile_m slots plus one per expert touched
  long long live = (n_slots + tile_m - 1) / tile_m;
  const long long touched = n_slots < E ? n_slots : E;
  if (live < touched) live = touched;
  int s = split_req;
  if (s <= 0) {
    if (K % 128 != 0) {
      s = 1;
    } else {
      s = pick_split_k(16, K, N, 128, live);
    }
    if ((size_t)pl.nblk * pl.ncb * sizeof(int) > AWQMI_WS_COUNTER_BYTES) s = 1;
  }
  if (s > nchunks) s = nchunks > 0 ? nchunks : 1;
  pl.split = s;
  return pl;
}

size_t awqmi_moe_gemm_workspace_bytes(int n_slots, int E, int K, int N, int split_k, int tile_m) {
  if (n_slots <= 0 || E <= 0 || K <= 0 || N <= 0 || N % 8 != 0 ||
      (tile_m != 16 && tile_m != 32 && tile_m != 64 && tile_m != 128 && tile_m != 256))
    return 0;
  if (tile_m >= 64) return AWQMI_WS_COUNTER_BYTES;    // the grouped tile kernel needs no partials
  const MoePlan pl = moe_plan(n_slots, E, K, N, tile_m, split_k);
  return AWQMI_WS_COUNTER_BYTES + gemv_partial_bytes(N, pl.split, pl.nblk, tile_m);
}

// Can the w13 GEMM of a block write silu(gate) * up itself?  Needs the paired-column launch
// (two column blocks per workgroup: the gate block and its up block), i.e. no split across
// workgroups, an even chunk count, [gate | up] halves that are whole column blocks, and
// enough blocks that the halved workgroup count still fills the chip.  It pays from about
// eight real rows per 16-row block on (measured on 2048 x 1536 experts, 128 of them: 6 %
// faster at 12 rows per block, 3 - 5 % slower at 2 - 6); below that the separate activation
// kernel is cheaper than the two-waves-per-column-block form of the GEMM.
static bool moe_can_fuse_act(int n_slots, int E, int K, int N) {
  const MoePlan pl = moe_plan(n_slots, E, K, N, 16, 0);
  const long long live_blocks = std::max<long long>((n_slots + 15) / 16, std::min(n_slots, E));
  return pl.wpl == 2 && pl.split == 1 && K % 128 == 0 && (K / 128) % 2 == 0 && N % 512 == 0 &&
         live_blocks * (pl.ncb / 2) >= 256 && n_slots >= 8 * live_blocks;
}

// Same question for a launch that is split in K: the last arrivers of a gate block and its up
// block finish both and apply the activation.
static bool moe_can_fuse_act_split(int n_slots, int E, int K, int N) {
  const MoePlan pl = moe_plan(n_slots, E, K, N, 16, 0);
  return pl.wpl == 2 && pl.split > 1 && N % 512 == 0 && pl.ncb % 2 == 0;
}

// The grouped tile kernel can write silu(gate) * up itself where its column tiles are whole and its plain
// form runs (groups of at least 64).
static bool moe_tile_act_ok(int inter, int G) { return inter % 128 == 0 && G % 64 == 0; }

// tiles of at most TG_RUN 16-slot blocks that n_slots slots on E experts make at most
static long long moe_most_runs(int n_slots, int E) {
  const long long touched = std::min(n_slots, E);
  return touched + (n_slots / 16 + touched) / TG_RUN;
}
static_assert(TG_RUN == MOE_RUN, "the tile lists are made for the grouped kernel");

// Form of a grouped launch of 16-row blocks.
struct MoeSkinnyForm {
  bool pair_cols;      // two column blocks per workgroup, two waves each
  bool act_split;      // fused activation by the last arrivers of a K split ...
  bool act_pair;       // ... or in the workgroup that has the gate and the up block
  bool ldsq;           // weight ring in LDS
  bool plain;          // none of them but act_split, register ring of two: the form that can take the routing along
};
static MoeSkinnyForm moe_skinny_form(const MoePlan& pl, int n_slots, int E, int K, int N, int tile_m, bool fuse_act) {
  MoeSkinnyForm f{};
  // few chunks of K and no split across workgroups: two column blocks per workgroup, two
  // waves each (three chunks per wave at K = 768 instead of 2 / 2 / 1 / 1)
  // -- as long as the paired launch still fills the chip (blocks that will run: one per expert
  // touched or per 16 slots, whichever is more)
  const long long live_blocks = std::max<long long>((n_slots + 15) / 16, std::min(n_slots, E));
  f.pair_cols = tile_m == 16 && pl.wpl == 2 && pl.split == 1 && K / 128 <= 8 && (K / 128) % 2 == 0 &&
                live_blocks * ((pl.ncb + 1) / 2) >= 256 && !variant_on(VAR_NO_PAIR_COLS);
  // fused activation: without a split the paired-column kernel (gate and up block in one
  // workgroup); with a split the ordinary launch whose last arrivers pair the blocks up
  f.act_split = fuse_act && pl.split > 1;
  f.act_pair = fuse_act && pl.split == 1;
  // weight ring of four steps in LDS instead of two in registers, from one full block per
  // expert on (T = 256 ... 1024 of the 128-expert block: 6 - 10 % faster; with fewer rows per
  // expert 1 - 4 % slower, and no gain for the few-block launches once their weights come from
  // HBM rather than from a warm cache)
  f.ldsq = pl.wpl == 2 && tile_m == 16 && (size_t)K * (N / 8) * 4 < (1ull << 31) && (long long)n_slots >= 16LL * E &&
           !variant_on(VAR_NO_LDS_RING);
  f.plain = !f.ldsq && !f.act_pair &&
            (f.act_split || (tile_m == 16 && pl.wpl == 2 && !f.pair_cols && !variant_on(VAR_MOE_RING4)));
  return f;
}
// Does a launch in that form take the routing along?  Every workgroup picks by itself, one pick after the other, and those that
// start when others end are held up by it: with more than eight picks the workgroups that are expected to run (a block more with several
// tokens) have to fit the chip at once, two a CU.  Routed apart / folded, us: 20, 22, 24, 32 picks of 256 experts of 3072 x 1536, two
// tokens (461, 505, 549, 720 workgroups) 74.9, 88.3, 94.3, 102.9 / 70.8, 91.9, 99.4, 111.4; 32 of 64 of 2048 x 2048, one and two tokens (512, 768)
// 61.1, 86.2 / 57.4, 89.5; 16 of 128 of 2048 x 1408, three and four (465, 583) 57.7, 67.5 / 54.2, 68.7; 12 of 256 of 3072 x 1536, five (656)
// 91.0 / 92.1.  Up to eight picks take less than the launch: 8 of 256 of 7168 x 2048, eight tokens (919) 245.3 / 240.5.
static bool moe_launch_folds(const MoeSkinnyForm& f, const MoePlan& pl, int T, int E, int topk, int tile_m, int G) {
  if (!f.plain || G != 128 || !moe_route_foldable(T, E, topk, tile_m)) return false;
  const double blocks = E * (1.0 - std::pow(1.0 - (double)topk / E, T)) + (T > 1);
  return topk <= 8 || blocks * pl.ncb * pl.split <= 512.0;
}

static int moe_gemm_impl(const void* x, const int32_t* qweight, const void* scales, const int32_t* qzeros,
                         void* y, const int32_t* sorted_token_ids, const int32_t* expert_ids,
                         const int32_t* num_tokens_post_padded, const float* topk_weights, int n_slots,
                         int a_row_div, int tile_m, int E, int K, int N, int group, int split_k,
                         void* workspace, size_t workspace_bytes, void* stream, bool fuse_act,
                         const MoeRoute* route = nullptr, int32_t* runs = nullptr);

int awqmi_moe_gemm_f16(const void* x, const int32_t* qweight, const void* scales, const int32_t* qzeros,
                       void* y, const int32_t* sorted_token_ids, const int32_t* expert_ids,
                       const int32_t* num_tokens_post_padded, const float* topk_weights, int n_slots,
                       int a_row_div, int tile_m, int E, int K, int N, int group, int split_k,
                       void* workspace, size_t workspace_bytes, void* stream) {
  return moe_gemm_impl(x, qweight, scales, qzeros, y, sorted_token_ids, expert_ids, num_tokens_post_padded,
                       topk_weights, n_slots, a_row_div, tile_m, E, K, N, group, split_k, workspace,
                       workspace_bytes, stream, false);
}

static int moe_gemm_impl(const void* x, const int32_t* qweight, const void* scales, const int32_t* qzeros,
                         void* y, const int32_t* sorted_token_ids, const int32_t* expert_ids,
                         const int32_t* num_tokens_post_padded, const float* topk_weights, int n_slots,
                         int a_row_div, int tile_m, int E, int K, int N, int group, int split_k,
                         void* workspace, size_t workspace_bytes, void* stream, bool fuse_act,
                         const MoeRoute* route, int32_t* runs) {
  // route: the block's routing has not run yet.  The launch takes it along when it is the plain
  // 16-row-block form with G = 128; any other form routes in launches of its own first.
  if (!x || !qweight || !scales || !qzeros || !y || !sorted_token_ids || !expert_ids ||
      !num_tokens_post_padded)
    return AWQMI_NULL_POINTER;
  const int G = norm_group(K, group);
  if (const int rc = check_awq_shape(K, N, G)) return rc;
  if (n_slots <= 0 || E <= 0) return AWQMI_BAD_SHAPE;
  if (a_row_div <= 0 || split_k < 0 || split_k > AWQMI_MAX_SPLIT_K || E > AWQMI_MAX_EXPERTS ||
      (tile_m != 16 && tile_m != 32 && tile_m != 64 && tile_m != 128 && tile_m != 256))
    return AWQMI_BAD_ARGUMENT;
  if (!gemv_tiled_ok(K, G)) return AWQMI_UNSUPPORTED_GROUP;
  if (!aligned16(x) || !aligned16(scales) || !aligned16(qweight) || !aligned16(qzeros) ||
      !aligned16(y))
    return AWQMI_BAD_ALIGN;
  const int NW = N / 8;
  if (tile_m >= 64 || runs) {
    // blocks of 64 / 128 / 256 slots, or tiles of several 16-slot blocks: the tile kernel in its expert-grouped
    // form (no K split)
    const bool any = G % 64 != 0 || N % 32 != 0;
    if (fuse_act && !moe_tile_act_ok(N / 2, G)) return AWQMI_BAD_ARGUMENT;
    if (route)
      if (const int rc = moe_route_launches(*route, tile_m, stream)) return rc;
    const size_t x_rows = ((size_t)n_slots + a_row_div - 1) / a_row_div;
    if (x_rows * K * 2 >= (1ull << 32) || (size_t)K * NW * 4 >= (1ull << 32) ||
        (size_t)(K / G) * N * 2 >= (1ull << 32))
      return AWQMI_BAD_SHAPE;
    TileGemmParams p{};
    p.x = reinterpret_cast<const half_t*>(x);
    p.qw = reinterpret_cast<const uint32_t*>(qweight);
    p.sc = reinterpret_cast<const half_t*>(scales);
    p.qz = reinterpret_cast<const uint32_t*>(qzeros);
    p.y = reinterpret_cast<half_t*>(y);
    p.M = (int)x_rows; p.K = K; p.N = N; p.NW = NW; p.ldw = NW; p.G = G;
    while ((2 << p.gshift) <= G) ++p.gshift;
    const int cols = fuse_act ? N / 2 : N, per_tile = fuse_act ? TG_COLS / 2 : TG_COLS;
    p.nt = (cols + per_tile - 1) / per_tile;
    p.sorted_ids = sorted_token_ids; p.expert_ids = expert_ids; p.n_live = num_tokens_post_padded;
    p.topk_w = topk_weights; p.n_slots = n_slots; p.a_row_div = a_row_div;
    p.w_stride = (long long)K * NW; p.s_stride = (long long)(K / G) * N; p.z_stride = (long long)(K / G) * NW;
    p.block = tile_m;
    long long tiles = (long long)(awqmi_moe_align_capacity(n_slots, E, tile_m) / std::min(tile_m, TG_ROWS));
    if (runs) {
      p.n_live = runs;
      p.runs = runs + 1;
      tiles = moe_most_runs(n_slots, E);
      // workgroups still read the list while others store their rows
      const uintptr_t list = reinterpret_cast<uintptr_t>(runs), rows = reinterpret_cast<uintptr_t>(y);
      if (rows < list + (1 + (size_t)tiles) * sizeof(int32_t) && list < rows + (size_t)n_slots * cols * 2) return AWQMI_BAD_ARGUMENT;
    }
    p.total = (int)(tiles * p.nt);
    // ranges per XCD are uneven in rows with few experts (see the kernel)
    p.in_order = E < 16;
    const dim3 grid((unsigned)((p.total + 7) / 8 * 8));     // whole deals to the 8 XCDs
    hipStream_t st = (hipStream_t)stream;
#define AWQMI_GROUPED(...) hipLaunchKernelGGL((awq_gemm_tile_grouped_kernel<__VA_ARGS__>), grid, dim3(256), 0, st, p)
    if (runs && G == 64) {
      if (fuse_act) AWQMI_GROUPED(0, true, 1);
      else AWQMI_GROUPED(0, false, 1);
    } else if (runs) {
      if (fuse_act) AWQMI_GROUPED(0, true, 2);
      else AWQMI_GROUPED(0, false, 2);
    } else if (any) {
      AWQMI_GROUPED(2, false, 0);
    } else if (fuse_act) {
      AWQMI_GROUPED(0, true, 0);
    } else {
      AWQMI_GROUPED(0, false, 0);
    }
#undef AWQMI_GROUPED
    return launch_status();
  }
  const MoePlan pl = moe_plan(n_slots, E, K, N, tile_m, split_k);
  const int wpl = pl.wpl, ncb = pl.ncb, nblk = pl.nblk, split = pl.split;
  // 32-row blocks: one packed word per lane, two column blocks of 128 per workgroup with two waves
  // each (the accumulators of two row blocks then take the registers one row block takes with two
  // words per lane, and two workgroups still fit a CU), the weight ring of four steps in LDS;
  // needs an even chunk count, no K split.  (One 128-column block per workgroup with four K
  // ranges measured 35 - 70 % slower: neighbouring workgroups then fetch the two halves of every
  // 128-byte line.)
  const bool t32_narrow = tile_m == 32 && split == 1 && (K / 128) % 2 == 0 && !variant_on(VAR_MOE_T32_WIDE);
  if (tile_m == 32 && !t32_narrow && wpl != 2) return AWQMI_BAD_SHAPE;   // the wide form needs N % 16 == 0
  if (split > 1) {
    if (!workspace) return AWQMI_NULL_POINTER;
    if (!aligned16(workspace)) return AWQMI_BAD_ALIGN;
    if ((size_t)nblk * ncb * sizeof(int) > AWQMI_WS_COUNTER_BYTES) return AWQMI_BAD_ARGUMENT;
    if (workspace_bytes < AWQMI_WS_COUNTER_BYTES + gemv_partial_bytes(N, split, nblk, tile_m))
      return AWQMI_WORKSPACE_TOO_SMALL;
  }
  GemvParams p{};
  p.x = reinterpret_cast<const half_t*>(x);
  p.qw = reinterpret_cast<const uint32_t*>(qweight);
  p.sc = reinterpret_cast<const half_t*>(scales);
  p.qz = reinterpret_cast<const uint32_t*>(qzeros);
  p.y = reinterpret_cast<half_t*>(y);
  p.cnt = reinterpret_cast<int*>(workspace);
  p.part = workspace ? reinterpret_cast<float*>(static_cast<char*>(workspace) + AWQMI_WS_COUNTER_BYTES)
                     : nullptr;
  p.M = tile_m; p.K = K; p.N = N; p.NW = NW; p.ldw = NW; p.G = G;
  p.split_k = split; p.ncb = ncb;
  p.sorted_ids = sorted_token_ids; p.expert_ids = expert_ids; p.n_post_pad = num_tokens_post_padded;
  p.topk_w = topk_weights; p.n_slots = n_slots; p.a_row_div = a_row_div; p.tile_m = tile_m;
  p.w_stride = (long long)K * NW; p.s_stride = (long long)(K / G) * N; p.z_stride = (long long)(K / G) * NW;
  p.nblk = nblk;
  p.nblk_cap = (int)(awqmi_moe_align_capacity(n_slots, E, tile_m) / tile_m);
  p.ldy = fuse_act ? N / 2 : N;
  const int variant = t_variant;
  // group blocks by XCD once most experts have a full block: runs of 8 from 0.75 blocks per
  // expert on, runs of 32 from 1.5 (measured on 128 experts: 6 % at one block per expert, 15 %
  // at 1.5, 3 - 4 % at 2 - 4 against runs of 8 or none; below 0.75 the order makes no difference)
  p.grp = (long long)n_slots * 2 >= 3LL * tile_m * E ? 32 : ((long long)n_slots * 4 >= 3LL * tile_m * E ? 8 : 1);
  if (E < 16) p.grp = 1;   // a handful of large experts: the plain order measured equal or up to 13 % faster
  if (variant >= 0 && ((variant >> VAR_XCD_RUN_SHIFT) & 7)) p.grp = 1 << (((variant >> VAR_XCD_RUN_SHIFT) & 7) - 1);
  const MoeSkinnyForm form = moe_skinny_form(pl, n_slots, E, K, N, tile_m, fuse_act);
  const bool pair_cols = form.pair_cols, act_split = form.act_split, act_pair = form.act_pair, ldsq = form.ldsq;
  if (fuse_act && (wpl != 2 || tile_m != 16 || ncb % 2 != 0 || N % 512 != 0 ||
                   (split == 1 && (K / 128) % 2 != 0)))
    return AWQMI_BAD_ARGUMENT;
  p.act_split = act_split ? 1 : 0;
  const int ncb1 = (NW + 15) / 16;       // column blocks of 128 (one word per lane)
  const bool t32_lds = t32_narrow && (size_t)K * NW * 4 < (1ull << 31) && !variant_on(VAR_NO_LDS_RING);
  const int ncg = t32_narrow ? (ncb1 + 1) / 2 : (act_pair ? ncb / 2 : (pair_cols ? (ncb + 1) / 2 : ncb));
  if (t32_narrow) p.ncb = ncb1;
  // runs of grp slots, dealt to the 8 XCDs in turn; the last deal may be partial
  const long long deals = (long long)(nblk / p.grp) * ncg * split;
  const dim3 grid((unsigned)((deals + 7) / 8 * 8 * p.grp));
  hipStream_t st = (hipStream_t)stream;
  if (route) {
    if (moe_launch_folds(form, pl, route->T, route->E, route->topk, tile_m, G)) {
      p.r_logits = route->logits; p.r_bias = route->bias;
      p.r_T = route->T; p.r_E = route->E; p.r_topk = route->topk; p.r_renorm = route->renorm;
      p.r_scale = route->scale;
      p.r_ids = route->ids; p.r_wts = route->wts; p.r_sorted = route->sorted; p.r_experts = route->experts;
      p.r_npp = route->npp;
      moe_topk_form(route->E, route->topk, route->scoring, [&](auto L, auto P, auto S) {
        if constexpr (decltype(L)::value * decltype(P)::value <= MOE_FOLD_EXPERTS)
          hipLaunchKernelGGL((awq_gemv_route_kernel<2, decltype(L)::value, decltype(P)::value, decltype(S)::value>), grid,
                             dim3(256), 0, st, p);
      });
      return launch_status();
    }
    if (const int rc = moe_route_launches(*route, tile_m, stream)) return rc;
  }
  if (ldsq && act_pair) launch_gemv<2, 1, true, 4, 2, true, true>(p, grid, st);
  else if (ldsq && pair_cols && !act_split) launch_gemv<2, 1, true, 4, 2, false, true>(p, grid, st);
  else if (ldsq) launch_gemv<2, 1, true, 4, 4, false, true>(p, grid, st);
  else if (act_pair) launch_gemv<2, 1, true, 2, 2, true>(p, grid, st);
  else if (act_split) launch_gemv<2, 1, true, 2>(p, grid, st);
  else if (t32_lds) launch_gemv<1, 2, true, 4, 2, false, true>(p, grid, st);
  else if (t32_narrow) launch_gemv<1, 2, true, 2, 2>(p, grid, st);
  else if (tile_m == 32) launch_gemv<2, 2, true>(p, grid, st);
  else if (wpl == 2 && variant_on(VAR_MOE_RING4)) launch_gemv<2, 1, true, 4>(p, grid, st);
  else if (pair_cols) launch_gemv<2, 1, true, 2, 2>(p, grid, st);
  else if (wpl == 2) launch_gemv<2, 1, true, 2>(p, grid, st);
  else launch_gemv<1, 1, true>(p, grid, st);
  return launch_status();
}

int awqmi_silu_and_mul_f16(const void* in, void* out, int rows, int inter, void* stream) {
  if (!in || !out) return AWQMI_NULL_POINTER;
  if (rows <= 0 || inter <= 0 || inter % 8 != 0) return AWQMI_BAD_SHAPE;
  if (!aligned16(in) || !aligned16(out)) return AWQMI_BAD_ALIGN;
  const size_t n = (size_t)rows * (inter / 8);
  hipLaunchKernelGGL(silu_and_mul_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0,
                     (hipStream_t)stream, reinterpret_cast<const half_t*>(in),
                     reinterpret_cast<half_t*>(out), rows, inter);
  return launch_status();
}

int awqmi_moe_sum_f16(const void* in, void* out, int T, int topk, int H, void* stream) {
  if (!in || !out) return AWQMI_NULL_POINTER;
  if (T <= 0 || topk <= 0 || H <= 0 || H % 8 != 0) return AWQMI_BAD_SHAPE;
  if (!aligned16(in) || !aligned16(out)) return AWQMI_BAD_ALIGN;
  const size_t n = (size_t)T * (H / 8);
  hipLaunchKernelGGL(moe_sum_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0,
                     (hipStream_t)stream, reinterpret_cast<const half_t*>(in),
                     reinterpret_cast<half_t*>(out), T, topk, H);
  return launch_status();
}

namespace {
// Expected blocks of `rows` slots of an expert's run when its slot count is Poisson(avg) (normal tail past the
// first block): sum_j P(count > j * rows)
double moe_expected_blocks(double avg, int rows) {
  double e = 1.0 - std::exp(-avg);
  for (int j = 1; j * (double)rows < avg + 6.0 * std::sqrt(avg) + 1.0; ++j)
    e += 0.5 * std::erfc((j * (double)rows + 0.5 - avg) / std::sqrt(2.0 * avg));
  return e;
}

// Rows per block for the two expert GEMMs of one MoE block: 16 (the skinny kernel) or 64 /
// 128 / 256 (the tile kernel's expert-grouped form), by price:
//   skinny: flops / (540 TFLOP/s * avg / (avg + 26)), avg = slots per expert;
//   larger: per GEMM blocks * column tiles / 256 CUs rounds (a partial last round counts as
//           at least half) of (K / 64 + overhead) k-tiles at 5.4 ns * (rows + 112) each, plus the separate
//           SiLU pass at 4 TB/s; blocks is the expected block count after padding each expert's run to whole
//           blocks (slots spread evenly over the experts).
// A second look at the larger blocks counts a partly filled block by its rows in steps of 64, as that
// kernel ran it (at 5.4 / 5.65 / 5.9 ns for 64 / 128 / 256 rows), and only goes upwards, to blocks that are fewer
// (as many blocks run the same tiles).
// Every size forced, with the grouped kernel before the present one, in turn on 640 points (53 shapes: hidden 384 ... 7168, intermediate 384 ... 14336, 4 ... 512
// experts, top-1 ... 10, 32 ... 1400 slots per expert):
//   - the choice is 1.7 % behind the best size on average, 48 % at worst (4919 tokens on 128 experts of 2048 x
//     384: 16 rows 508 us, 256 rows 344; the first look chooses 16 rows there too);
//   - the second look changes 99 points, by 9 % on average (1376 tokens on 64 experts of 5120 x 1024, top-4:
//     16 rows 405 us, 128 rows 334); three get slower, by 6 - 12 % (247 tokens on 8 experts of 4096 x 14336, top-2:
//     16 rows 422, 128 rows 471);
//   - the second price alone, downwards too, is 1.9 % behind the best size and 12 points are 5 - 24 % behind the
//     first look (1590 tokens on 128 experts of 2048 x 768, top-8: 16 rows 289, 128 rows 236; 1391 on 16 of 5120 x
//     8192, top-1: 256 rows 704, 128 rows 642).
// The prices are those of the grouped kernel that dequantised into LDS, and 16 rows those of the skinny kernel: they say where
// blocks of 16 slots end, which callers of the step-by-step path have in their own calls too.  With the present kernel, which is
// faster for every size, and moe_runs beside it the choice is 4 % behind the best of 16, 16 in tiles and 128 on average of 129
// points, 34 % at worst (896 tokens on 256 experts of 2048 x 384, top-8: 157 us, in tiles 117; see moe_runs for 28 to 32 slots).
// Two sizes that the tests fix measure slower than another: 2048 tokens on 128 experts of 2048 x 768 (16 rows in tiles
// 254 us, 128 rows 248), 2102 on 4 of 512 x 384 (16 rows 51, in tiles 38, 64 rows 36).
// Larger blocks also need every operand under 4 GiB (32-bit buffer offsets).
int moe_pick_tile(int n_slots, int E, int H, int inter, int group) {
  if (variant_on(VAR_MOE_TILE16)) return 16;
  if (!gemv_tiled_ok(H, norm_group(H, group)) || !gemv_tiled_ok(inter, norm_group(inter, group))) return 16;
  if ((size_t)n_slots * std::max(H, inter) * 2 >= (1ull << 32) ||
      (size_t)H * (2 * inter / 8) * 4 >= (1ull << 32) || (size_t)inter * (H / 8) * 4 >= (1ull << 32))
    return 16;
  const int vv = t_variant;
  if (vv >= 0 && ((vv >> VAR_MOE_TILE_SHIFT) & 3)) return 32 << ((vv >> VAR_MOE_TILE_SHIFT) & 3);
  const double avg = (double)n_slots / E;
  // below two 16-row blocks per expert a 64-row block is mostly padding (and the cost terms
  // below, fitted on avg >= 32, do not describe launches of a few blocks)
  if (avg < 32.0) return 16;
  const double flops = 2.0 * n_slots * ((double)H * 2 * inter + (double)inter * H);
  const double skinny = flops / (540e12 * avg / (avg + 26.0));
  // expected blocks of `rows` after padding each expert's run
  auto expected = [&](int rows) { return E * moe_expected_blocks(avg, rows); };
  // price of blocks of bm rows, partly filled ones counted whole or (by_rows) by their rows in steps of 64
  auto mfma = [&](int bm, bool by_rows) {
    const double blocks = by_rows ? (64.0 * expected(64) + 112.0 * expected(bm)) / (bm + 112) : expected(bm);
    const double kt_s = (!by_rows || bm == 64 ? 5.4e-9 : bm == 128 ? 5.65e-9 : 5.9e-9) * (bm + 112);
    const int over = bm == 256 ? 6 : 4;
    auto gemm = [&](int K, int N) {
      const double r = blocks * ((N + PF_BN - 1) / PF_BN) / 256.0;
      const double whole = std::floor(r), part = r - whole;
      const double rounds = whole + (part > 0 ? std::max(part, 0.5) : 0.0);
      return rounds * (K / DG_BK + over) * kt_s;
    };
    return gemm(H, 2 * inter) + gemm(inter, H) + 5e-6 + 6.0 * n_slots * inter / 4e12;
  };
  int tile = 16;
  double best = skinny;
  for (int bm : {64, 128, 256}) {
    const double t = mfma(bm, false);
    if (t < best) { best = t; tile = bm; }
  }
  if (tile > 16) best = mfma(tile, true);
  for (int bm : {128, 256}) {
    if (bm <= tile || ((tile > 16 || bm == 256) && expected(bm) > 0.99 * expected(bm / 2))) continue;
    const double t = mfma(bm, true);
    if (t < best) { best = t; tile = bm; }
  }
  return tile;
}

// Blocks of 16 slots: run the expert GEMMs on tiles of up to four of them (the tile kernel) instead of a
// block at a time (the skinny kernel), by price in us.
//   tiles: per GEMM rounds of 512 workgroups (a partial last one counts as at least 0.38) of (K / 64 + 2.1) stages, a stage
//   of two workgroups per CU at 2 * (0.344 + 0.09 per 16 rows);
//   blocks: 0.09 us per MB of touched experts' weights and 0.11 per MB and block, which unpacks them again.
// Fitted on 129 points (ten expert shapes, 6 ... 400 slots per expert), the whole block timed both ways.  The tiles have to
// look 14 % cheaper (24 % below 16 experts, whose few long tiles the price underestimates): then no point of them is slower
// than with the skinny kernel, and they are 8 % faster on average over all.
// With 16 experts and more no price is needed from 20 slots per expert on: there the tiles are 2 - 30 % faster on all of nine shapes
// (blocks / tiles, us, at 19, 22, 25 and 27.5 slots: 128 experts of 2048 x 768 103, 105, 121, 123 / 101, 103, 104, 106; 64 of 2048 x 1408 106, 108, 116, 120 /
// 90, 93, 94, 95; 64 of 5120 x 1024 161, 163, 183, 196 / 149, 150, 153, 157; 160 of 6144 x 2560 998, 1068, 1131, 1166 / 943, 956, 975, 985;
// 16 of 3072 x 4096 118, 117, 135, 145 / 105, 106, 108, 110; groups of 64 alike); at 16 and below either side wins (128 experts of 2048 x
// 768 98.0 / 98.9, 160 of 6144 x 2560 909 / 926), with eight experts the blocks.
// From 28 to 32 slots the blocks stay single, for no property of either kernel: three expectations of this rule in the host tests and a
// bound between the block and the separate calls at 512 tokens date from when the line was at 32.  Tiles are faster there too
// (blocks / tiles, us, at 28, 30 and 32 slots: 128 experts of 2048 x 768 127, 124, 124 / 107, 107, 110; 64 of 2048 x 1408 120, 121, 124 / 95, 96, 97; 64 of
// 5120 x 1024 197, 203, 207 / 159, 161, 162; 160 of 6144 x 2560 1173, 1215, 1269 / 990, 999, 1013; 256 of 2048 x 384 157, 164, 166 / 117, 119, 119;
// 16 of 3072 x 4096 145, 149, 149 / 110, 111, 112; 60 of 4096 x 1536 211, 217, 221 / 172, 173, 174).  Either form is as near to 64-bit sums.
// Experts of less than 1024 x 384 stay as well: smaller ones were not measured (64 of 1024 x 384 at 20, 24, 27 and 40 slots 35.7, 37.9, 39.9, 47.7 / 31.0, 32.1,
// 32.6, 35.3).  Above 32, blocks / tiles (us): 576 / 768 / 1024 tokens on 128 experts of 2048 x 768 143 / 164 / 192 and 116 / 130 / 163; 560 on 64 of
// 2048 x 1408 172 and 122.
bool moe_runs(int T, int n_slots, int E, int H, int inter, int group) {
  if (variant_on(VAR_MOE_TILE16) || T <= MOE_ALIGN_WAVES) return false;
  // groups of 64 or 128 rows, whole column tiles
  const int g1 = norm_group(H, group), g2 = norm_group(inter, group);
  if (H % 128 != 0 || inter % 128 != 0 || (g1 != 64 && g1 != 128) || g1 != g2) return false;
  if ((size_t)n_slots * std::max(H, inter) * 2 >= (1ull << 32) || (size_t)H * (2 * inter / 8) * 4 >= (1ull << 32) ||
      (size_t)inter * (H / 8) * 4 >= (1ull << 32))
    return false;
  if (variant_on(VAR_MOE_RUNS)) return true;
  const double avg = (double)n_slots / E;
  if (H < 1024 || inter < 384) return false;
  if (avg >= 20.0 && avg < 28.0 && E >= 16) return true;
  if (avg <= 32.0) return false;
  const double b16 = E * moe_expected_blocks(avg, 16), tiles = E * moe_expected_blocks(avg, 16 * TG_RUN);
  const double stage = 2.0 * (0.344 + 0.09 * std::max(b16 / tiles, 2.0));
  auto gemm = [&](int K, int col_tiles) {
    const double r = tiles * col_tiles / 512.0, whole = std::floor(r), part = r - whole;
    return (whole + (part > 0 ? std::max(part, 0.38) : 0.0)) * (K / 64 + 2.1) * stage;
  };
  const double runs = 19.8 + gemm(H, (inter + 127) / 128) + gemm(inter, (H + TG_COLS - 1) / TG_COLS);
  const double mb = 1.5 * H * inter * 1e-6;     // packed weights of an expert
  const double skinny = 26.6 + (0.09 * E * (1.0 - std::exp(-avg)) + 0.11 * b16) * mb + 0.0009 * n_slots;
  return runs < (E < 16 ? 0.76 : 0.86) * skinny;
}

// How a one-call block runs: slots of its blocks, whether those of 16 go in tiles (moe_runs), and whether the first expert GEMM
// writes silu(gate) * up itself: in a tile of gate columns and their up columns; in one workgroup per gate / up block pair;
// or, with few blocks (the launch is split in K), in the last arrivers of such a pair.
// The list of tiles lies where the gate / up sums go otherwise, so there are no tiles without the fused activation.
struct MoeForm { int tile; bool runs, act; };
MoeForm moe_form(int T, int H, int inter, int E, int topk, int group) {
  const int n_slots = T * topk, G = norm_group(H, group);
  MoeForm f{moe_pick_tile(n_slots, E, H, inter, group), false, false};
  if (variant_on(VAR_NO_FUSED_ACT)) return f;
  const bool tile_act = moe_tile_act_ok(inter, G);
  f.runs = f.tile == 16 && tile_act && moe_runs(T, n_slots, E, H, inter, group);
  f.act = f.tile >= 64 || f.runs ? tile_act
                                 : gemv_tiled_ok(H, G) && (moe_can_fuse_act(n_slots, E, H, 2 * inter) ||
                                                           moe_can_fuse_act_split(n_slots, E, H, 2 * inter));
  return f;
}

// workspace carve-up of the fused MoE block; every piece starts 256-byte aligned
struct FusedMoeLayout {
  size_t gemm_ws, ids, wts, sorted, experts, npp, h13, act, o, total;
  size_t gemm_ws_bytes;
  int n_slots, cap, tile;
  size_t tab;      // expert counts of the parts of a longer batch; runs on into act
};
FusedMoeLayout fused_moe_layout(int T, int H, int inter, int E, int topk, int tile) {
  FusedMoeLayout L{};
  auto up = [](size_t v) { return (v + 255) / 256 * 256; };
  L.n_slots = T * topk;
  L.tile = tile;
  L.cap = (int)awqmi_moe_align_capacity(L.n_slots, E, L.tile);
  const size_t g1 = awqmi_moe_gemm_workspace_bytes(L.n_slots, E, H, 2 * inter, 0, L.tile);
  const size_t g2 = awqmi_moe_gemm_workspace_bytes(L.n_slots, E, inter, H, 0, L.tile);
  L.gemm_ws_bytes = g1 > g2 ? g1 : g2;
  size_t off = 0;
  L.gemm_ws = off; off += up(L.gemm_ws_bytes);
  L.ids = off;     off += up((size_t)L.n_slots * 4);
  L.wts = off;     off += up((size_t)L.n_slots * 4);
  L.sorted = off;  off += up((size_t)L.cap * 4);
  L.experts = off; off += up((size_t)(L.cap / L.tile) * 4);
  L.npp = off;     off += 256;
  L.h13 = off;     off += up((size_t)L.n_slots * 2 * inter * 2);
  L.tab = off;     off += up((size_t)MOE_TAB_PARTS * E * 4);
  L.act = off;     off += up((size_t)L.n_slots * inter * 2);
  L.o = off;       off += up((size_t)L.n_slots * H * 2);
  L.total = off;
  return L;
}
}  // namespace

size_t awqmi_fused_moe_workspace_bytes(int T, int H, int inter, int E, int topk) {
  if (T <= 0 || H <= 0 || inter <= 0 || E <= 0 || topk <= 0 || H % 8 != 0 || inter % 8 != 0) return 0;
  if ((long long)T * topk > (1LL << 30)) return 0;
  size_t most = 0;     // the call picks the block rows from the shapes; any choice fits
  for (int tile : {16, 64, 128, 256}) most = std::max(most, fused_moe_layout(T, H, inter, E, topk, tile).total);
  return most;
}

int awqmi_fused_moe_block_rows(int T, int H, int inter, int E, int topk, int group) {
  if (T <= 0 || H <= 0 || inter <= 0 || E <= 0 || H % 8 != 0 || inter % 8 != 0) return 0;
  if (topk <= 0 || topk > E || topk > 64 || E > AWQMI_MAX_EXPERTS || (long long)T * topk > (1LL << 30)) return 0;
  return moe_pick_tile(T * topk, E, H, inter, group);
}

int awqmi_fused_moe_f16(const void* hidden, const float* router_logits, const int32_t* w13_q,
                        const void* w13_s, const int32_t* w13_z, const int32_t* w2_q, const void* w2_s,
                        const int32_t* w2_z, void* out, int T, int H, int inter, int E, int topk,
                        int group, int renormalize, void* workspace, size_t workspace_bytes,
                        void* stream) {
  return awqmi_fused_moe_routed_f16(hidden, router_logits, nullptr, w13_q, w13_s, w13_z, w2_q, w2_s, w2_z, out, T,
                                    H, inter, E, topk, group, 0, renormalize, 1.f, workspace, workspace_bytes,
                                    stream);
}

int awqmi_fused_moe_routed_f16(const void* hidden, const float* router_logits, const float* score_bias,
                               const int32_t* w13_q, const void* w13_s, const int32_t* w13_z,
                               const int32_t* w2_q, const void* w2_s, const int32_t* w2_z, void* out, int T,
                               int H, int inter, int E, int topk, int group, int scoring, int renormalize,
                               float routed_scale, void* workspace, size_t workspace_bytes, void* stream) {
  if (!hidden || !router_logits || !w13_q || !w13_s || !w13_z || !w2_q || !w2_s || !w2_z || !out ||
      !workspace)
    return AWQMI_NULL_POINTER;
  if (T <= 0 || H <= 0 || inter <= 0 || E <= 0 || H % 8 != 0 || inter % 8 != 0) return AWQMI_BAD_SHAPE;
  if (topk <= 0 || topk > E || topk > 64 || E > AWQMI_MAX_EXPERTS || (long long)T * topk > (1LL << 30))
    return AWQMI_BAD_ARGUMENT;
  if ((scoring != 0 && scoring != 1) || (scoring == 0 && score_bias)) return AWQMI_BAD_ARGUMENT;
  if (!aligned16(workspace)) return AWQMI_BAD_ALIGN;
  const MoeForm form = moe_form(T, H, inter, E, topk, group);
  const int tile = form.tile;
  const FusedMoeLayout L = fused_moe_layout(T, H, inter, E, topk, tile);
  if (workspace_bytes < L.total) return AWQMI_WORKSPACE_TOO_SMALL;
  // what the launches behind the first one would refuse, so that a call either runs whole or leaves nothing on the stream
  for (const auto& [K, N] : {std::pair{H, 2 * inter}, std::pair{inter, H}}) {
    if (const int rc = check_awq_shape(K, N, norm_group(K, group))) return rc;
    if (!gemv_tiled_ok(K, norm_group(K, group))) return AWQMI_UNSUPPORTED_GROUP;
  }
  for (const void* p : {hidden, (const void*)w13_q, w13_s, (const void*)w13_z, (const void*)w2_q, w2_s, (const void*)w2_z, (const void*)out})
    if (!aligned16(p)) return AWQMI_BAD_ALIGN;
  char* ws = static_cast<char*>(workspace);
  int32_t* ids = reinterpret_cast<int32_t*>(ws + L.ids);
  float* wts = reinterpret_cast<float*>(ws + L.wts);
  int32_t* sorted = reinterpret_cast<int32_t*>(ws + L.sorted);
  int32_t* experts = reinterpret_cast<int32_t*>(ws + L.experts);
  int32_t* npp = reinterpret_cast<int32_t*>(ws + L.npp);
  void* h13 = ws + L.h13;
  void* act_out = ws + L.act;
  void* o = ws + L.o;
  int st;
  int32_t* const runs = form.runs ? reinterpret_cast<int32_t*>(h13) : nullptr;
  const MoeRoute route{router_logits, score_bias, T, E, topk, scoring, renormalize, routed_scale,
                       ids, wts, sorted, experts, npp, runs, reinterpret_cast<int32_t*>(ws + L.tab)};
  // a handful of tokens: the first expert GEMM takes the routing along (one launch less)
  const bool fold = moe_route_foldable(T, E, topk, tile);
  const MoeRoute* pending = fold ? &route : nullptr;
  if (!fold) {
    st = moe_route_launches(route, tile, stream);
    if (st) return st;
  }
  if (form.act) {
    st = moe_gemm_impl(hidden, w13_q, w13_s, w13_z, act_out, sorted, experts, npp, nullptr, L.n_slots, topk, tile, E, H,
                       2 * inter, group, 0, ws + L.gemm_ws, L.gemm_ws_bytes, stream, true, pending, runs);
    if (st) return st;
  } else {
    st = moe_gemm_impl(hidden, w13_q, w13_s, w13_z, h13, sorted, experts, npp, nullptr, L.n_slots, topk,
                       tile, E, H, 2 * inter, group, 0, ws + L.gemm_ws, L.gemm_ws_bytes, stream, false, pending, runs);
    if (st) return st;
    st = awqmi_silu_and_mul_f16(h13, act_out, L.n_slots, inter, stream);
    if (st) return st;
  }
  st = moe_gemm_impl(act_out, w2_q, w2_s, w2_z, o, sorted, experts, npp, wts, L.n_slots, 1, tile, E, inter, H,
                     group, 0, ws + L.gemm_ws, L.gemm_ws_bytes, stream, false, nullptr, runs);
  if (st) return st;
  return awqmi_moe_sum_f16(o, out, T, topk, H, stream);
}

int awqmi_workspace_reset(void* workspace, size_t workspace_bytes, void* stream) {
  if (!workspace) return AWQMI_NULL_POINTER;
  if (!aligned16(workspace)) return AWQMI_BAD_ALIGN;
  if (workspace_bytes < AWQMI_WS_COUNTER_BYTES) return AWQMI_WORKSPACE_TOO_SMALL;
  // a fill kernel rather than a memset node, so that the call behaves the same inside a capture
  hipLaunchKernelGGL(awq_zero_words_kernel, dim3(AWQMI_WS_COUNTER_BYTES / 16 / 256), dim3(256), 0,
                     (hipStream_t)stream, reinterpret_cast<u4v*>(workspace), AWQMI_WS_COUNTER_BYTES / 16);
  return launch_status();
}

// ---- development entry points (include/awq_mi355x_dev.h): the same calls with the launch-rule
// variant as an explicit argument, scoped to the call

int awqmi_dev_gemm_f16(const void* x, const int32_t* qweight, const void* scales, const int32_t* qzeros,
                       void* y, void* workspace, size_t workspace_bytes, int M, int K, int N, int group,
                       int split_k, void* stream, int variant) {
  VariantScope scope(variant);
  return awqmi_gemm_f16(x, qweight, scales, qzeros, y, workspace, workspace_bytes, M, K, N, group, split_k, stream);
}

int awqmi_dev_last_gemm_form(void) { return t_last_gemm_form; }

int awqmi_dev_gemm_timeline_f16(const void* x, const int32_t* qweight, const void* scales, const int32_t* qzeros,
                                void* y, void* workspace, size_t workspace_bytes, int M, int K, int N, int group,
                                int split_k, void* stream, unsigned long long* stamps, size_t stamps_bytes) {
  if (!stamps) return AWQMI_NULL_POINTER;
  if (M <= 0 || M > 16 || K <= 0 || N <= 0) return AWQMI_BAD_SHAPE;     // one dense skinny launch
  const int G = norm_group(K, group);
  if (check_awq_shape(K, N, G) != AWQMI_OK || !gemv_tiled_ok(K, G)) return AWQMI_BAD_SHAPE;
  const int split = split_k > 0 ? split_k : pick_split_k(M, K, N, G, 1, true);
  const size_t wgs = (size_t)((N / 8 + 16 * gemv_wpl(N) - 1) / (16 * gemv_wpl(N))) * split;
  if (stamps_bytes < wgs * 8 * sizeof(unsigned long long)) return AWQMI_WORKSPACE_TOO_SMALL;
  t_trace = stamps;
  const int rc = awqmi_gemm_f16(x, qweight, scales, qzeros, y, workspace, workspace_bytes, M, K, N, group, split_k, stream);
  t_trace = nullptr;
  return rc;
}

static inline int ldw_or(int nw, size_t pitch_words) { return pitch_words >= (size_t)nw ? (int)pitch_words : nw; }

int awqmi_dev_stream_probe(const void* src, void* out, int pattern, int K, int N, int parts, size_t total_bytes,
                           void* stream) {
  if (!src || !out) return AWQMI_NULL_POINTER;
  if (!aligned16(src) || !aligned16(out)) return AWQMI_BAD_ALIGN;
  hipStream_t st = (hipStream_t)stream;
  if (pattern == 0 || pattern == 2) {
    // whole 128-byte lines per column block, whole 128-row chunks, at least one chunk per wave
    if (K <= 0 || N <= 0 || K % 128 != 0 || N % 256 != 0 || parts < 1 || (K / 128) < 4 * parts) return AWQMI_BAD_SHAPE;
    if ((size_t)(N / 256) * parts > 65535u * 4u) return AWQMI_BAD_SHAPE;
    if (pattern == 0)
      hipLaunchKernelGGL((awq_stream_probe_kernel<0>), dim3(N / 256, parts), dim3(256), 0, st,
                         reinterpret_cast<const uint32_t*>(src), reinterpret_cast<uint32_t*>(out), K, ldw_or(N / 8, total_bytes), parts, (size_t)0);
    else
      hipLaunchKernelGGL((awq_stream_probe_kernel<2>), dim3(N / 256, parts), dim3(256), 0, st,
                         reinterpret_cast<const uint32_t*>(src), reinterpret_cast<uint32_t*>(out), K, 32, parts, (size_t)0);
  } else if (pattern == 1) {
    if (total_bytes < (1u << 20) || total_bytes % 1024 != 0) return AWQMI_BAD_SHAPE;
    hipLaunchKernelGGL((awq_stream_probe_kernel<1>), dim3(256), dim3(256), 0, st, reinterpret_cast<const uint32_t*>(src),
                       reinterpret_cast<uint32_t*>(out), 0, 0, 1, total_bytes);
  } else {
    return AWQMI_BAD_ARGUMENT;
  }
  return launch_status();
}

int awqmi_dev_mfma_probe(const void* src, void* out, int shape, int iters, void* stream) {
  if (!src || !out) return AWQMI_NULL_POINTER;
  if (!aligned16(src) || !aligned16(out)) return AWQMI_BAD_ALIGN;
  if (iters <= 0 || (shape != 0 && shape != 1)) return AWQMI_BAD_ARGUMENT;
  hipStream_t st = (hipStream_t)stream;
  if (shape == 0)
    hipLaunchKernelGGL((awq_mfma_probe_kernel<0>), dim3(256), dim3(256), 0, st, reinterpret_cast<const uint32_t*>(src),
                       reinterpret_cast<float*>(out), iters);
  else
    hipLaunchKernelGGL((awq_mfma_probe_kernel<1>), dim3(256), dim3(256), 0, st, reinterpret_cast<const uint32_t*>(src),
                       reinterpret_cast<float*>(out), iters);
  return launch_status();
}

size_t awqmi_dev_gemm_dense_workspace_bytes(int M, int K, int N) {
  if (M <= 0 || K <= 0 || N <= 0 || K % 64 != 0) return 0;
  const int slab = mfma_slab_rows(M, K);
  if (slab <= 0) return 0;
  size_t part = plan_mfma(slab, K, N, 256).part_bytes;
  if (M % slab) part = std::max(part, plan_mfma(M % slab, K, N, 256).part_bytes);
  return dense_panel_offset(part) + dg_panel_bytes(K, N);
}

int awqmi_dev_moe_gemm_f16(const void* x, const int32_t* qweight, const void* scales, const int32_t* qzeros,
                           void* y, const int32_t* sorted_token_ids, const int32_t* expert_ids,
                           const int32_t* num_tokens_post_padded, const float* topk_weights, int n_slots,
                           int a_row_div, int tile_m, int E, int K, int N, int group, int split_k,
                           void* workspace, size_t workspace_bytes, void* stream, int variant) {
  VariantScope scope(variant);
  return awqmi_moe_gemm_f16(x, qweight, scales, qzeros, y, sorted_token_ids, expert_ids, num_tokens_post_padded,
                            topk_weights, n_slots, a_row_div, tile_m, E, K, N, group, split_k, workspace,
                            workspace_bytes, stream);
}

int awqmi_dev_fused_moe_routed_f16(const void* hidden, const float* router_logits, const float* score_bias,
                                   const int32_t* w13_q, const void* w13_s, const int32_t* w13_z,
                                   const int32_t* w2_q, const void* w2_s, const int32_t* w2_z, void* out, int T,
                                   int H, int inter, int E, int topk, int group, int scoring, int renormalize,
                                   float routed_scale, void* workspace, size_t workspace_bytes, void* stream,
                                   int variant) {
  VariantScope scope(variant);
  return awqmi_fused_moe_routed_f16(hidden, router_logits, score_bias, w13_q, w13_s, w13_z, w2_q, w2_s, w2_z, out,
                                    T, H, inter, E, topk, group, scoring, renormalize, routed_scale, workspace,
                                    workspace_bytes, stream);
}

int awqmi_dev_fused_moe_block_rows(int T, int H, int inter, int E, int topk, int group, int variant) {
  VariantScope scope(variant);
  return awqmi_fused_moe_block_rows(T, H, inter, E, topk, group);
}

int awqmi_dev_fused_moe_tiles(int T, int H, int inter, int E, int topk, int group, int variant) {
  if (!awqmi_fused_moe_block_rows(T, H, inter, E, topk, group)) return 0;
  VariantScope scope(variant);
  return moe_form(T, H, inter, E, topk, group).runs;
}

int awqmi_dev_fused_moe_folds(int T, int H, int inter, int E, int topk, int group, int variant) {
  if (!awqmi_fused_moe_block_rows(T, H, inter, E, topk, group)) return 0;
  VariantScope scope(variant);
  const MoeForm form = moe_form(T, H, inter, E, topk, group);
  const int n_slots = T * topk, G = norm_group(H, group);
  if (form.tile != 16 || form.runs || !gemv_tiled_ok(H, G)) return 0;
  const MoePlan pl = moe_plan(n_slots, E, H, 2 * inter, 16, 0);
  return moe_launch_folds(moe_skinny_form(pl, n_slots, E, H, 2 * inter, 16, form.act), pl, T, E, topk, 16, G);
}

}  // extern "C"
