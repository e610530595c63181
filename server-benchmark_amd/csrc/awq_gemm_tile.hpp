// Fused AWQ GEMM of more rows than the skinny kernel takes: Y[M,N] = X[M,K] @ dequant(W) on fp16
// MFMA with fp32 accumulation, every weight unpacked in the registers of the wave that multiplies it.
//
// Workgroup tile 16 RT x 256, four waves side by side: each has all rows and 64 columns, 4 x RT
// v_mfma_f32_16x16x32_f16 accumulators (the shape that gives the most flops under the power limit, see
// awq_gemm_dense.hpp).  A weight is therefore unpacked once per tile, by the wave that needs it, and goes
// through LDS packed: X and packed W both travel from global memory straight into an LDS ring of D stages of 64 k.
//
// Unpacking.  Lane (n, q) of a 16 x 16 x 32 A operand holds k = 8 q .. 8 q + 7 of one column.  The 16 n of a tile are the two
// halves of eight packed words: lane n takes half n & 1 of word n >> 1, and the four nibbles of its half are its
// columns of the wave's four tiles.  Eight words (eight k) are 32 weights: per pair of words one v_perm that puts the two
// halves side by side, one shift, then and-or, subtract and multiply per nibble: 14 instructions for 8 weights, exact fp16
// (w - z) * s as awq_dequantize rounds it.  An output lane ends up with 16 consecutive columns of a row, which it
// stores as 32 bytes without a trip through LDS.
//
// LDS: X [row][128 B], 16-byte slot l of row r at l ^ ((r >> 1) & 7); W [k][128 B], the 32 bytes of wave w at chunk
// w ^ ((k >> 3) & 3), so that the four k groups of a read touch different banks (no conflicts measured).
//
// The k-step loop is written out: every MFMA is followed by its share of the next k-step's unpacking, the fragment read eight
// tiles ahead and the loads of the stage D - 1 ahead.  The waits are explicit.
//
// What bounds it: high tiles the power limit (8192 x 59136 at 2048 rows: matrix pipe busy 77 % of the cycles at 1.83 GHz), low
// ones the issue port, where a 16-cycle MFMA leaves room for two vector instructions: a stage takes a wave 32 MFMAs per 64
// rows and 133 vector instructions whatever the rows (at 64 rows 38 % MFMA, 21 % waiting for LDS or the barrier; with the unpacking
// taken out 59 of 90 us).  Against the kernel before it (weights dequantised into LDS by all waves, 32 x 32 x 16 MFMAs,
// tiles of 64 rows' steps), us: 8192 x 59136 at 80 / 128 / 400 / 1000 / 2047 rows 145 / 149 / 430 / 889 / 1701 -> 95 / 125 / 325 /
// 757 / 1500; 29568 x 8192 at 96 / 400 / 1000 81 / 226 / 433 -> 58 / 171 / 383; 3584 x 4608 at 64 / 1000 18.1 / 51 -> 15.7 / 42.
// Tiles of up to 128 rows share a CU in pairs (us, one / two workgroups: 8192 x 59136 at 256 rows in 128-row tiles 234 / 216, 3584 x
// 37888 100 / 85, 1024 x 12288 at 2047 60 / 53; a single round is even, 123 / 126).  32- and 48-row tiles against the skinny and the
// one-pass kernel stand at low_tile_pays and mid_shape.
// Measured and dropped: eight waves on two K halves of a tile, two per SIMD (8192 x 59136 at 64 rows 80 against 84 us, split
// layers slower); a ring of distinct LDS objects with the compiler's own waits (even, four times the code).
#pragma once
#include <type_traits>

#include "awq_common.hpp"
#include "awq_gemm_dense.hpp"

namespace awqmi {

struct TileGemmParams {
  const half_t* x;
  const uint32_t* qw;
  const half_t* sc;
  const uint32_t* qz;
  half_t* y;
  int M, K, N, NW, G;
  int ldw;        // words between consecutive rows of qweight (NW, or more when the rows are padded)
  int gshift;     // log2(G) when G < 64
  int mt, nt;     // tile counts
  int per_xcd;    // ceil(dp_tiles / 8)
  // Work split.  Tiles [0, dp_tiles) run one workgroup per tile over all of K (launch ids
  // [0, 8 * per_xcd)).  The remaining sk_tiles tiles (a last round that would leave CUs idle) are split in K over
  // sk_split workgroups each (launch ids from 8 * per_xcd on, part-major) and leave fp32 partial tiles in the
  // workspace; a second, short kernel on the same stream sums them in part order and writes fp16 (a single finishing
  // workgroup per tile would have to pull all of them by itself, which took longer than the GEMM).
  int dp_tiles, sk_tiles, sk_split;
  float* sk_part;   // [sk_tiles][sk_split][tg_part_floats]
  // Expert-grouped launch (awq_gemm_tile_grouped_kernel)
  const int* sorted_ids;
  const int* expert_ids;
  const int* n_live;        // padded slots (blocks) or tiles (runs) in use
  const int* runs;          // first 16-slot block and blocks of each tile
  const float* topk_w;      // optional per-slot output weight
  int n_slots, block;       // slots; slots of a block
  int a_row_div;            // X row of a slot = slot / a_row_div
  int total;                // column tiles x most blocks or tiles
  int in_order;             // tiles in launch order instead of ranges per XCD
  long long w_stride, s_stride, z_stride;   // elements per expert
};

constexpr int TG_COLS = 256;             // columns of a workgroup tile
// Offset of an X row that is not there: past the range of the buffer (below 4 GiB), so that the load brings zeros without traffic.
// (The range check takes the row's part that lies in the scalar offset into account; in the last 256 bytes below 4 GiB it
// would be a piece of X, for rows that nobody stores.)
constexpr uint32_t X_NOWHERE = 0xFFFFFF00u;
constexpr int TG_W_BYTES = 64 * 128;     // packed weights of a stage: 64 k x 256 columns

// LDS of one stage: X rows, packed weights, then each wave's group parameters
__host__ __device__ constexpr int tg_x_bytes(int rt) { return rt * 16 * 128; }
__host__ __device__ constexpr int tg_param_bytes(int any) { return any ? 160 * any : 256; }
__host__ __device__ constexpr int tg_slot_bytes(int rt, int any) { return tg_x_bytes(rt) + TG_W_BYTES + 4 * tg_param_bytes(any); }
// workgroups of a CU, LDS of each for the ring (the rest holds the slot lists of a grouped launch), and its stages
__host__ __device__ constexpr int tg_occupancy(int rt, int any) { return rt <= (any > 2 ? 3 : any ? 5 : 8) ? 2 : 1; }
__host__ __device__ constexpr int tg_lds_bytes(int most, int occ) { return (160 * 1024 / occ - 128 * most - 256) / 1024 * 1024; }
__host__ __device__ constexpr int tg_depth(int rt, int any, int lds) {
  const int fit = lds / tg_slot_bytes(rt, any);
  return fit < 7 ? fit : 7;
}
static_assert(tg_depth(4, 2, tg_lds_bytes(4, tg_occupancy(4, 2))) >= 4, "a tile of 64 rows keeps three stages on their way");
// floats of a K split's partial tile
__host__ __device__ constexpr size_t tg_part_floats(int rt) { return (size_t)rt * 16 * 256; }
// X fragments in flight: a divisor of the 2 RT fragments of a stage
__host__ __device__ constexpr int tg_ring(int rt) {
  return rt == 2 || rt == 8 ? 4 : rt == 3 ? 3 : 2 * rt % 8 == 0 ? 8 : 2 * rt % 7 == 0 ? 7 : 2 * rt % 6 == 0 ? 6 : 2 * rt % 5 == 0 ? 5 : rt;
}

#if defined(__HIP_DEVICE_COMPILE__)
typedef __attribute__((address_space(3))) unsigned char lds_byte;
template <class T>
__device__ __forceinline__ T lds_read(uint32_t a) {
  return *reinterpret_cast<const __attribute__((address_space(3))) T*>(a);
}

// The direct-to-LDS loads are asm statements: the compiler would put a wait for every one of them
// that may write what an LDS read reads, and with the stage's slot computed at run time it cannot tell
// them apart.  The waits are the kernel's own (tg_wait_and_barrier).
// acc += a * b, then 16 bytes a lane from rsrc into LDS at lds + 16 * lane; the MFMA is the wait state between
// the write of m0 and the load that reads it.
// ACC: where the accumulator is.
enum { IN_AGPR, IN_VGPR, NEW_VGPR };      // accumulation registers, vector registers, the same with nothing in it yet
#define TG_MFMA "v_mfma_f32_16x16x32_f16 %0, %1, %2, %0\n\t"
#define TG_MFMA_NEW "v_mfma_f32_16x16x32_f16 %0, %1, %2, 0\n\t"
#define TG_ASM(BEFORE, AFTER, ...)                                                                                   \
  do {                                                                                                               \
    if constexpr (ACC == NEW_VGPR) asm volatile(BEFORE TG_MFMA_NEW AFTER : "=&v"(c) : "v"(a), "v"(b), __VA_ARGS__ : "memory"); \
    else if constexpr (ACC == IN_VGPR) asm volatile(BEFORE TG_MFMA AFTER : "+v"(c) : "v"(a), "v"(b), __VA_ARGS__ : "memory");  \
    else asm volatile(BEFORE TG_MFMA AFTER : "+a"(c) : "v"(a), "v"(b), __VA_ARGS__ : "memory");                      \
  } while (0)
template <int ACC>
__device__ __forceinline__ void tg_mfma(f4& c, u4v a, h8 b) {
  if constexpr (ACC == NEW_VGPR) asm volatile(TG_MFMA_NEW : "=&v"(c) : "v"(a), "v"(b));
  else if constexpr (ACC == IN_VGPR) asm volatile(TG_MFMA : "+v"(c) : "v"(a), "v"(b));
  else asm volatile(TG_MFMA : "+a"(c) : "v"(a), "v"(b));
}
template <int ACC>
__device__ __forceinline__ void tg_mfma_load(f4& c, u4v a, h8 b, uint32_t lds, u4v rsrc, uint32_t voff, uint32_t soff) {
  TG_ASM("s_mov_b32 m0, %3\n\t", "buffer_load_dwordx4 %4, %5, %6 offen lds", "s"(lds), "v"(voff), "s"(rsrc), "s"(soff));
}
// ... of the lanes in `mask` only (every lane is active around it)
template <int ACC>
__device__ __forceinline__ void tg_mfma_load_some(f4& c, u4v a, h8 b, uint32_t lds, u4v rsrc, uint32_t voff, uint64_t mask) {
  TG_ASM("s_mov_b32 m0, %3\n\t", "s_mov_b64 exec, %6\n\tbuffer_load_dwordx4 %4, %5, 0 offen lds\n\ts_mov_b64 exec, -1",
         "s"(lds), "v"(voff), "s"(rsrc), "s"(mask));
}
// ... from one address per lane
template <int ACC>
__device__ __forceinline__ void tg_mfma_load_at(f4& c, u4v a, h8 b, uint32_t lds, uint64_t addr, uint64_t mask) {
  TG_ASM("s_mov_b32 m0, %3\n\t", "s_mov_b64 exec, %5\n\tglobal_load_lds_dwordx4 %4, off\n\ts_mov_b64 exec, -1", "s"(lds), "v"(addr),
         "s"(mask));
}
#undef TG_ASM
__device__ __forceinline__ void tg_load(uint32_t lds, u4v rsrc, uint32_t voff, uint32_t soff) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
               :: "s"(lds), "v"(voff), "s"(rsrc), "s"(soff) : "memory");
}
__device__ __forceinline__ void tg_load_some(uint32_t lds, u4v rsrc, uint32_t voff, uint64_t mask) {
  asm volatile("s_mov_b32 m0, %0\n\ts_mov_b64 exec, %3\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds\n\ts_mov_b64 exec, -1"
               :: "s"(lds), "v"(voff), "s"(rsrc), "s"(mask) : "memory");
}
__device__ __forceinline__ void tg_load_at(uint32_t lds, uint64_t addr, uint64_t mask) {
  asm volatile("s_mov_b32 m0, %0\n\ts_mov_b64 exec, %2\n\tglobal_load_lds_dwordx4 %1, off\n\ts_mov_b64 exec, -1"
               :: "s"(lds), "v"(addr), "s"(mask) : "memory");
}
// 4 bytes a lane of the lanes in `mask` into LDS at lds + 4 * lane (every lane is active around it)
__device__ __forceinline__ void tg_load_word(uint32_t lds, const void* addr, uint64_t mask) {
  asm volatile("s_mov_b32 m0, %0\n\ts_mov_b64 exec, %2\n\tglobal_load_lds_dword %1, off\n\ts_mov_b64 exec, -1"
               :: "s"(lds), "v"(addr), "s"(mask) : "memory");
}
// Scalar load of what no kernel in flight writes
__device__ __forceinline__ int tg_scalar(const int* p) {
  return __builtin_amdgcn_readfirstlane(*(const __attribute__((address_space(4))) int*)(uintptr_t)p);
}
__device__ __forceinline__ u4v tg_rsrc(const void* base, size_t bytes) {
  const uint64_t a = reinterpret_cast<uint64_t>(base);
  return u4v{(uint32_t)a, (uint32_t)(a >> 32) & 0xFFFFu, bytes > 0xFFFFFFFFull ? 0xFFFFFFFFu : (uint32_t)bytes, 0x00020000u};
}
// At most VM of this wave's loads outstanding, then the workgroup barrier: one statement, no LDS access
// moves across it.
template <int VM>
__device__ __forceinline__ void tg_wait_and_barrier() {
  asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(VM) : "memory");
}

// RT: 16-row tiles of the workgroup tile.  ANY = 0: G a multiple of 64 (a stage lies in one group) and N of 32.
// ANY = groups of a stage that there is room for, 2 or 8: also G a power of two from 64 / ANY on, and any N.  Room for 8 leaves a
// tile of 64 rows three stages of the ring if two share a CU, which do not cover HBM; groups of 32 and ragged columns, which take 2, have four (us, 8 / 2:
// 3840 x 36736, G = 32, at 54 rows 64 / 45; 2048 x 50512, G = 32, at 50 39 / 29; 2048 x 37272, G = 64, at 57 37 / 28).  With room for 8,
// tiles of 64 and 80 rows have a CU each and six or seven stages: 5 % faster on 31 layers in groups of 8 and 16 at 49 - 64 rows, even above.
// GROUPED: rows are slots of one expert e, s_sid the slot of each row (n_slots or more: none), s_tw its output weight.
// ACT (grouped): the matrix is [gate | up]; the tile is 128 gate columns from n0 on and their up columns, and
// writes silu(gate) * up.
// SCALE32 = stages of a group (1 or 2, 0: off): weights enter the product as the integers w - z, and a group's sum is
// scaled in fp32 when the group ends -- the skinny kernel's precision, for tiles that take its place.  The group's sum and the
// total are both in vector registers, so that tiles are at most 64 rows high, and stages go in pairs (ke - kb is even); the scaling is dealt out over the next
// group's first k-step.
template <int RT, int D, int ANY, bool GROUPED, bool ACT, int SCALE32 = 0>
__device__ __forceinline__ void awq_tile(const TileGemmParams& p, const int m0, const int n0, const int kb, const int ke,
                                         float* const part, const int e, const uint32_t smem, const int* const s_sid,
                                         const float* const s_tw) {
  constexpr int XB = tg_x_bytes(RT), SLOT = tg_slot_bytes(RT, ANY), PW = tg_param_bytes(ANY);
  constexpr int ZO = ANY ? 128 * ANY : 128;   // zero points behind the scales
  constexpr int XL = (RT + 1) / 2;            // X loads of a wave and stage
  constexpr int NL = XL + (ANY ? 4 : 3);      // all loads: weights (2), group parameters, X
  constexpr int XF = tg_ring(RT);
  constexpr int NP = 4 * RT;                  // MFMAs of a k-step
  // row tiles with their accumulators in the accumulation registers: not the whole file, or the compiler moves some of them
  // at the loop's edges, where it does not know when an asm statement's result is ready
  constexpr int AG = SCALE32 ? 0 : RT < 14 ? RT : 14;
  static_assert(!SCALE32 || (!ANY && SCALE32 <= 2), "");
  // loads of a stage are dealt out over it (over its first k-step with a ring of three)
  constexpr int LP = D == 3 ? NP - 2 : 2 * NP - 4;
  static_assert(D >= 3 && (D - 2) * NL < 64 && LP >= NL, "every load has an MFMA of its own");
  // MID: the next stage is waited for in the middle of a stage, ahead of the first read of it, instead of at the stage's start, and a
  // barrier of its own at the start frees the slot of the last stage.  With a ring of three a load then has 1.25 stages to arrive
  // instead of 0.75; longer rings leave it time enough (80 rows, ring of four, 209 us without and 213 with it).  With the pad rows'
  // loads out of range (X_NOWHERE), both versions in turn on one card, four layers, us before / after: 72B at 100 rows 259 / 245, 7B
  // (groups of 64) 122.7 / 112.9, at 128 rows 127.1 / 120.7, 5120-wide at 100 rows 121.7 / 114.9, at 200 176 / 163, at 1000 530 / 517; at
  // 256 187 - 190 / 183 - 187, within what the runs differ; a block of 1500 tokens on 128 experts of 2048 x 768, top-8, 176 / 171, of
  // 3000 even (305).
  constexpr bool MID = D == 3;
  constexpr int UF = 6;                       // MFMAs of the second k-step ahead of its unpacking
  static_assert(!MID || XF <= RT, "fragments of the next stage are read in the second k-step");
  static_assert(!MID || 1 + (NL - 1) * LP / NL < NP, "the wait in mid-stage counts on all loads of a stage being in its first k-step");
  static_assert(!MID || !SCALE32, "the scales of a group's sum are read in the other form only");

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int fi = lane & 15, fq = lane >> 4;
  const size_t es = GROUPED ? (size_t)e : 0;
  const u4v rx = tg_rsrc(p.x, (size_t)p.M * p.K * 2);
  const u4v rw = tg_rsrc(p.qw + es * p.w_stride, (size_t)p.K * p.ldw * 4);
  const u4v rz = tg_rsrc(p.qz + es * p.z_stride, (size_t)(p.K / p.G) * p.NW * 4);
  const u4v rs = tg_rsrc(p.sc + es * p.s_stride, (size_t)(p.K / p.G) * p.N * 2);

  // ---- global -> LDS roles
  uint32_t x_voff[XL];
#pragma unroll
  for (int i = 0; i < XL; ++i) {
    int idx = 4 * i + wave;
    if ((RT & 1) && idx >= 2 * RT) idx -= 2;
    const int r = 8 * idx + (lane >> 3);
    int gr = m0 + r;
    bool real = gr < p.M;
    if (GROUPED) {
      const int sid = s_sid[r];
      real = sid < p.n_slots;
      gr = sid / p.a_row_div;
    }
    x_voff[i] = real ? (uint32_t)(((size_t)gr * p.K + 8 * ((lane & 7) ^ dg_swz(r))) * 2) : X_NOWHERE;
  }
  auto x_lds = [&](int i) __attribute__((always_inline)) -> uint32_t {
    int idx = 4 * i + wave;
    if ((RT & 1) && idx >= 2 * RT) idx -= 2;
    return (uint32_t)idx * 1024u;
  };
  const uint32_t row_w = (uint32_t)p.ldw * 4u;
  // first packed column of the wave's half h (four words each)
  const int w0 = n0 / 8, up = ACT ? p.NW / 2 : 0;
  auto word = [&](int wv, int h) __attribute__((always_inline)) { return ACT ? w0 + 4 * wv + h * up : w0 + 8 * wv + 4 * h; };
  // group parameters: the wave's eight packed columns are 128 bytes of scales and 32 of zero points a group
  const int gps = ANY ? max(64 / p.G, 1) : 1;         // groups of a stage
  const int spg = ANY ? max(p.G / 64, 1) : p.G / 64;  // stages of a group
  int gl = __builtin_amdgcn_readfirstlane(kb / spg), gr = kb - gl * spg;    // first group of the next stage to load, its place in it
  if (ANY) gl *= gps;
  uint32_t w_voff, s_voff, z_voff;
  uint64_t p_addr;
  uint32_t p_step;
  {
    const int lc = (lane & 7) ^ (2 * wave);
    int wc = word(lc >> 1, lc & 1);
    if (wc >= p.NW) wc = 0;
    w_voff = (uint32_t)((8 * wave + (lane >> 3)) * p.ldw + wc) * 4u;
    int sw = word(wave, (lane >> 2) & 1) + (lane & 3), zw = word(wave, lane & 1);
    if (sw >= p.NW) sw = 0;
    if (zw >= p.NW) zw = 0;
    s_voff = (uint32_t)((lane >> 3) * p.N + 8 * sw) * 2u;       // ANY: lane = (group, word) ...
    z_voff = (uint32_t)((lane >> 1) * p.NW + zw) * 4u;          // ... and (group, four words)
    const bool zl = lane >= 8;                                  // else: eight lanes of scales, two of zero points
    p_addr = zl ? reinterpret_cast<uint64_t>(p.qz + es * p.z_stride + (size_t)gl * p.NW + zw)
                : reinterpret_cast<uint64_t>(p.sc + es * p.s_stride + (size_t)gl * p.N + 8 * sw);
    p_step = zl ? p.NW * 4u : p.N * 2u;
  }
  const uint64_t s_mask = gps == 8 ? ~0ull : (1ull << (8 * gps)) - 1, z_mask = (1ull << (2 * gps)) - 1;
  const uint32_t w_lds = XB + (uint32_t)wave * 1024u, p_lds = XB + TG_W_BYTES + (uint32_t)wave * PW;

  // ---- LDS -> register roles
  const int c = fi >> 1;
  uint32_t fx_off[2], ps_off[2], pz_off[2];
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) {
    fx_off[ks] = (uint32_t)(fi * 128 + (((4 * ks + fq) ^ dg_swz(fi)) << 4));
    const int row = ANY && p.G < 64 ? (32 * ks + 8 * fq) >> p.gshift : 0;
    ps_off[ks] = p_lds + (uint32_t)(row * 128 + c * 16);
    pz_off[ks] = p_lds + (uint32_t)(ZO + row * 32 + c * 4);
  }
  const uint32_t fw_off = (uint32_t)(XB + 8 * fq * 128 + (((2 * wave + (c >> 2)) ^ (2 * fq)) << 4) + (c & 3) * 4);
  const uint32_t sel_w = (fi & 1) ? 0x07060302u : 0x05040100u;
  const uint32_t sel_s = (fi & 1) ? 0x03020302u : 0x01000100u;

  f4 acc[4][RT], part_acc[4][SCALE32 ? RT : 1];       // totals; SCALE32: sums of the current group
  u4v gs[2] = {u4v{0u, 0u, 0u, 0u}, u4v{0u, 0u, 0u, 0u}};    // SCALE32: scales of the lane's 16 columns, last group
  NibbleMasks nm;
  nm.init();

  uint32_t zraw, zz[4], ss[4];
  u4v sraw;
  uint32_t wd[2][8];
  u4v wf[2][4];
  h8 xf[XF];
  auto read_params = [&](uint32_t slot, int ks) __attribute__((always_inline)) {
    zraw = lds_read<uint32_t>(slot + pz_off[ANY ? ks : 0]);
    if constexpr (!SCALE32) sraw = lds_read<u4v>(slot + ps_off[ANY ? ks : 0]);
  };
  auto expand = [&]() __attribute__((always_inline)) {
    const uint32_t za = __builtin_amdgcn_perm(zraw, zraw, sel_s), zb = za >> 8;
    zz[0] = (za & nm.lo) | MAGIC_LO;
    zz[1] = (za & nm.hi) | MAGIC_HI;
    zz[2] = (zb & nm.lo) | MAGIC_LO;
    zz[3] = (zb & nm.hi) | MAGIC_HI;
    if constexpr (!SCALE32)
#pragma unroll
      for (int j = 0; j < 4; ++j) ss[j] = __builtin_amdgcn_perm(sraw[j], sraw[j], sel_s);
  };
  // SCALE32: tile (j, im) of the last group, scaled, into the total
  auto flush = [&](int j, int im) __attribute__((always_inline)) {
    const h8 s[2] = {as_h8(gs[0]), as_h8(gs[1])};
#pragma unroll
    for (int r = 0; r < 4; ++r)
      acc[j][im][r] = __builtin_fmaf((float)s[r >> 1][2 * j + (r & 1)], part_acc[j][SCALE32 ? im : 0][r], acc[j][im][r]);
  };
  auto read_words = [&](int set, uint32_t fw, int ks, int rp) __attribute__((always_inline)) {
    wd[set][2 * rp] = lds_read<uint32_t>(fw + ks * 4096 + rp * 256);
    wd[set][2 * rp + 1] = lds_read<uint32_t>(fw + ks * 4096 + rp * 256 + 128);
  };
  uint32_t ua = 0, ub = 0, t1[16], t2[16];
  // step i of 18: pair the halves of item i's rows, subtract item i - 1, scale item i - 2 (SCALE32: no scaling)
  auto unpack = [&](int i, int set, int w) __attribute__((always_inline)) {
    if (i < 16) {
      const int rp = i >> 2, j = i & 3;
      if (j == 0) {
        ua = __builtin_amdgcn_perm(wd[w][2 * rp + 1], wd[w][2 * rp], sel_w);
        ub = ua >> 8;
      }
      const uint32_t u = j < 2 ? ua : ub;
      t1[i] = (j & 1) ? (u & nm.hi) | MAGIC_HI : (u & nm.lo) | MAGIC_LO;
    }
    if (i >= 1 && i < 17) t2[i - 1] = pk_sub(t1[i - 1], zz[(i - 1) & 3]);
    if (SCALE32 && i >= 1 && i < 17) wf[set][(i - 1) & 3][(i - 1) >> 2] = t2[i - 1];
    if (!SCALE32 && i >= 2) wf[set][(i - 2) & 3][(i - 2) >> 2] = pk_mul(t2[i - 2], ss[(i - 2) & 3]);
  };
  // The operands of the next k-step are complete, and the first MFMA reads them two wait states later.
  auto pin = [&](int set) __attribute__((always_inline)) {
    asm volatile("s_nop 1" : "+v"(wf[set][0]), "+v"(wf[set][1]), "+v"(wf[set][2]), "+v"(wf[set][3]));
    __builtin_amdgcn_sched_barrier(0);
  };

  // ---- loads of one stage: kl the stage, slot its LDS
  int kl = kb;
  uint32_t fill = smem;
  auto next_load = [&]() __attribute__((always_inline)) {
    fill += SLOT;
    if (fill == smem + D * SLOT) fill = smem;
    // stages past the last one load the last one again, which nobody reads
    if (kl + 1 < ke) {
      ++kl;
      if (++gr == spg) {
        gr = 0;
        gl += gps;
        if (!ANY) p_addr += p_step;
      }
    }
  };
  auto s_addr = [&]() __attribute__((always_inline)) { return s_voff + (uint32_t)(gl * p.N) * 2u; };
  auto z_addr = [&]() __attribute__((always_inline)) { return z_voff + (uint32_t)(gl * p.NW) * 4u; };
  auto w_addr = [&](int i) __attribute__((always_inline)) { return w_voff + ((uint32_t)kl * 64u + 32u * i) * row_w; };

  uint32_t cur = smem;      // LDS of the stage being multiplied
  // One k-step, KS its number in the stage, out of operand set KS; meanwhile the other set is unpacked for the
  // next k-step and the words after that are read.  cur / nxt: LDS of this stage and the next one.
  // FIRST / LAST: the stage is its group's first / last one (SCALE32).
  auto kstep = [&](auto KS, auto FIRST, auto LAST, const uint32_t (&xc)[2], const uint32_t (&xn)[2], uint32_t fwn, uint32_t nxt) __attribute__((always_inline)) {
    constexpr int ks = decltype(KS)::value;
    constexpr bool first = SCALE32 && decltype(FIRST)::value && ks == 0, last = !SCALE32 || decltype(LAST)::value;
    auto row = [&](auto WHERE, int im) __attribute__((always_inline)) {
      constexpr int ACC = decltype(WHERE)::value;
#pragma unroll
      for (int jj = 0; jj < 4; ++jj) {
        // one operand changes from one MFMA to the next
        const int j = (im & 1) ? 3 - jj : jj, m = 4 * im + jj;
        f4& a = SCALE32 ? part_acc[j][SCALE32 ? im : 0] : acc[j][im];
        if (first) flush(j, im);
        const u4v& w = wf[ks][j];
        const h8& x = xf[(ks * RT + im) % XF];
        int ld = -1;
#pragma unroll
        for (int i = 0; i < NL; ++i)
          if (1 + i * LP / NL == ks * NP + m) ld = i;
        if (ld < 0) tg_mfma<ACC>(a, w, x);
        else if (ld < 2) tg_mfma_load<ACC>(a, w, x, fill + w_lds + ld * 4096, rw, w_addr(ld), 0);
        else if (!ANY && ld == 2) tg_mfma_load_at<ACC>(a, w, x, fill + p_lds, p_addr, 0x3ffull);
        else if (ANY && ld == 2) tg_mfma_load_some<ACC>(a, w, x, fill + p_lds, rs, s_addr(), s_mask);
        else if (ANY && ld == 3) tg_mfma_load_some<ACC>(a, w, x, fill + p_lds + ZO, rz, z_addr(), z_mask);
        else tg_mfma_load<ACC>(a, w, x, fill + x_lds(ld - (NL - XL)), rx, x_voff[ld < NL - XL ? 0 : ld - (NL - XL)], (uint32_t)kl * 128u);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (MID) {
          // second k-step: parameters and words of the next stage, and what the parameters are for
          if (ANY && ks == 0 && m == 0) expand();
          if (ks == 1 && m == 0) read_params(nxt, 0);
          if (ks == 1 && m < 8) read_words(m >> 2, fwn, m >> 2, m & 3);
          if (ks == 1 && m == UF - 1) expand();
          if (ANY && ks == 1 && m == UF) read_params(nxt, 1);
          constexpr int U = ks ? UF : 0;
#pragma unroll
          for (int i = m < U ? 0 : 18 * (m - U) / (NP - U); i < (m < U ? 0 : 18 * (m - U + 1) / (NP - U)); ++i) unpack(i, ks ^ 1, ks ^ 1);
        } else {
          // parameters of the next stage; SCALE32: of the next group, and the scales of the one that ends
          if (last && m == 0 && (ANY || ks == 1)) expand();
          if (last && m == 1 && (ANY || ks == 0)) read_params(nxt, ks);
          if (SCALE32 && last && ks == 1 && (m == 1 || m == 2)) gs[m - 1] = lds_read<u4v>(cur + p_lds + 32 * fq + 16 * (m - 1));
#pragma unroll
          for (int i = 18 * m / NP; i < 18 * (m + 1) / NP; ++i) unpack(i, ks ^ 1, ks ^ 1);
          if (m < 4) read_words(ks, fwn, ks, m);
        }
        if (jj == 3) {
          const int f = ks * RT + im + XF;
          if (f < 2 * RT) xf[f % XF] = lds_read<h8>(xc[f / RT] + (f % RT) * 2048);
          else xf[f % XF] = lds_read<h8>(xn[(f - 2 * RT) / RT] + ((f - 2 * RT) % RT) * 2048);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    };
#pragma unroll
    for (int im = 0; im < AG; ++im) row(std::integral_constant<int, IN_AGPR>{}, im);
#pragma unroll
    for (int im = AG; im < RT; ++im) row(std::integral_constant<int, first ? NEW_VGPR : IN_VGPR>{}, im);
    pin(ks ^ 1);
  };
  using I0 = std::integral_constant<int, 0>;
  using I1 = std::integral_constant<int, 1>;

  // ---- prologue: D - 1 stages on their way, the first one unpacked
#pragma unroll
  for (int d = 0; d < D - 1; ++d) {
    tg_load(fill + w_lds, rw, w_addr(0), 0);
    tg_load(fill + w_lds + 4096, rw, w_addr(1), 0);
    if constexpr (ANY) {
      tg_load_some(fill + p_lds, rs, s_addr(), s_mask);
      tg_load_some(fill + p_lds + ZO, rz, z_addr(), z_mask);
    } else {
      tg_load_at(fill + p_lds, p_addr, 0x3ffull);
    }
#pragma unroll
    for (int i = 0; i < XL; ++i) tg_load(fill + x_lds(i), rx, x_voff[i], (uint32_t)kl * 128u);
    next_load();
  }
  // The accumulators start as products of zeros, while the first loads are on their way (as constants the
  // compiler would make them anew on every path into the loop and move them around at its edges).
  u4v zero = {0u, 0u, 0u, 0u};
  asm volatile("s_nop 1" : "+v"(zero));
#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if (i < AG) asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %1, 0" : "=a"(acc[j][i]) : "v"(zero));
      else asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %1, 0" : "=v"(acc[j][i]) : "v"(zero));
      if constexpr (SCALE32 != 0) asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %1, 0" : "=v"(part_acc[j][i]) : "v"(zero));
    }
  uint32_t xc[2] = {cur + fx_off[0], cur + fx_off[1]};
  tg_wait_and_barrier<(D - 2) * NL>();
#pragma unroll
  for (int rp = 0; rp < 4; ++rp) {
    read_words(0, cur + fw_off, 0, rp);
    read_words(1, cur + fw_off, 1, rp);
  }
#pragma unroll
  for (int f = 0; f < XF; ++f) xf[f] = lds_read<h8>(xc[f / RT] + (f % RT) * 2048);
  read_params(cur, 0);
  expand();
  if (ANY) read_params(cur, 1);
#pragma unroll
  for (int i = 0; i < 18; ++i) unpack(i, 0, 0);
  pin(0);

  auto stage = [&](auto FIRST, auto LAST) __attribute__((always_inline)) {
    // every wave has read the last stage, whose slot takes the stage D - 1 ahead; and, here or in the middle, the next stage
    // has landed (own loads; the barrier extends that to every wave's)
    if constexpr (MID) asm volatile("s_barrier" ::: "memory");
    else tg_wait_and_barrier<(D - 3) * NL>();
    __builtin_amdgcn_sched_barrier(0);
    uint32_t nxt = cur + SLOT;
    if (nxt == smem + D * SLOT) nxt = smem;
    uint32_t xn[2] = {nxt + fx_off[0], nxt + fx_off[1]};
    uint32_t fwn = nxt + fw_off;
    // (opaque: the reads' offsets stay in their offset fields)
    asm volatile("" : "+v"(xn[0]), "+v"(xn[1]), "+v"(fwn));
    kstep(I0{}, FIRST, LAST, xc, xn, fwn, nxt);
    if constexpr (MID) {
      tg_wait_and_barrier<NL>();
      __builtin_amdgcn_sched_barrier(0);
    }
    kstep(I1{}, FIRST, LAST, xc, xn, fwn, nxt);
    next_load();
    cur = nxt;
    xc[0] = xn[0];
    xc[1] = xn[1];
  };
  int n = ke - kb;
  constexpr std::bool_constant<SCALE32 != 2> each{};      // SCALE32 = 2: an even number of stages, two a group
  for (; n > 1; n -= 2) {
    stage(std::true_type{}, each);
    stage(each, std::true_type{});
  }
  if (!SCALE32 && n) stage(std::true_type{}, std::true_type{});
  // no load may still be writing this workgroup's LDS when it ends; the last MFMAs' results are in their registers
  asm volatile("s_waitcnt vmcnt(0)\n\ts_nop 7\n\ts_nop 7\n\ts_nop 7" ::: "memory");

  // The accumulators of one row of tiles at a time leave their registers behind this statement (moved all at once, ahead
  // of the wait above, some of them would be read too early or spilled).
  auto settle = [&](int im) __attribute__((always_inline)) {
    if constexpr (SCALE32 != 0) {
      asm volatile("" : "+v"(part_acc[0][im]), "+v"(part_acc[1][im]), "+v"(part_acc[2][im]), "+v"(part_acc[3][im]));
#pragma unroll
      for (int j = 0; j < 4; ++j) flush(j, im);
    } else if (im < AG) asm volatile("" : "+a"(acc[0][im]), "+a"(acc[1][im]), "+a"(acc[2][im]), "+a"(acc[3][im]));
    else asm volatile("" : "+v"(acc[0][im]), "+v"(acc[1][im]), "+v"(acc[2][im]), "+v"(acc[3][im]));
  };
  const int col = ACT ? n0 + 32 * wave + 16 * (fq & 1) + 8 * (fq >> 1) : n0 + 64 * wave + 16 * fq;
#pragma unroll
  for (int im = 0; im < RT; ++im) {
    settle(im);
    if (!GROUPED && part) {
#pragma unroll
      for (int j = 0; j < 4; ++j) *reinterpret_cast<f4*>(part + ((size_t)(im * 4 + j) * 256 + tid) * 4) = acc[j][im];
      continue;
    }
    int row = m0 + 16 * im + fi;
    float tw = 1.f;
    bool ok = row < p.M;
    if (GROUPED) {
      row = s_sid[16 * im + fi];
      ok = row < p.n_slots;
      tw = s_tw[16 * im + fi];
    }
    h8 o[2];
#pragma unroll
    for (int hf = 0; hf < 2; ++hf)
#pragma unroll
      for (int t = 0; t < 8; ++t) o[hf][t] = (half_t)(acc[t >> 1][im][2 * hf + (t & 1)] * tw);
    if constexpr (ACT) {
      // lanes below 32 hold 16 gate columns, their partners the same up columns: trade halves, then each has both
      // of eight columns
      u4v g = as_u4(o[0]), u = as_u4(o[1]);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const auto s = __builtin_amdgcn_permlane32_swap(g[i], u[i], false, false);
        g[i] = s[0];
        u[i] = s[1];
      }
      const h8 gh = as_h8(g), uh = as_h8(u);
      h8 a;
#pragma unroll
      for (int t = 0; t < 8; ++t) a[t] = silu_mul(gh[t], uh[t]);
      if (ok && col < p.N / 2) *reinterpret_cast<h8*>(p.y + (size_t)row * (p.N / 2) + col) = a;
    } else {
#pragma unroll
      for (int hf = 0; hf < 2; ++hf)
        if (ok && col + 8 * hf < p.N) *reinterpret_cast<h8*>(p.y + (size_t)row * p.N + col + 8 * hf) = o[hf];
    }
  }
}
#endif  // __HIP_DEVICE_COMPILE__

template <int RT, int ANY, int SCALE32 = 0>
__global__ __launch_bounds__(256, tg_occupancy(RT, ANY)) void awq_gemm_tile_kernel(const TileGemmParams p) {
#if defined(__HIP_DEVICE_COMPILE__)
  constexpr int D = tg_depth(RT, ANY, tg_lds_bytes(RT, tg_occupancy(RT, ANY)));
  __shared__ __align__(1024) unsigned char smem[D * tg_slot_bytes(RT, ANY)];
  const int id = blockIdx.x;
  const int KT = p.K / 64;
  int nid = 0, kb = 0, ke = KT;
  float* part = nullptr;
  if (id < 8 * p.per_xcd) {
    nid = (id & 7) * p.per_xcd + (id >> 3);
    if (nid >= p.dp_tiles) return;
  } else {
    const int j = id - 8 * p.per_xcd;
    const int tl = j % p.sk_tiles, pt = j / p.sk_tiles;
    nid = p.dp_tiles + tl;
    constexpr int U = SCALE32 ? 2 : 1;      // stages that stay together
    kb = (int)((long long)(KT / U) * pt / p.sk_split) * U;
    ke = (int)((long long)(KT / U) * (pt + 1) / p.sk_split) * U;
    part = p.sk_part + (size_t)(tl * p.sk_split + pt) * tg_part_floats(RT);
  }
  const int gsize = PF_GROUP_M * p.nt;
  const int first_m = (nid / gsize) * PF_GROUP_M;
  const int gm = min(p.mt - first_m, PF_GROUP_M);
  const int mt_i = first_m + (nid % gsize) % gm;
  const int nt_i = (nid % gsize) / gm;
  awq_tile<RT, D, ANY, false, false, SCALE32>(p, mt_i * (16 * RT), nt_i * 256, kb, ke, part, 0, (uint32_t)(uintptr_t)(lds_byte*)smem,
                                     nullptr, nullptr);
#endif
}

// Expert-grouped launch.  The sorted slots come in blocks of one expert each (moe_align).
// Without p.runs a tile is a block, of 64 or 128 slots, or half of one of 256.  With it (SCALE32) blocks are of 16 slots, and
// a tile is up to TG_RUN consecutive ones of one expert (a list made by the align kernels), so that an expert's weights are
// unpacked once per tile and not per block.
//
// A workgroup takes the lowest tile that holds its real slots: its cost follows the rows, and an expert's run often
// ends in a few dozen.
//
// 128 slots and two workgroups per CU: K is short (12 and 32 stages on experts of 2048 x 768), so that a tile's start and its
// output are a quarter of its time, and with tiles of 256 slots, one workgroup per CU, nothing runs beside them.
// Whole block of 8192 / 4096 / 1536 tokens on 128 such experts, top-8: 256 slots 743 / 437 / 217 us, 128 slots
// 709 / 399 / 184, 48 slots and three workgroups 907 / 485 / 226.
//
// The live tiles (their number is on the device only) are dealt to the eight XCDs in contiguous ranges, tile-major, so
// that the column tiles of a block share its gathered X rows and the blocks of an expert its weights through one L2; with
// few experts the ranges are uneven in rows and launch order is better.
constexpr int TG_ROWS = 128;   // slots of a tile at most
constexpr int TG_RUN = 4;      // 16-slot blocks of a SCALE32 tile at most
constexpr int TG_GROUPED_WGS = 2;   // workgroups of a CU (groups of 32, 3000 tokens on 128 experts of 2048 x 768: one 422 us, two 345)
template <int ANY, bool ACT, int SCALE32>
__global__ __launch_bounds__(256, TG_GROUPED_WGS) void awq_gemm_tile_grouped_kernel(const TileGemmParams p) {
#if defined(__HIP_DEVICE_COMPILE__)
  constexpr int ROWS = SCALE32 ? 16 * TG_RUN : TG_ROWS, LDS = tg_lds_bytes(TG_ROWS / 16, TG_GROUPED_WGS);
  __shared__ __align__(1024) unsigned char smem[LDS];
  __shared__ int s_sid[ROWS];
  __shared__ float s_tw[ROWS];
  const int tid = threadIdx.x;
  constexpr bool runs = SCALE32 != 0;
  const int tile_rows = min(p.block, ROWS);
  const int live = min((runs ? tg_scalar(p.n_live) : tg_scalar(p.n_live) / tile_rows) * p.nt, p.total);
  int nid = blockIdx.x;
  if (!p.in_order) {
    const int per = (live + 7) >> 3;
    nid = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
    if ((int)(blockIdx.x >> 3) >= per) return;
  }
  if (nid >= live) return;
  const int t = __builtin_amdgcn_readfirstlane(nid / p.nt);
  int first = t * tile_rows, most = tile_rows;
  if (runs) {
    const int run = tg_scalar(p.runs + t);
    first = (run >> 5) * 16;
    most = (run & 31) * 16;
  }
  // the expert id is on its way while the slots are staged: its weights' addresses wait for it
  const int eu = tg_scalar(p.expert_ids + __builtin_amdgcn_readfirstlane(first / p.block));
  const int lane = tid & 63;
  if (tid < ROWS) {
    const int sid = tid < most ? p.sorted_ids[first + tid] : p.n_slots;
    s_sid[tid] = sid;
    if (!p.topk_w) s_tw[tid] = 1.f;
  }
  __syncthreads();
  // the last real slot's row + 1: rows behind it are padding.  Every wave looks at all of them; the output weights, which nothing
  // needs before the tile's end, go to LDS by themselves
  int last = 0;
#pragma unroll
  for (int i = 0; i < ROWS; i += 64) {
    const int sid = s_sid[i + lane];
    const unsigned long long real = __ballot(sid < p.n_slots);
    if (real) last = i + 64 - __clzll(real);
    if (p.topk_w && __builtin_amdgcn_readfirstlane(tid >> 6) == i / 64) tg_load_word((uint32_t)(uintptr_t)(lds_byte*)(s_tw + i), p.topk_w + sid, real);
  }
  const int rows = __builtin_amdgcn_readfirstlane(last);
  const int n0 = (nid % p.nt) * (ACT ? TG_COLS / 2 : TG_COLS);
  const uint32_t lds = (uint32_t)(uintptr_t)(lds_byte*)smem;
  auto tile = [&](auto R) __attribute__((always_inline)) {
    constexpr int RT = decltype(R)::value;
    awq_tile<RT, tg_depth(RT, ANY, LDS), ANY, true, ACT, SCALE32>(p, 0, n0, 0, p.K / 64, nullptr, eu, lds, s_sid, s_tw);
  };
  if constexpr (!SCALE32) {
    if (rows > 112) return tile(std::integral_constant<int, 8>{});
    if (rows > 96) return tile(std::integral_constant<int, 7>{});
    if (rows > 80) return tile(std::integral_constant<int, 6>{});
    if (rows > 64) return tile(std::integral_constant<int, 5>{});
  }
  if (rows > 48) tile(std::integral_constant<int, 4>{});
  else if (rows > 32) tile(std::integral_constant<int, 3>{});
  else if (rows > 0) tile(std::integral_constant<int, 2>{});
#endif
}

// Sum of a split tile's parts, in part order: a workgroup per row tile, a thread per four columns of a row.  All parts of
// a thread are on their way at once (a loop of four paid a trip to memory for every part behind the fourth).  Launch and all, us a launch
// less at splits of 4 - 8: 0.35 on 2048 x 5120 and 4096 x 2048 (both at 20 / 64 rows 22.9 / 27.8 -> 22.1 / 27.1), 1 on 3584 .. 18944 weight rows (four
// layers in groups of 64 at 20 / 64 rows 82.4 / 92.8 -> 79.4 / 90.5); level from some 128 rows on and on 8192 columns and more, where it is the bytes (4.9 us at 64 rows).
template <int RT>
__global__ __launch_bounds__(1024) void awq_gemm_tile_reduce_kernel(const TileGemmParams p) {
  __shared__ __align__(16) h2 out[256][8];      // [thread of the tile kernel][its 16 columns]
  const int tid = threadIdx.x, j = tid >> 8, t = tid & 255;
  const int tl = blockIdx.x / RT, im = blockIdx.x % RT;
  const int nid = p.dp_tiles + tl;
  const int gsize = PF_GROUP_M * p.nt;
  const int first_m = (nid / gsize) * PF_GROUP_M;
  const int gm = min(p.mt - first_m, PF_GROUP_M);
  const int row0 = (first_m + (nid % gsize) % gm) * (16 * RT) + 16 * im, col0 = (nid % gsize) / gm * 256;
  const float* base = p.sk_part + (size_t)tl * p.sk_split * tg_part_floats(RT) + ((size_t)(im * 4 + j) * 256 + t) * 4;
  f4 v = {0.f, 0.f, 0.f, 0.f};
  auto sum = [&](auto N) {
    constexpr int n = decltype(N)::value;
    f4 q[n];
#pragma unroll
    for (int s = 0; s < n; ++s) q[s] = *reinterpret_cast<const f4*>(base + (size_t)s * tg_part_floats(RT));
#pragma unroll
    for (int s = 0; s < n; ++s) v += q[s];
    base += n * tg_part_floats(RT);
  };
  int left = p.sk_split;
  for (; left >= 8; left -= 8) sum(std::integral_constant<int, 8>{});
  switch (left) {
    case 7: sum(std::integral_constant<int, 7>{}); break;
    case 6: sum(std::integral_constant<int, 6>{}); break;
    case 5: sum(std::integral_constant<int, 5>{}); break;
    case 4: sum(std::integral_constant<int, 4>{}); break;
    case 3: sum(std::integral_constant<int, 3>{}); break;
    case 2: sum(std::integral_constant<int, 2>{}); break;
    case 1: sum(std::integral_constant<int, 1>{}); break;
  }
  out[t][j] = h2{(half_t)v[0], (half_t)v[1]};
  out[t][4 + j] = h2{(half_t)v[2], (half_t)v[3]};
  __syncthreads();
  if (tid >= 512) return;
  // eight columns a thread, a row's one after the other
  const int fi = tid >> 5, wave = (tid >> 3) & 3, fq = (tid >> 1) & 3, hf = tid & 1;
  const int row = row0 + fi, col = col0 + 8 * (tid & 31);
  if (row < p.M && col < p.N)
    *reinterpret_cast<h8*>(p.y + (size_t)row * p.N + col) = *reinterpret_cast<const h8*>(&out[64 * wave + 16 * fq + fi][4 * hf]);
}

}  // namespace awqmi
