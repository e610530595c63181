// AWQ GEMM for 33 .. 64 rows: Y[M,N] = X[M,K] @ dequant(W), one pass over the weights, every weight
// unpacked once and in registers.
//
// The load side is the skinny kernel's: one wave owns 256 output columns (two packed words per
// lane, 16 lanes side by side = one 128-byte line of a row, the four 16-lane groups take four
// 8-row slabs of a 32-row step) and a contiguous range of 128-row chunks of K; a workgroup is four
// waves on the same columns and different K ranges, one per SIMD.  Weights stay in registers, three
// to four steps ahead; activations go through the wave's own piece of LDS by direct-to-LDS loads, two
// steps a slot.  The multiply side: a lane's 8 x 8 nibble block becomes exact
// fp16 (w - z) * s, as awq_dequantize rounds it, and is the A operand of v_mfma_f32_16x16x32_f16
// against four 16-row blocks of X.  No dequantised weight goes through LDS and there is no barrier in
// the loop.
//
// What bounds it: the wave's own issue.  A 32-row step is 64 MFMAs and 224 unpack instructions and
// takes 1.0 us (62 us for 64 steps with 32 workgroups on the chip), against 0.7 us in which HBM
// delivers the 16 KiB of a CU (counters on 8192 x 59136: 63 % of a wave's cycles issue, 23 % are ready and do not,
// 14 % wait for memory or LDS; on 8192 x 10240 and 8192 x 8192 it is 49, 27 - 30 and 21 - 24 %).  8192 x 59136 at 64 rows
// takes 79 us (3.2 TB/s of packed weights), the tile kernel 85; the tile is ahead on layers of fewer than 320 Mi weights
// (see mid_shape).  Measured and dropped: two waves per SIMD with 128 columns each
// (64-byte pieces of a row per load, X read twice: 105 us), 32 x 32 x 16 MFMAs with one word per lane
// (twice the load instructions: 94 us), X in 64-byte pieces (84 us).
//
// With the weights as the A operand lane (j, h) ends up with all eight columns of eight
// neighbouring words of row j: 128 contiguous bytes of output.
#pragma once
#include "awq_common.hpp"

namespace awqmi {

struct MidGemmParams {
  const half_t* x;
  const uint32_t* qw;
  const half_t* sc;
  const uint32_t* qz;
  half_t* y;
  float* part;      // [split][ncb][4 row blocks][16 tiles][64 lanes] x 4 fp32 partial sums
  int M, K, N, NW, G;
  int ldw;          // words between rows of qweight
  int ncb, split_k;
};

constexpr int MID_MAX_ROWS = 64;
constexpr size_t MID_SLOT_FLOATS = 64 * 256;

// acc += a * b, accumulator tied in place (as a builtin the register allocator moves accumulators
// between the two halves of the register file: four moves per MFMA).  The compiler sees no hazards
// of an asm statement: operands that vector instructions wrote need two wait states before it, and
// the accumulators are read only behind the wait that ends the loop's body.
__device__ __forceinline__ void mid_mfma(f4& acc, h8 a, h8 b) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(acc) : "v"(a), "v"(b));
#endif
}

// KSPG: quantisation groups per 128-row chunk (4: G = 32, 2: G = 64, 1: G a multiple of 128)
template <int KSPG>
__global__ __launch_bounds__(256, 1) void awq_gemm_mid_kernel(const MidGemmParams p) {
  constexpr int MB = 4, NT = 16, RING = 4;
  constexpr int SPG = 4 / KSPG;                  // steps between changes of the group parameters
  constexpr int WB = 8192;                       // bytes of a wave's X of two steps: 64 rows x 64 k
  // X ring, two steps a slot: each of the two slots is one LDS object, so that the wait before a
  // fragment read counts only the loads issued behind that slot's.  (The cross-wave sum behind the loop
  // takes 128 KiB.)
  __shared__ __align__(1024) unsigned char xr0[4 * WB], xr1[4 * WB], xr2[4 * WB], xr3[4 * WB];
  unsigned char* const xr[4] = {xr0, xr1, xr2, xr3};
  const int tid = threadIdx.x, lane = tid & 63, j = lane & 15, h = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int cb = blockIdx.x, sp = blockIdx.y;

  // Lanes past the last word column / rows past the last read word 0 / row 0 instead; their results
  // are never stored.
  int wc = cb * 32 + 2 * j;
  if (wc >= p.NW) wc = 0;
  // X: instruction b fetches 64 k of rows 8 b .. 8 b + 7, whole 128-byte lines; 16-byte piece o of row
  // r lands in slot o ^ swz(r) of the row's line, swz(r) = (r ^ (r >> 3)) & 7, under which the 16 rows
  // of a fragment read touch 16 different bank groups.  (64-byte pieces, 32 k a time, measured
  // slower: the loads of a CU are bound by their number of lines.)
  uint32_t x_off[8];
#pragma unroll
  for (int b = 0; b < 8; ++b) {
    const int r = 8 * b + (lane >> 3);
    x_off[b] = (uint32_t)(((size_t)(r < p.M ? r : 0) * p.K + 8 * ((lane ^ (lane >> 3) ^ b) & 7)) * 2);
  }
  int f_off[MB];      // even step; the odd one's k is piece ^ 4
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) f_off[mb] = mb * 2048 + j * 128 + ((h ^ ((j ^ (j >> 3) ^ (2 * mb)) & 7)) << 4);
  const uint32_t q_off = (uint32_t)(((size_t)8 * h * p.ldw + wc) * 4);
  const half_t* const sc = p.sc + 8 * (size_t)wc;
  const uint32_t* const qz = p.qz + wc;

  const int nchunks = p.K >> 7;
  const unsigned parts = 4u * (unsigned)p.split_k, pw = (unsigned)sp * 4u + (unsigned)wave;
  const int c_begin = (int)(pw * (unsigned)nchunks / parts);
  const int c_end = (int)((pw + 1) * (unsigned)nchunks / parts);
  const int cpg = KSPG == 1 ? p.G >> 7 : 1;      // chunks per group (KSPG = 1)

  u2v q[RING][8];
  f4 acc[MB][NT];
  u2v znext;
  u4v snext[2];
  uint32_t zz[2][8], ss[2][8];      // per nibble: zero point (+ magic) and scale, both halves alike
  NibbleMasks nm;
  nm.init();

  // Loads of a step, in buffer form; behind the wave's last step `live` is 0 and the loop needs no second
  // copy without them: the weight loads are of the matrix's first 32 rows (inside it whatever the range of
  // 0 does with them; the values are not used), the X loads are out of range and put zeros into a slot that
  // is not read again.
  const int q_bytes = (int)((size_t)p.K * p.ldw * 4), x_bytes = (int)((size_t)p.M * p.K * 2);
  // row i of a lane's eight of step ks into ring slot d
  auto issue_w = [&](int d, int i, int ks, bool live) __attribute__((always_inline)) {
#if defined(__HIP_DEVICE_COMPILE__)
    const __amdgpu_buffer_rsrc_t rq =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<uint32_t*>(p.qw), 0, live ? q_bytes : 0, 0x00020000);
    const uint32_t row = (uint32_t)p.ldw * 4u, so = live ? (uint32_t)ks * 32u * row : 0u;
    q[d][i] = __builtin_amdgcn_raw_buffer_load_b64(rq, q_off, so + i * row, 2);
#endif
  };
  auto issue_x = [&](int s, int ks, bool live) __attribute__((always_inline)) {
#if defined(__HIP_DEVICE_COMPILE__)
    typedef __attribute__((address_space(3))) void lds_void;
    const __amdgpu_buffer_rsrc_t rx =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<half_t*>(p.x), 0, live ? x_bytes : 0, 0x00020000);
#pragma unroll
    for (int b = 0; b < 8; ++b)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, (lds_void*)(xr[s] + wave * WB + b * 1024), 16, x_off[b],
                                               live ? ks * 64 : 0, 0, 0);
#endif
  };
  auto load_group = [&](int g) __attribute__((always_inline)) {
    znext = *reinterpret_cast<const u2v*>(qz + (size_t)g * p.NW);
#pragma unroll
    for (int w = 0; w < 2; ++w) snext[w] = *reinterpret_cast<const u4v*>(sc + (size_t)g * p.N + 8 * w);
  };
  auto expand_byte = [&](auto BTAG) __attribute__((always_inline)) {
    constexpr int B = decltype(BTAG)::value;
#pragma unroll
    for (int w = 0; w < 2; ++w) {
      const uint32_t zw = w ? znext.y : znext.x;
      const uint32_t tz = byte_pair<B>(zw, zw);
      zz[w][2 * B] = (tz & nm.lo) | MAGIC_LO;
      zz[w][2 * B + 1] = (tz & nm.hi) | MAGIC_HI;
      constexpr int cl = awq_col_of_nibble(2 * B), ch = awq_col_of_nibble(2 * B + 1);
      const uint32_t sl = snext[w][cl >> 1], sh = snext[w][ch >> 1];
      ss[w][2 * B] = __builtin_amdgcn_perm(sl, sl, (cl & 1) ? 0x03020302u : 0x01000100u);
      ss[w][2 * B + 1] = __builtin_amdgcn_perm(sh, sh, (ch & 1) ? 0x03020302u : 0x01000100u);
    }
  };
  using I0 = std::integral_constant<int, 0>;
  using I1 = std::integral_constant<int, 1>;
  using I2 = std::integral_constant<int, 2>;
  using I3 = std::integral_constant<int, 3>;
  auto compute = [&](int d, int s, int ks_next, bool live) __attribute__((always_inline)) {
    h8 a[MB];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
      a[mb] = *reinterpret_cast<const h8*>(xr[s] + wave * WB + (f_off[mb] ^ (64 * (d & 1))));
    // Registers RP of the operands of byte B of word w: tiles 8 w + 2 B (lo) and 8 w + 2 B + 1 (hi), in two
    // parts to be dealt out between MFMAs (a packed result is not read by the very next instruction:
    // the compiler would put a wait state in between).
    u4v lo[2], hi[2];
    uint32_t tl = 0, th = 0;
    auto unpack = [&](int set, int w, auto BTAG, int rp, int part) __attribute__((always_inline)) {
      constexpr int B = decltype(BTAG)::value;
      if (part == 0) {
        const uint32_t t = w ? byte_pair<B>(q[d][2 * rp + 1].y, q[d][2 * rp].y) : byte_pair<B>(q[d][2 * rp + 1].x, q[d][2 * rp].x);
        tl = pk_sub((t & nm.lo) | MAGIC_LO, zz[w][2 * B]);
        th = (t & nm.hi) | MAGIC_HI;
      } else {
        th = pk_sub(th, zz[w][2 * B + 1]);
        lo[set][rp] = pk_mul(tl, ss[w][2 * B]);
        hi[set][rp] = pk_mul(th, ss[w][2 * B + 1]);
      }
    };
    // Eight MFMAs of one byte; the next byte's operands are unpacked between them, half a register
    // pair behind each.
    auto stage = [&](int k, int wn, auto BN, bool more) __attribute__((always_inline)) {
      // a vector instruction's result may be read by an MFMA two wait states later
      // (the operands pass through the statement, so that all of them are written before it)
      asm volatile("s_nop 1" : "+v"(lo[k & 1]), "+v"(hi[k & 1]));
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < 2 * MB; ++i) {
        const int mb = i < MB ? i : 2 * MB - 1 - i;
        mid_mfma(acc[mb][2 * k + (i >= MB)], as_h8(i < MB ? lo[k & 1] : hi[k & 1]), a[mb]);
        if (more) unpack((k + 1) & 1, wn, BN, i >> 1, i & 1);
        // the weights of three steps on, into the slot that the last step has left
        if (i == 3) issue_w((d + 3) & 3, k, ks_next, live);
        __builtin_amdgcn_sched_barrier(0);
      }
    };
#pragma unroll
    for (int i = 0; i < 8; ++i) unpack(0, 0, I0{}, i >> 1, i & 1);
    __builtin_amdgcn_sched_barrier(0);
    stage(0, 0, I1{}, true);
    stage(1, 0, I2{}, true);
    stage(2, 0, I3{}, true);
    stage(3, 1, I0{}, true);
    stage(4, 1, I1{}, true);
    stage(5, 1, I2{}, true);
    stage(6, 1, I3{}, true);
    stage(7, 1, I3{}, false);
  };
#pragma unroll
  for (int mb = 0; mb < MB; ++mb)
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[mb][t] = f4{0.f, 0.f, 0.f, 0.f};
  const int last_group = p.K / p.G - 1;
  if (c_begin < c_end) {
    load_group(KSPG == 1 ? c_begin / cpg : c_begin * KSPG);
    issue_x(0, 4 * c_begin, true);
#pragma unroll
    for (int d = 0; d < RING - 1; ++d) {
#pragma unroll
      for (int i = 0; i < 8; ++i) issue_w(d, i, 4 * c_begin + d, true);
      if (d == 1) issue_x(1, 4 * c_begin + 2, true);
    }
    for (int c = c_begin; c < c_end; ++c) {
      const bool more = c + 1 < c_end;
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        if (d % SPG == 0) {
          expand_byte(I0{});
          expand_byte(I1{});
          expand_byte(I2{});
          expand_byte(I3{});
          // parameters of the next group this wave meets
          load_group(min(KSPG == 1 ? (c + 1) / cpg : (c * 4 + d) / SPG + 1, last_group));
          __builtin_amdgcn_sched_barrier(0);
        }
        compute(d, d / 2, 4 * c + d + 3, d == 0 || more);
        __builtin_amdgcn_sched_barrier(0);
        if (d & 1) issue_x(d / 2, 4 * c + d + 3, more);
        __builtin_amdgcn_sched_barrier(0);
      }
      // the last MFMAs' results are in their registers before anything behind the loop reads them
      asm volatile("s_nop 15");
      __builtin_amdgcn_sched_barrier(0);
    }
  }

  // ---- sum over the four K ranges: waves w and w ^ 1 trade two row blocks each, then w and w ^ 2 one;
  // wave w ends up with row block 2 (w & 1) + (w >> 1), summed as (0 + 1) + (2 + 3) ----
  // (in the X ring's memory: every wave has read its fragments, and no load into it is in flight, the
  // zero-filling ones behind a wave's last step among them)
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  // lane index from scratch: kept over the loop, it would cost registers there
  const int el = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u)), ej = el & 15, eh = el >> 4;
  auto xch = [&](int w, int i) __attribute__((always_inline)) -> f4& {
    return *reinterpret_cast<f4*>(xr[i >> 3] + w * WB + (i & 7) * 1024 + el * 16);
  };
  f4 v[2][NT];
  const bool odd = wave & 1, high = wave >> 1;
#pragma unroll
  for (int b = 0; b < 2; ++b)
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      xch(wave, b * NT + t) = odd ? acc[b][t] : acc[2 + b][t];
      v[b][t] = odd ? acc[2 + b][t] : acc[b][t];
    }
  __syncthreads();
#pragma unroll
  for (int b = 0; b < 2; ++b)
#pragma unroll
    for (int t = 0; t < NT; ++t) v[b][t] += xch(wave ^ 1, b * NT + t);
  __syncthreads();
#pragma unroll
  for (int t = 0; t < NT; ++t) xch(wave, t) = high ? v[0][t] : v[1][t];
  __syncthreads();
  f4 o[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) o[t] = (high ? v[1][t] : v[0][t]) + xch(wave ^ 2, t);

  const int mb = 2 * (wave & 1) + (wave >> 1);
  if (mb * 16 >= p.M) return;
  if (p.split_k > 1) {
    // summed in part order and written out by awq_gemm_mid_reduce_kernel, launched behind this one
    f4* const mine = reinterpret_cast<f4*>(p.part) + (((size_t)sp * p.ncb + cb) * 4 + mb) * (NT * 64) + el;
#pragma unroll
    for (int t = 0; t < NT; ++t) mine[t * 64] = o[t];
    return;
  }
  const int row = mb * 16 + ej;
  if (row >= p.M) return;
  // o[8 w + nibble][r]: word 2 (4 h + r) + w of the column block, column awq_col_of_nibble(nibble)
#pragma unroll
  for (int r = 0; r < 4; ++r)
#pragma unroll
    for (int w = 0; w < 2; ++w) {
      const int word = cb * 32 + 2 * (4 * eh + r) + w;
      h8 out;
#pragma unroll
      for (int c = 0; c < 8; ++c) out[c] = (half_t)o[8 * w + awq_nibble_of_col(c)][r];
      if (word < p.NW) *reinterpret_cast<h8*>(p.y + (size_t)row * p.N + 8 * word) = out;
    }
}

// Sum of the partial tiles of a K split, in part order.  One workgroup per column block and row
// block; thread (word parity, lane, register pair) sums two words' eight columns.
__global__ __launch_bounds__(256) void awq_gemm_mid_reduce_kernel(const MidGemmParams p) {
  typedef float f2 __attribute__((ext_vector_type(2)));
  const int tid = threadIdx.x, rp = tid & 1, lane = (tid >> 1) & 63, half = tid >> 7;
  const int j = lane & 15, h = lane >> 4;
  const int cb = blockIdx.x, mb = blockIdx.y;
  const size_t stride = (size_t)p.ncb * MID_SLOT_FLOATS;
  const float* base = p.part + (((size_t)cb * 4 + mb) * 2 + half) * (8 * 64 * 4) + lane * 4 + 2 * rp;
  f2 v[8];
#pragma unroll
  for (int t = 0; t < 8; ++t) v[t] = f2{0.f, 0.f};
#pragma unroll 4
  for (int s = 0; s < p.split_k; ++s)
#pragma unroll
    for (int t = 0; t < 8; ++t) v[t] += *reinterpret_cast<const f2*>(base + s * stride + t * 256);
  const int row = mb * 16 + j;
  if (row >= p.M) return;
#pragma unroll
  for (int r = 0; r < 2; ++r) {
    const int word = cb * 32 + 2 * (4 * h + 2 * rp + r) + half;
    h8 out;
#pragma unroll
    for (int c = 0; c < 8; ++c) out[c] = (half_t)v[awq_nibble_of_col(c)][r];
    if (word < p.NW) *reinterpret_cast<h8*>(p.y + (size_t)row * p.N + 8 * word) = out;
  }
}

}  // namespace awqmi
