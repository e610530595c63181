// Routing-side kernels of the expert-grouped AWQ path: softmax + top-k, the stable
// sort/pad of routed slots by expert, the SiLU(gate) * up activation between the two expert
// GEMMs, and the final sum over a token's slots.  All are latency-sized integer / elementwise
// work; the expert GEMMs themselves are the MOE instantiation of the skinny kernel.
#pragma once
#include <type_traits>
#include "awq_common.hpp"

namespace awqmi {

// Wave-wide max / sum by DPP row shifts and row broadcasts (full-rate VALU, no LDS crossbar
// trips); the result is taken from lane 63 and returned wave-uniform.
template <bool IS_MAX>
__device__ __forceinline__ float wave_reduce_f32(float v) {
  const int ident = IS_MAX ? (int)0xff800000u : 0;   // -inf / 0.0f
  auto step = [&](auto CTRL, auto ROWS) {
    const int o = __builtin_amdgcn_update_dpp(ident, __builtin_bit_cast(int, v), decltype(CTRL)::value,
                                              decltype(ROWS)::value, 0xf, false);
    const float f = __builtin_bit_cast(float, o);
    v = IS_MAX ? fmaxf(v, f) : v + f;
  };
  using std::integral_constant;
  step(integral_constant<int, 0x111>{}, integral_constant<int, 0xf>{});   // row_shr:1
  step(integral_constant<int, 0x112>{}, integral_constant<int, 0xf>{});   // row_shr:2
  step(integral_constant<int, 0x114>{}, integral_constant<int, 0xf>{});   // row_shr:4
  step(integral_constant<int, 0x118>{}, integral_constant<int, 0xf>{});   // row_shr:8: lane 15 of a row = row total
  step(integral_constant<int, 0x142>{}, integral_constant<int, 0xa>{});   // row_bcast:15 into rows 1, 3
  step(integral_constant<int, 0x143>{}, integral_constant<int, 0xc>{});   // row_bcast:31 into rows 2, 3
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 63));
}

// Top-k of one token by LANES lanes of a wave, PER experts per lane (E <= LANES * PER); pick k ends up in lane k of the
// token's lanes (id, w; topk <= LANES).
// SIGMOID = false: softmax scores; selection runs on the raw logits (softmax is monotonic).
// SIGMOID = true: score = sigmoid(logit); selection runs on score + bias[e] (bias may be
// null), the weight is the score itself.  Ties go to the lowest expert id; NaN keys lose against every number and are
// then taken in expert order, so that every id stays inside [0, E) (the weight is NaN and carries the bad logit forward).
// Weights are optionally renormalised over the selected experts and multiplied by `scale`.
//
// LANES = 64 (one token a wave): each pick is one wave-wide max of the remaining keys, then a ballot of the lanes that hold
// it (lowest expert id first); the winner's id and key are wave-uniform from there on.
template <int PER, bool SIGMOID>
__device__ __forceinline__ void moe_pick_wave(const float* __restrict__ row, const float* __restrict__ bias, int E,
                                              int topk, int renorm, float scale, int& id, float& w) {
  const int lane = threadIdx.x & 63;
  float v[PER];      // selection key
  float sc[PER];     // score (SIGMOID only)
  bool open[PER];    // expert exists and is not picked yet
  float lmax = -INFINITY;
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int e = lane + 64 * i;
    open[i] = e < E;
    const float x = e < E ? row[e] : -INFINITY;
    if (SIGMOID) {
      sc[i] = 1.f / (1.f + __expf(-x));
      v[i] = e < E ? sc[i] + (bias ? bias[e] : 0.f) : -INFINITY;
    } else {
      sc[i] = 0.f;
      v[i] = x;
      lmax = fmaxf(lmax, x);
    }
  }
  float mx = 0.f, sum = 1.f;
  if (!SIGMOID) {
    mx = wave_reduce_f32<true>(lmax);
    float ls = 0.f;
#pragma unroll
    for (int i = 0; i < PER; ++i)
      if (lane + 64 * i < E) ls += __expf(v[i] - mx);
    sum = wave_reduce_f32<false>(ls);
  }

  float sel_sum = 0.f;
  float my_w = 0.f;   // lane j keeps the weight of pick j (topk <= 64)
  int my_id = 0;
  for (int it = 0; it < topk; ++it) {
    float loc = -INFINITY;
#pragma unroll
    for (int i = 0; i < PER; ++i)
      if (open[i]) loc = fmaxf(loc, v[i]);
    const float best = wave_reduce_f32<true>(loc);
    int bidx = E;                                    // stays E only if every key left is NaN
#pragma unroll
    for (int i = PER - 1; i >= 0; --i) {             // descending, so the lowest id wins
      const unsigned long long b = __ballot(open[i] && v[i] == best);
      if (b) bidx = 64 * i + __builtin_ctzll(b);
    }
    if (bidx == E) {
      // only NaN keys are left (fmaxf skipped them, nothing equals `best`): the lowest expert that is still open
#pragma unroll
      for (int i = PER - 1; i >= 0; --i) {
        const unsigned long long b = __ballot(open[i]);
        if (b) bidx = 64 * i + __builtin_ctzll(b);
      }
    }
    float bsc = 0.f;
    if (SIGMOID) {
#pragma unroll
      for (int i = 0; i < PER; ++i)
        if ((bidx >> 6) == i)
          bsc = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, sc[i]), bidx & 63));
    }
    float bkey = best;                               // the winner's own key (NaN when only NaN keys are left)
    if (!SIGMOID) {
#pragma unroll
      for (int i = 0; i < PER; ++i)
        if ((bidx >> 6) == i)
          bkey = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v[i]), bidx & 63));
    }
    const float pw = SIGMOID ? bsc : __expf(bkey - mx) / sum;
    sel_sum += pw;
    if (lane == it) { my_w = pw; my_id = bidx; }
#pragma unroll
    for (int i = 0; i < PER; ++i)
      if (lane + 64 * i == bidx) open[i] = false;
  }
  id = my_id;
  w = (renorm ? my_w / sel_sum : my_w) * scale;
}

// All 16 lanes of a row get op over the row (DPP row rotations).
template <class T, class OP>
__device__ __forceinline__ T row_reduce(T v, OP op) {
  auto step = [&](auto CTRL) {
    v = op(v, __builtin_bit_cast(T, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), decltype(CTRL)::value, 0xf, 0xf, true)));
  };
  using std::integral_constant;
  step(integral_constant<int, 0x128>{});   // row_ror:8
  step(integral_constant<int, 0x124>{});
  step(integral_constant<int, 0x122>{});
  step(integral_constant<int, 0x121>{});
  return v;
}

// LANES = 16 (four tokens a wave): lane l of a token holds experts PER l .. PER l + PER - 1.  The keys are integers that
// order as the floats do (-0 as 0, NaN below -inf, a picked or absent expert below that).  A pick is a max over the
// lane's keys and over the row, the lowest id that holds it, likewise a minimum over the row, and one select per key
// to close it: some 50 vector instructions for four tokens, where the wave-wide form spends as many on one.  Weights are worked out once, by the lane that holds the pick.
template <int PER, bool SIGMOID>
__device__ __forceinline__ void moe_pick_row(const float* __restrict__ row, const float* __restrict__ bias, int E,
                                             int topk, int renorm, float scale, int& id, float& w) {
  constexpr int GONE = (int)0x80000000u, NOT_A_NUMBER = GONE + 1;
  const int l = threadIdx.x & 15, e0 = PER * l;
  // (absent experts read one that is there: no load and no select sits behind a branch)
  float x[PER];
  if ((E & 3) == 0 && (reinterpret_cast<uintptr_t>(row) & 15) == 0) {
#pragma unroll
    for (int i = 0; i < PER; i += 4) {
      const f4 q = *reinterpret_cast<const f4*>(row + min(e0 + i, E - 4));
#pragma unroll
      for (int j = 0; j < 4; ++j) x[i + j] = q[j];
    }
  } else {
#pragma unroll
    for (int i = 0; i < PER; ++i) x[i] = row[min(e0 + i, E - 1)];
  }
  if (SIGMOID) {
#pragma unroll
    for (int i = 0; i < PER; ++i) x[i] = 1.f / (1.f + __expf(-x[i]));
    if (bias)
#pragma unroll
      for (int i = 0; i < PER; ++i) x[i] += bias[min(e0 + i, E - 1)];
  }
  int key[PER];
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int b = __builtin_bit_cast(int, x[i] + 0.f);
    const int k = x[i] == x[i] ? b ^ ((b >> 31) & 0x7fffffff) : NOT_A_NUMBER;
    key[i] = e0 + i < E ? k : GONE;
  }
  auto value = [](int k) { return k == NOT_A_NUMBER ? NAN : __builtin_bit_cast(float, k ^ ((k >> 31) & 0x7fffffff)); };
  int my_id = 0, my_key = 0, top = 0;
  for (int it = 0; it < topk; ++it) {
    int loc = key[0];
#pragma unroll
    for (int i = 1; i < PER; ++i) loc = max(loc, key[i]);
    const int best = row_reduce(loc, [](int a, int b) { return max(a, b); });
    if (it == 0) top = best;
    int first = 0x7fffffff;                // the lane's first expert that holds the best key
#pragma unroll
    for (int i = PER - 1; i >= 0; --i) first = key[i] == best ? i : first;
    const int win = row_reduce(first < PER ? e0 + first : first, [](int a, int b) { return min(a, b); });
    my_id = l == it ? win : my_id;
    my_key = l == it ? best : my_key;
    const int own = win - e0;
#pragma unroll
    for (int i = 0; i < PER; ++i) key[i] = own == i ? GONE : key[i];
  }
  float pw;
  if (SIGMOID) {
    pw = 1.f / (1.f + __expf(-row[my_id]));
  } else {
    const float mx = value(top);           // NaN if every key is
    float sum = 0.f;
#pragma unroll
    for (int i = 0; i < PER; ++i) sum += e0 + i < E ? __expf(x[i] - mx) : 0.f;
    pw = __expf(value(my_key) - mx) / row_reduce(sum, [](float a, float b) { return a + b; });
  }
  const float sel_sum = row_reduce(l < topk ? pw : 0.f, [](float a, float b) { return a + b; });
  id = my_id;
  w = (renorm ? pw / sel_sum : pw) * scale;
}

// Tokens t0 .. t0 + 64 / LANES - 1 (t0 < T) by one wave: ids and weights to memory.  Returns the expert of this lane's
// pick, -1 where the lane has none.
template <int LANES, int PER, bool SIGMOID>
__device__ __forceinline__ int moe_topk_tokens(const float* __restrict__ logits, const float* __restrict__ bias, int t0,
                                               int T, int E, int topk, int renorm, float scale, int* __restrict__ ids,
                                               float* __restrict__ wts) {
  const int lane = threadIdx.x & 63, l = lane % LANES, t = t0 + lane / LANES;
  const float* const row = logits + (size_t)min(t, T - 1) * E;
  int id;
  float w;
  if constexpr (LANES == 16) moe_pick_row<PER, SIGMOID>(row, bias, E, topk, renorm, scale, id, w);
  else moe_pick_wave<PER, SIGMOID>(row, bias, E, topk, renorm, scale, id, w);
  if (t >= T || l >= topk) return -1;
  ids[(size_t)t * topk + l] = id;
  wts[(size_t)t * topk + l] = w;
  return id;
}

template <int LANES, int PER, bool SIGMOID>
__global__ __launch_bounds__(256) void moe_topk_kernel(const float* __restrict__ logits,
                                                       const float* __restrict__ bias, int T, int E,
                                                       int topk, int renorm, float scale,
                                                       int* __restrict__ ids, float* __restrict__ wts) {
  const int t0 = (blockIdx.x * 4 + (threadIdx.x >> 6)) * (64 / LANES);
  if (t0 >= T) return;
  moe_topk_tokens<LANES, PER, SIGMOID>(logits, bias, t0, T, E, topk, renorm, scale, ids, wts);
}

// Tiles of the expert GEMMs made of up to MOE_RUN consecutive 16-slot blocks of one expert: runs[0] tiles, then
// first block * 32 + blocks of each (runs null: none wanted).
constexpr int MOE_RUN = 4;

// OR over the wave, wave-uniform.
__device__ __forceinline__ unsigned wave_or(unsigned v) {
  auto step = [&](auto CTRL, auto ROWS) {
    v |= (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, decltype(CTRL)::value, decltype(ROWS)::value, 0xf, false);
  };
  using std::integral_constant;
  step(integral_constant<int, 0x111>{}, integral_constant<int, 0xf>{});   // row_shr:1
  step(integral_constant<int, 0x112>{}, integral_constant<int, 0xf>{});   // row_shr:2
  step(integral_constant<int, 0x114>{}, integral_constant<int, 0xf>{});   // row_shr:4
  step(integral_constant<int, 0x118>{}, integral_constant<int, 0xf>{});   // row_shr:8
  step(integral_constant<int, 0x142>{}, integral_constant<int, 0xa>{});   // row_bcast:15 into rows 1, 3
  step(integral_constant<int, 0x143>{}, integral_constant<int, 0xc>{});   // row_bcast:31 into rows 2, 3
  return (unsigned)__builtin_amdgcn_readlane((int)v, 63);
}

// Inclusive prefix sum over the wave by DPP row shifts and row broadcasts.
__device__ __forceinline__ int wave_prefix_sum(int v) {
  auto step = [&](auto CTRL, auto ROWS) {
    v += __builtin_amdgcn_update_dpp(0, v, decltype(CTRL)::value, decltype(ROWS)::value, 0xf, false);
  };
  using std::integral_constant;
  step(integral_constant<int, 0x111>{}, integral_constant<int, 0xf>{});   // row_shr:1
  step(integral_constant<int, 0x112>{}, integral_constant<int, 0xf>{});   // row_shr:2
  step(integral_constant<int, 0x114>{}, integral_constant<int, 0xf>{});   // row_shr:4
  step(integral_constant<int, 0x118>{}, integral_constant<int, 0xf>{});   // row_shr:8
  step(integral_constant<int, 0x142>{}, integral_constant<int, 0xa>{});   // row_bcast:15 into rows 1, 3
  step(integral_constant<int, 0x143>{}, integral_constant<int, 0xc>{});   // row_bcast:31 into rows 2, 3
  return v;
}

// Exclusive prefix sum of padded[] by one wave, a lane owning a contiguous range of experts; and the tiles of
// each expert's run, as even as whole blocks allow.
__device__ __forceinline__ void moe_starts(const int* padded, int* start, int E, int lane, int* s_total,
                                           int* __restrict__ npp, int* __restrict__ runs) {
  const int per = (E + 63) / 64;
  int local = 0, tiles = 0;
  for (int k = 0; k < per; ++k) {
    const int e = lane * per + k;
    if (e < E) {
      local += padded[e];
      if (runs) tiles += (padded[e] / 16 + MOE_RUN - 1) / MOE_RUN;
    }
  }
  const int incl = wave_prefix_sum(local), tincl = runs ? wave_prefix_sum(tiles) : 0;
  int pos = incl - local, tpos = tincl - tiles;
  for (int k = 0; k < per; ++k) {
    const int e = lane * per + k;
    if (e >= E) break;
    start[e] = pos;
    if (runs) {
      const int b = padded[e] / 16, n = (b + MOE_RUN - 1) / MOE_RUN;
      for (int i = 0; i < n; ++i) {
        const int b0 = b * i / n, b1 = b * (i + 1) / n;
        runs[1 + tpos++] = (pos / 16 + b0) * 32 + (b1 - b0);
      }
    }
    pos += padded[e];
  }
  if (lane == 63) {
    *s_total = incl;
    if (npp) npp[0] = incl;
    if (runs) runs[0] = tincl;
  }
}

// Single workgroup of 16 waves.  Dynamic LDS: cnt[16][E] + padded[E] + start[E].
// Wave w owns the contiguous slice [w*seg, (w+1)*seg) of the flat slot list, so placing
// slices in wave order and slots in index order inside a slice gives a stable sort.  Inside a
// batch of 64 slots a lane's rank among equal expert ids is the number of lower lanes with
// the same id (a lane mask built from one ballot per id bit, no LDS round trips); the running
// position per (wave, expert) lives in LDS and is bumped by one LDS atomic per slot after all
// lanes of the batch have read it.
constexpr int MOE_ALIGN_WAVES = 16;
// PART = false: the whole job in one workgroup.  One workgroup scatters about one slot per clock, whatever it does, so
// that longer lists are split over the workgroups of a launch: PART = true places slots [s0, s1) only, from first[e] (LDS) on,
// see moe_align_parts_kernel.
template <bool PART>
__device__ __forceinline__ void moe_align_block(const int* __restrict__ ids, int n, int E, int tile_m,
                                                int cap, int* __restrict__ sorted,
                                                int* __restrict__ expert_ids, int* __restrict__ npp,
                                                int* __restrict__ runs, int* sm, int s0 = 0, int s1 = 0,
                                                const int* first = nullptr) {
  constexpr int NWV = MOE_ALIGN_WAVES;
  int* cnt = sm;               // [NWV][E], later the running write position
  int* padded = sm + NWV * E;  // [E]
  int* start = padded + E;     // [E]
  __shared__ int s_total;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  if (!PART) { s0 = 0; s1 = n; }

  for (int i = tid; i < NWV * E; i += 1024) cnt[i] = 0;
  __syncthreads();

  const int seg = ((s1 - s0 + NWV * 64 - 1) / (NWV * 64)) * 64;
  const int sb = s0 + wave * seg, se = min(s1, sb + seg);
  // ids are read eight batches of 64 at a time (eight loads in flight instead of one
  // dependent load per batch); the first eight batches stay in registers for the second pass
  constexpr int NB = 8;
  int head[NB];
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    const int i = sb + 64 * b + lane;
    head[b] = i < se ? ids[i] : -1;
  }
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    const int e = head[b];
    if (e >= 0 && e < E) atomicAdd(&cnt[wave * E + e], 1);
  }
  for (int c0 = sb + 64 * NB; c0 < se; c0 += 64 * NB) {
    int more[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      const int i = c0 + 64 * b + lane;
      more[b] = i < se ? ids[i] : -1;
    }
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      const int e = more[b];
      if (e >= 0 && e < E) atomicAdd(&cnt[wave * E + e], 1);
    }
  }
  __syncthreads();

  if constexpr (PART) {
    for (int e = tid; e < E; e += 1024) {
      int pos = first[e];
      for (int w = 0; w < NWV; ++w) { const int c = cnt[w * E + e]; cnt[w * E + e] = pos; pos += c; }
    }
    __syncthreads();
  } else {
  for (int e = tid; e < E; e += 1024) {
    int tot = 0;
    for (int w = 0; w < NWV; ++w) tot += cnt[w * E + e];
    padded[e] = (tot + tile_m - 1) / tile_m * tile_m;
  }
  __syncthreads();
  if (wave == 0) moe_starts(padded, start, E, lane, &s_total, npp, runs);
  __syncthreads();
  const int total = s_total;
  for (int e = tid; e < E; e += 1024) {
    int pos = start[e];
    const int e0 = pos;
    for (int w = 0; w < NWV; ++w) { const int c = cnt[w * E + e]; cnt[w * E + e] = pos; pos += c; }
    for (int i = pos; i < e0 + padded[e]; ++i) sorted[i] = n;            // pad entries
    for (int b = 0; b < padded[e] / tile_m; ++b) expert_ids[e0 / tile_m + b] = e;
  }
  for (int i = total + tid; i < cap; i += 1024) sorted[i] = n;           // unused tail
  for (int i = total / tile_m + tid; i < cap / tile_m; i += 1024) expert_ids[i] = -1;
  __syncthreads();
  }   // !PART

  const int nbits = 32 - __builtin_clz(max(E - 1, 1));
  auto place = [&](int i, int e) {
    const bool valid = e >= 0 && e < E;
    // lanes of the batch that hold the same expert id: one ballot per id bit
    unsigned long long same = __ballot(valid);
    for (int b = 0; b < nbits; ++b) {
      const bool bit = (e >> b) & 1;
      const unsigned long long bal = __ballot(bit);
      same &= bit ? bal : ~bal;
    }
    const int rank = __popcll(same & ((1ull << lane) - 1ull));   // equal ids in lower lanes
    int base = 0;
    if (valid) base = cnt[wave * E + e];
    __builtin_amdgcn_wave_barrier();
    if (valid) {
      sorted[base + rank] = i;
      atomicAdd(&cnt[wave * E + e], 1);
    }
  };
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    if (sb + 64 * b < se) place(sb + 64 * b + lane, head[b]);     // wave-uniform condition
  }
  for (int c0 = sb + 64 * NB; c0 < se; c0 += 64 * NB) {
    int more[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      const int i = c0 + 64 * b + lane;
      more[b] = i < se ? ids[i] : -1;
    }
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      if (c0 + 64 * b < se) place(c0 + 64 * b + lane, more[b]);
    }
  }
}

__global__ __launch_bounds__(1024) void moe_align_kernel(const int* __restrict__ ids, int n, int E,
                                                         int tile_m, int cap,
                                                         int* __restrict__ sorted,
                                                         int* __restrict__ expert_ids,
                                                         int* __restrict__ npp, int* __restrict__ runs) {
  extern __shared__ int sm[];
  moe_align_block<false>(ids, n, E, tile_m, cap, sorted, expert_ids, npp, runs, sm);
}

// Longer batches in two launches, part b of each one's workgroups being tokens [b * part, (b + 1) * part):
// the first picks the experts (16 lanes a token) and counts its part's picks, the second places them.
//
// (Four launches before from 16384 slots on: top-k, count, scan in one workgroup, place; 12.6 + 4.9 + 12.0 + 7.8 us for 8192 tokens,
// 128 experts, top-8, against 8.7 + 9.2.)
constexpr int MOE_PARTS_MAX = 128;
template <int PER, bool SIGMOID>
__global__ __launch_bounds__(1024) void moe_route_count_kernel(const float* __restrict__ logits, const float* __restrict__ bias,
                                                               int T, int E, int topk, int renorm, float scale,
                                                               int* __restrict__ ids, float* __restrict__ wts, int part,
                                                               int* __restrict__ part_cnt) {
  __shared__ int cnt[1024];      // E <= 1024
  const int tid = threadIdx.x, threads = blockDim.x;
  for (int e = tid; e < E; e += threads) cnt[e] = 0;
  __syncthreads();
  const int begin = (int)blockIdx.x * part, end = min(T, begin + part);
  for (int t0 = begin + (tid >> 6) * 4; t0 < end; t0 += (threads >> 6) * 4) {
    const int e = moe_topk_tokens<16, PER, SIGMOID>(logits, bias, t0, end, E, topk, renorm, scale, ids, wts);
    if (e >= 0) atomicAdd(&cnt[e], 1);
  }
  __syncthreads();
  for (int e = tid; e < E; e += threads) part_cnt[(size_t)blockIdx.x * E + e] = cnt[e];
}

// With a token a wave the picks need the whole chip, and have a launch of their own; a part's are counted from memory.  Block of 256 x 128, us,
// picked and counted by 128 workgroups / apart / top-k, count, scan and place: 2048, 8192, 16384 tokens, 8 of 1024 experts 89.5, 224, 402 / 86.9, 186,
// 319 / 113, 214, 345; 8 of 257 67.2, 179, 323 / 65.5, 156, 271 / 74.0, 166, 281; 65536 tokens, 2 of 1024 447 / 336 / 363.
__global__ __launch_bounds__(1024) void moe_count_kernel(const int* __restrict__ ids, int n, int E, int part,
                                                         int* __restrict__ part_cnt) {
  __shared__ int cnt[1024];      // E <= 1024
  const int tid = threadIdx.x;
  for (int e = tid; e < E; e += 1024) cnt[e] = 0;
  __syncthreads();
  const int s0 = min(n, (int)blockIdx.x * part), s1 = min(n, s0 + part);
  for (int i = s0 + tid; i < s1; i += 1024) atomicAdd(&cnt[ids[i]], 1);
  __syncthreads();
  for (int e = tid; e < E; e += 1024) part_cnt[(size_t)blockIdx.x * E + e] = cnt[e];
}

// Every workgroup adds up the table of counts (parts x E) by itself: each expert's slots in all and those of the parts before
// its own.  With the expert's start that is where its slots go; the padding, the block owners and the unused tails
// are shared out over the workgroups.  Dynamic LDS: moe_parts_lds(E).
__host__ __device__ constexpr int moe_parts_lds(int E) { return ((MOE_ALIGN_WAVES * E > 2048 ? MOE_ALIGN_WAVES * E : 2048) + 4 * E) * 4; }
__global__ __launch_bounds__(1024) void moe_align_parts_kernel(const int* __restrict__ ids, int n, int E, int part,
                                                               int tile_m, int cap, const int* __restrict__ part_cnt,
                                                               int* __restrict__ sorted, int* __restrict__ expert_ids,
                                                               int* __restrict__ npp, int* __restrict__ runs) {
  extern __shared__ int sm[];
  __shared__ int s_total;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, b = blockIdx.x, parts = gridDim.x;
  int* const padded = sm + max(MOE_ALIGN_WAVES * E, 2048);
  int* const start = padded + E;
  int* const count = start + E;
  int* const first = count + E;
  // threads (slice, expert): a slice takes every slices-th part; the sums of the slices meet in LDS
  const int slices = 1024 / E;
  if (tid < slices * E) {
    const int e = tid % E, s = tid / E;
    int all = 0, before = 0;
#pragma unroll 16
    for (int q = s; q < parts; q += slices) {
      const int c = part_cnt[(size_t)q * E + e];
      all += c;
      before += q < b ? c : 0;
    }
    sm[tid] = all;
    sm[1024 + tid] = before;
  }
  __syncthreads();
  if (tid < E) {
    int all = 0, before = 0;
    for (int s = 0; s < slices; ++s) {
      all += sm[s * E + tid];
      before += sm[1024 + s * E + tid];
    }
    count[tid] = all;
    first[tid] = before;
    padded[tid] = (all + tile_m - 1) / tile_m * tile_m;
  }
  __syncthreads();
  if (wave == 0) moe_starts(padded, start, E, lane, &s_total, b == 0 ? npp : nullptr, b == 0 ? runs : nullptr);
  __syncthreads();
  const int total = s_total;
  if (tid < E) first[tid] += start[tid];
  for (int e = b + wave * parts; e < E; e += MOE_ALIGN_WAVES * parts) {
    const int e0 = start[e], e1 = e0 + padded[e];
    for (int i = e0 + count[e] + lane; i < e1; i += 64) sorted[i] = n;
    for (int k = e0 / tile_m + lane; k < e1 / tile_m; k += 64) expert_ids[k] = e;
  }
  const int at = b * 1024 + tid, step = parts * 1024;
  for (int i = total + at; i < cap; i += step) sorted[i] = n;
  for (int i = total / tile_m + at; i < cap / tile_m; i += step) expert_ids[i] = -1;
  const int s0 = min(n, b * part), s1 = min(n, s0 + part);
  moe_align_block<true>(ids, n, E, tile_m, cap, sorted, nullptr, nullptr, nullptr, sm, s0, s1, first);
}

// Routing and align in one launch for up to MOE_ALIGN_WAVES * 64 / LANES tokens (the same single workgroup then sorts the
// T * topk slots): a decode step of a few sequences spends more on the second launch than on either kernel's work.
template <int LANES, int PER, bool SIGMOID>
__global__ __launch_bounds__(1024) void moe_route_align_kernel(const float* __restrict__ logits,
                                                               const float* __restrict__ bias, int T,
                                                               int E, int topk, int renorm, float scale,
                                                               int* ids, float* __restrict__ wts, int tile_m,
                                                               int cap, int* __restrict__ sorted,
                                                               int* __restrict__ expert_ids,
                                                               int* __restrict__ npp, int* __restrict__ runs) {
  extern __shared__ int sm[];
  __shared__ int s_ids[MOE_ALIGN_WAVES * 64];      // 16 waves of 64 / LANES tokens with up to LANES picks each
  const int lane = threadIdx.x & 63, t0 = (int)(threadIdx.x >> 6) * (64 / LANES);
  if (t0 < T) {
    const int e = moe_topk_tokens<LANES, PER, SIGMOID>(logits, bias, t0, T, E, topk, renorm, scale, ids, wts);
    if (e >= 0) s_ids[(t0 + lane / LANES) * topk + lane % LANES] = e;
  }
  __syncthreads();
  moe_align_block<false>(s_ids, T * topk, E, tile_m, cap, sorted, expert_ids, npp, runs, sm);
}

__global__ __launch_bounds__(256) void silu_and_mul_kernel(const half_t* __restrict__ in,
                                                           half_t* __restrict__ out, int rows,
                                                           int inter) {
  // 8 halves per thread; inter % 8 == 0
  const int per_row = inter / 8;
  const size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (idx >= (size_t)rows * per_row) return;
  const size_t r = idx / per_row, c = (idx % per_row) * 8;
  const h8 g = *reinterpret_cast<const h8*>(in + r * 2 * inter + c);
  const h8 u = *reinterpret_cast<const h8*>(in + r * 2 * inter + inter + c);
  h8 o;
#pragma unroll
  for (int i = 0; i < 8; ++i) o[i] = silu_mul(g[i], u[i]);
  *reinterpret_cast<h8*>(out + r * inter + c) = o;
}

__global__ __launch_bounds__(256) void moe_sum_kernel(const half_t* __restrict__ in,
                                                      half_t* __restrict__ out, int T, int topk,
                                                      int H) {
  const int per_row = H / 8;
  const size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (idx >= (size_t)T * per_row) return;
  const size_t t = idx / per_row, c = (idx % per_row) * 8;
  float s[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  // eight slot rows in flight at a time (a loop of single loads pays one memory round trip
  // per slot); the sum runs in slot order either way
  for (int j0 = 0; j0 < topk; j0 += 8) {
    h8 v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int j = min(j0 + u, topk - 1);
      v[u] = *reinterpret_cast<const h8*>(in + (t * topk + j) * H + c);
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      if (j0 + u < topk) {
#pragma unroll
        for (int i = 0; i < 8; ++i) s[i] += (float)v[u][i];
      }
    }
  }
  h8 o;
#pragma unroll
  for (int i = 0; i < 8; ++i) o[i] = (half_t)s[i];
  *reinterpret_cast<h8*>(out + t * H + c) = o;
}

}  // namespace awqmi
