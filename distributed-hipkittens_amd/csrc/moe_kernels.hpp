// Routing, scatter (permute), requantisation, combine and quantiser kernels
// for the gfx950 FP8 MoE path.  These are HBM/latency-bound integer and byte
// kernels: 16-byte coalesced accesses, LDS counters, wave-level ballots and
// shuffles -- no matrix cores.
//
// The reference contains none of these operations (no router, histogram,
// permutation or combine exists under /root/reference); their semantics are
// the path's frozen specification, restated on the CPU in oracle/spec.py.
#pragma once

#include "common.hpp"

#include <type_traits>

namespace hkmoe {

constexpr int kRouteTok = 32;      // tokens per routing/scatter workgroup
constexpr int kRouteThreads = 256; // scatter: 4 waves per 32-token block
constexpr int kTopkThreads = 512;  // top-k: 8 waves, 4 tokens each (16 lanes per token)
constexpr int kMaxExperts = 1024;
constexpr int kMaxTopK = 32;
constexpr int kScanThreads = 1024;
constexpr int kTileCounters = 16;  // HKMOE_TILE_COUNTERS
constexpr int kNarrowCounters = 4;  // narrow kernel item counters (GEMM 1, GEMM 2), then their
                                    // active-slot counters

// Logit as an unsigned key of the same order; equal logits (-0 and +0 too) have
// equal keys.  A NaN is below every number, and 0 is below every key.
__device__ __forceinline__ uint32_t route_key(float v) {
  const uint32_t u = __float_as_uint(v + 0.0f);  // -0 -> +0
  const uint32_t k = u ^ (static_cast<uint32_t>(static_cast<int32_t>(u) >> 31) | 0x80000000u);
  return __builtin_isnan(v) ? 1u : k;
}
__device__ __forceinline__ float route_value(uint32_t key) {
  const uint32_t u = (key & 0x80000000u) ? key ^ 0x80000000u : ~key;
  return __uint_as_float(key == 1u ? 0x7fc00000u : u);
}

// Reduction over the row of 16 lanes by DPP swaps (quad pairs, quad swap,
// half-row and row mirrors); every lane gets the result.
template <typename Op>
__device__ __forceinline__ uint32_t row16_reduce(uint32_t v, Op op) {
  auto step = [&](auto ctrl) __attribute__((always_inline)) {
    v = op(v, static_cast<uint32_t>(__builtin_amdgcn_update_dpp(static_cast<int>(v), static_cast<int>(v),
                                                                decltype(ctrl)::value, 0xf, 0xf, false)));
  };
  step(std::integral_constant<int, 0xB1>{});   // quad_perm [1,0,3,2]
  step(std::integral_constant<int, 0x4E>{});   // quad_perm [2,3,0,1]
  step(std::integral_constant<int, 0x141>{});  // row_half_mirror
  step(std::integral_constant<int, 0x140>{});  // row_mirror
  return v;
}

// ---------------------------------------------------------------------------
// 1. top-k + softmax + per-block histogram.  16 lanes (one row of the wave) per
//    token, 4 tokens per wave; lane s of a token's row holds experts c*16 + s,
//    c < CH (CH: power of two >= ceil(E / 16)).  Each of the k rounds takes
//    the row's largest key (integer maxima, then DPP swaps), the lowest expert
//    that has it (integer minima), and clears that key: VALU only, and a round's work
//    is shared by four tokens.  Carrying (value, expert) pairs through every
//    comparison took about twice the instructions.
// ---------------------------------------------------------------------------
// Token t's top-k on its row of 16 lanes: writes topk_idx / topk_w; lane sub gets
// the experts of slots sub and sub + 16 (where < top_k).
struct TopkLane {
  int e0, e1;
};
template <int CH>
__device__ __forceinline__ TopkLane route_token(const float* __restrict__ logits, int t, int num_experts, int top_k,
                                                int32_t* __restrict__ topk_idx, float* __restrict__ topk_w) {
  const int sub = threadIdx.x & 15;
  const float* row = logits + static_cast<int64_t>(t) * num_experts;
  uint32_t key[CH];
#pragma unroll
  for (int c = 0; c < CH; ++c) {
    const int id = c * 16 + sub;
    key[c] = (id < num_experts) ? route_key(row[id]) : 0u;
  }
  uint32_t first = 0, mk0 = 1, mk1 = 1;  // winners j (lane j % 16): j < 16 in mk0 / mi0, else mk1 / mi1
  int mi0 = 0, mi1 = 0;
  for (int j = 0; j < top_k; ++j) {
    uint32_t m = key[0];
#pragma unroll
    for (int c = 1; c < CH; ++c) m = max(m, key[c]);
    m = row16_reduce(m, [](uint32_t x, uint32_t y) { return max(x, y); });
    uint32_t best = 0xffffffffu;
#pragma unroll
    for (int c = CH - 1; c >= 0; --c) best = (key[c] == m) ? static_cast<uint32_t>(c * 16) : best;
    best = best == 0xffffffffu ? best : best + sub;
    best = row16_reduce(best, [](uint32_t x, uint32_t y) { return min(x, y); });
    const int mine = static_cast<int>(best) - sub;  // 16c in the lane that holds the winner
#pragma unroll
    for (int c = 0; c < CH; ++c) key[c] = (mine == c * 16) ? 0u : key[c];
    if (j == 0) first = m;
    if ((j & 15) == sub) {
      if (j < 16) { mk0 = m; mi0 = static_cast<int>(best); } else { mk1 = m; mi1 = static_cast<int>(best); }
    }
  }
  const float v0 = route_value(first), mv0 = route_value(mk0), mv1 = route_value(mk1);
  // softmax over the winners: exp(v_j - v_0) / sum_j exp(v_j - v_0), the sum
  // taken in j order
  const float ex0 = (sub < top_k) ? expf(mv0 - v0) : 0.0f;
  const float ex1 = (sub + 16 < top_k) ? expf(mv1 - v0) : 0.0f;
  float tot = 0.0f;
  for (int j = 0; j < top_k; ++j) tot = tot + __shfl(j < 16 ? ex0 : ex1, j & 15, 16);
  if (sub < top_k) {
    topk_idx[static_cast<int64_t>(t) * top_k + sub] = mi0;
    topk_w[static_cast<int64_t>(t) * top_k + sub] = ex0 / tot;
  }
  if (sub + 16 < top_k) {
    topk_idx[static_cast<int64_t>(t) * top_k + sub + 16] = mi1;
    topk_w[static_cast<int64_t>(t) * top_k + sub + 16] = ex1 / tot;
  }
  return TopkLane{mi0, mi1};
}

template <int CH>
__global__ __launch_bounds__(kTopkThreads) void route_topk_kernel(
    const float* __restrict__ logits, int num_tokens, int num_experts, int top_k,
    int32_t* __restrict__ topk_idx, float* __restrict__ topk_w, int32_t* __restrict__ block_counts) {
  static_assert(kTopkThreads == 16 * kRouteTok, "one 16-lane row per token");
  __shared__ int hist[kMaxExperts];
  const int sub = threadIdx.x & 15;
  for (int e = threadIdx.x; e < num_experts; e += kTopkThreads) hist[e] = 0;
  __syncthreads();

  const int t = blockIdx.x * kRouteTok + (threadIdx.x >> 4);
  if (t < num_tokens) {  // uniform over the token's row
    const TopkLane r = route_token<CH>(logits, t, num_experts, top_k, topk_idx, topk_w);
    if (sub < top_k) atomicAdd(&hist[r.e0], 1);
    if (sub + 16 < top_k) atomicAdd(&hist[r.e1], 1);
  }
  __syncthreads();
  for (int e = threadIdx.x; e < num_experts; e += kTopkThreads)
    block_counts[static_cast<int64_t>(blockIdx.x) * num_experts + e] = hist[e];
}

// ---------------------------------------------------------------------------
// 2. offsets, in two launches.
//  a. expert_block_scan: per expert, the exclusive prefix of its counts over
//     the routing blocks (block_base) and its total (counts).  kOffExperts
//     experts per workgroup, each over kOffParts ranges of blocks, so the
//     block counts are read by many CUs at once (a single workgroup spent
//     most of its time waiting for them).
//  b. expert_offsets: one workgroup of 1024 threads, thread = expert: scans
//     over experts (offsets, M-tile offsets), the M-tile list, counters.
// With at most kOffFuseBlocks routing blocks (decode-sized batches) the
// expert_offsets thread of each expert also does (a) itself, reading the few
// counts in one pass: one launch instead of two.
// ---------------------------------------------------------------------------
constexpr int kOffExperts = 16;                        // experts per block-scan workgroup
constexpr int kOffParts = kScanThreads / kOffExperts;  // block ranges per expert
constexpr int kOffCache = 32;                          // counts a thread keeps in registers
constexpr int kOffFuseBlocks = 16;                     // routing blocks done by expert_offsets

__global__ __launch_bounds__(kScanThreads) void expert_block_scan_kernel(
    const int32_t* __restrict__ block_counts, int nblk, int num_experts, int32_t* __restrict__ counts,
    int32_t* __restrict__ block_base) {
  __shared__ int part_sum[kOffParts][kOffExperts];
  const int tid = threadIdx.x;
  const int el = tid % kOffExperts, part = tid / kOffExperts;
  const int e = blockIdx.x * kOffExperts + el;
  const int per = (nblk + kOffParts - 1) / kOffParts;
  const int b0 = min(nblk, part * per), b1 = min(nblk, b0 + per);
  const bool act = e < num_experts;
  // up to kOffCache counts are loaded at once and kept for the block_base
  // pass; longer ranges are read twice, 16 loads in flight at a time
  const bool cached = per <= kOffCache;
  int cache[kOffCache];
  int s = 0;
  if (act && cached) {
#pragma unroll
    for (int u = 0; u < kOffCache; ++u)
      cache[u] = (b0 + u < b1) ? block_counts[static_cast<int64_t>(b0 + u) * num_experts + e] : 0;
#pragma unroll
    for (int u = 0; u < kOffCache; ++u) s += cache[u];
  } else if (act) {
    for (int b = b0; b < b1; b += 16) {
      int c[16];
#pragma unroll
      for (int u = 0; u < 16; ++u)
        c[u] = (b + u < b1) ? block_counts[static_cast<int64_t>(b + u) * num_experts + e] : 0;
#pragma unroll
      for (int u = 0; u < 16; ++u) s += c[u];
    }
  }
  part_sum[part][el] = s;
  __syncthreads();
  if (!act) return;
  // prefix over the ranges before this one, and the expert's total
  int before = 0, total = 0;
  for (int q = 0; q < kOffParts; ++q) {
    const int v = part_sum[q][el];
    if (q < part) before += v;
    total += v;
  }
  if (part == 0) counts[e] = total;
  int run = before;
  if (cached) {
#pragma unroll
    for (int u = 0; u < kOffCache; ++u) {
      if (b0 + u < b1) block_base[static_cast<int64_t>(b0 + u) * num_experts + e] = run;
      run += cache[u];
    }
  } else {
    for (int b = b0; b < b1; b += 16) {
      int c[16];
#pragma unroll
      for (int u = 0; u < 16; ++u)
        c[u] = (b + u < b1) ? block_counts[static_cast<int64_t>(b + u) * num_experts + e] : 0;
#pragma unroll
      for (int u = 0; u < 16; ++u) {
        if (b + u < b1) block_base[static_cast<int64_t>(b + u) * num_experts + e] = run;
        run += c[u];
      }
    }
  }
}

// Exclusive scans of N values per thread over the workgroup, all in one pass.
template <int N>
__device__ __forceinline__ void block_exclusive_scan_n(int (&v)[N], int (*wave_tot)[N]) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int incl[N];
#pragma unroll
  for (int i = 0; i < N; ++i) incl[i] = v[i];
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int n = __shfl_up(incl[i], o, 64);
      if (lane >= o) incl[i] += n;
    }
  }
  if (lane == 63) {
#pragma unroll
    for (int i = 0; i < N; ++i) wave_tot[wave][i] = incl[i];
  }
  __syncthreads();
  if (wave == 0) {
    const int nw = blockDim.x >> 6;
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int wv = lane < nw ? wave_tot[lane][i] : 0;
      int wi = wv;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const int n = __shfl_up(wi, o, 64);
        if (lane >= o) wi += n;
      }
      if (lane < nw) wave_tot[lane][i] = wi - wv;
    }
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < N; ++i) v[i] = wave_tot[wave][i] + incl[i] - v[i];
}

// The tables that follow from the experts' row counts (thread = expert, cnt 0
// past num_experts): offsets, M-tile offsets and list, counters reset.  Returns the
// expert's first row.
struct OffsetsLds {
  int wave_tot[kScanThreads / 64][5];
  int n_head, n_tail;
};
__device__ __forceinline__ int expert_offsets_tables(int e, int cnt, OffsetsLds& lds, int num_experts,
                                                     int32_t* __restrict__ offsets,
                                                     int32_t* __restrict__ mtile_offsets,
                                                     int32_t* __restrict__ mtile_list, int tile_m, float* amax_reset,
                                                     int32_t* tile_counters, int narrow_max, int32_t* narrow_info) {
  const int mt = (cnt + tile_m - 1) / tile_m;
  // M-tile list [(expert, first row)]: first the experts with at least one
  // full tile, each with all its tiles (full ones, then its partial one), in
  // expert order; then the single partial tiles of the smaller experts; last,
  // with narrow_max > 0, the experts of 1..narrow_max rows, which the narrow
  // kernel takes (their count goes to narrow_info[0]).  Tiles of nearly equal
  // cost sit together in the grouped GEMMs' schedule, so the workgroups that
  // share a tile block stay in step and reuse its operands in L2, and a large
  // expert's partial tile runs while its weights are still in L2 / MALL
  // instead of streaming them once more.
  const int q_full = cnt / tile_m;
  const int q_part = (cnt % tile_m) ? 1 : 0;
  const int q_head = q_full > 0 ? q_full + q_part : 0;
  const int q_narrow = (q_full == 0 && cnt > 0 && cnt <= narrow_max) ? 1 : 0;
  const int q_tail = (q_full > 0 || q_narrow) ? 0 : q_part;
  // one pass of exclusive scans over the experts: row offsets, M-tile
  // offsets, and the list positions of the three kinds of tiles
  int sc[5] = {cnt, mt, q_head, q_tail, q_narrow};
  block_exclusive_scan_n<5>(sc, lds.wave_tot);
  const int off = sc[0], moff = sc[1], head_base = sc[2], tail_base = sc[3], narrow_base = sc[4];
  if (e < num_experts) {
    offsets[e] = off;
    mtile_offsets[e] = moff;
  }
  if (e == num_experts - 1) {
    offsets[num_experts] = off + cnt;
    mtile_offsets[num_experts] = moff + mt;
    lds.n_head = head_base + q_head;
    lds.n_tail = tail_base + q_tail;
    if (mtile_list != nullptr && narrow_info != nullptr) narrow_info[0] = narrow_base + q_narrow;
  }
  if (mtile_list != nullptr) {
    __syncthreads();
    if (e < num_experts) {
      for (int s = 0; s < q_head; ++s) {
        mtile_list[2 * (head_base + s)] = e;
        mtile_list[2 * (head_base + s) + 1] = off + s * tile_m;
      }
      if (q_tail) {
        mtile_list[2 * (lds.n_head + tail_base)] = e;
        mtile_list[2 * (lds.n_head + tail_base) + 1] = off;
      }
      if (q_narrow) {
        mtile_list[2 * (lds.n_head + lds.n_tail + narrow_base)] = e;
        mtile_list[2 * (lds.n_head + lds.n_tail + narrow_base) + 1] = off;
      }
    }
  }
  const int tid = threadIdx.x;
  if (narrow_info != nullptr && tid >= 1 && tid < 1 + kNarrowCounters) narrow_info[tid] = 0;
  if (tid == 0 && amax_reset != nullptr) *amax_reset = 0.0f;
  if (tile_counters != nullptr && tid < kTileCounters) tile_counters[tid] = 0;
  return off;
}

// What small experts must save for the narrow kernels to take them beside larger
// ones: per_expert less per_row per row each, need in all (ns).  need 0: no condition.
struct NarrowRule {
  int32_t need = 0, per_expert = 0, per_row = 0;
};

// Largest expert for the narrow kernel: narrow_max, or 0 (none) where an expert is
// larger and the small ones do not save enough.  thread = expert; every thread calls it.
__device__ __forceinline__ int narrow_limit(int cnt, int narrow_max, const NarrowRule& rule) {
  __shared__ int saved;
  if (threadIdx.x == 0) saved = 0;
  if (rule.need <= 0 || !__syncthreads_or(cnt > narrow_max)) return narrow_max;
  int v = cnt > 0 && cnt <= narrow_max ? rule.per_expert - rule.per_row * cnt : 0;
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o, kWave);
  if ((threadIdx.x & 63) == 0) atomicAdd(&saved, v);
  __syncthreads();
  return saved >= rule.need ? narrow_max : 0;
}

__global__ __launch_bounds__(kScanThreads) void expert_offsets_kernel(
    int num_experts, int32_t* __restrict__ counts, int32_t* __restrict__ offsets,
    int32_t* __restrict__ mtile_offsets, int32_t* __restrict__ mtile_list, int tile_m,
    float* amax_reset, int32_t* tile_counters, int narrow_max, NarrowRule rule, int32_t* narrow_info,
    const int32_t* __restrict__ block_counts, int fused_nblk, int32_t* __restrict__ block_base) {
  __shared__ OffsetsLds lds;
  const int e = threadIdx.x;  // E <= kScanThreads
  int cnt = 0;
  if (fused_nblk >= 0) {
    // fused_nblk (<= kOffFuseBlocks) routing blocks: this expert's prefix over
    // them and its total, as expert_block_scan_kernel computes them (-1: the
    // block scan ran before)
    if (e < num_experts) {
      int c[kOffFuseBlocks];
#pragma unroll
      for (int b = 0; b < kOffFuseBlocks; ++b) c[b] = b < fused_nblk ? block_counts[b * num_experts + e] : 0;
#pragma unroll
      for (int b = 0; b < kOffFuseBlocks; ++b) {
        if (b < fused_nblk) block_base[b * num_experts + e] = cnt;
        cnt += c[b];
      }
      counts[e] = cnt;
    }
  } else if (e < num_experts) {
    cnt = counts[e];
  }
  narrow_max = narrow_limit(cnt, narrow_max, rule);
  expert_offsets_tables(e, cnt, lds, num_experts, offsets, mtile_offsets, mtile_list, tile_m, amax_reset,
                        tile_counters, narrow_max, narrow_info);
}

// Routing of at most kSmallTok tokens in one launch: top-k (16 lanes per token, as
// route_topk_kernel), offsets and the stable permutation.  Each expert keeps
// the set of its tokens as a 64-bit mask in LDS (a token names an expert at most once),
// so its count is a population count and a slot's place among the expert's rows
// the count of the mask below its token.  Three launches and their latencies in a
// decode step's critical path become one: E=128, k=8: 14.5 -> 8.1 us at T=1 (plus two
// launch gaps), 21.8 -> 12.7 us at T=64.
constexpr int kSmallTok = 64;
template <int CH>
__global__ __launch_bounds__(kScanThreads) void route_small_kernel(
    const float* __restrict__ logits, int num_tokens, int num_experts, int top_k, int32_t* __restrict__ topk_idx,
    float* __restrict__ topk_w, int32_t* __restrict__ counts, int32_t* __restrict__ offsets,
    int32_t* __restrict__ mtile_offsets, int32_t* __restrict__ mtile_list, int tile_m, float* amax_reset,
    int32_t* tile_counters, int narrow_max, NarrowRule rule, int32_t* narrow_info, int32_t* __restrict__ perm,
    int32_t* __restrict__ inv_perm) {
  static_assert(kScanThreads == 16 * kSmallTok && kScanThreads >= kMaxExperts, "thread = token lane, then expert");
  __shared__ OffsetsLds lds;
  __shared__ uint32_t tokens[kMaxExperts][2];  // bit t of the expert's token set
  __shared__ int first[kMaxExperts];
  const int tid = threadIdx.x, sub = tid & 15, t = tid >> 4;
  tokens[tid][0] = tokens[tid][1] = 0;
  __syncthreads();
  TopkLane r{0, 0};
  if (t < num_tokens) {  // uniform over the token's row
    r = route_token<CH>(logits, t, num_experts, top_k, topk_idx, topk_w);
    if (sub < top_k) atomicOr(&tokens[r.e0][t >> 5], 1u << (t & 31));
    if (sub + 16 < top_k) atomicOr(&tokens[r.e1][t >> 5], 1u << (t & 31));
  }
  __syncthreads();
  const int cnt = tid < num_experts ? __popc(tokens[tid][0]) + __popc(tokens[tid][1]) : 0;
  if (tid < num_experts) counts[tid] = cnt;
  narrow_max = narrow_limit(cnt, narrow_max, rule);
  first[tid] = expert_offsets_tables(tid, cnt, lds, num_experts, offsets, mtile_offsets, mtile_list, tile_m, amax_reset,
                                     tile_counters, narrow_max, narrow_info);
  __syncthreads();
  if (t < num_tokens) {
    auto place = [&](int e, int j) {
      const uint64_t set = tokens[e][0] | (static_cast<uint64_t>(tokens[e][1]) << 32);
      const int p = first[e] + __popcll(set & ((uint64_t{1} << t) - 1));
      const int f = t * top_k + j;
      perm[p] = f;
      inv_perm[f] = p;
    };
    if (sub < top_k) place(r.e0, sub);
    if (sub + 16 < top_k) place(r.e1, sub + 16);
  }
}

// ---------------------------------------------------------------------------
// 3. stable scatter + row gather.  Same token chunks as route_topk_kernel.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(kRouteThreads) void scatter_kernel(
    const int32_t* __restrict__ topk_idx, int num_tokens, int num_experts, int top_k,
    const int32_t* __restrict__ offsets, const int32_t* __restrict__ block_base,
    int32_t* __restrict__ perm, int32_t* __restrict__ inv_perm, const uint8_t* __restrict__ x_q,
    const float* __restrict__ x_scale, int64_t hidden, int block_scaled, uint8_t* __restrict__ xp,
    float* __restrict__ xps_t, int64_t rows_total) {
  __shared__ int ctr[kMaxExperts];
  __shared__ int pos[kRouteTok * kMaxTopK];
  const int lane = threadIdx.x & 63;
  const int t0 = blockIdx.x * kRouteTok;
  const int ntok = min(kRouteTok, num_tokens - t0);
  const int nslot = ntok * top_k;
  const int64_t f0 = static_cast<int64_t>(t0) * top_k;
  for (int e = threadIdx.x; e < num_experts; e += kRouteThreads)
    ctr[e] = offsets[e] + block_base[static_cast<int64_t>(blockIdx.x) * num_experts + e];
  __syncthreads();

  if (threadIdx.x < 64) {
    int nbits = 0;
    while ((1 << nbits) < num_experts) ++nbits;
    for (int s0 = 0; s0 < nslot; s0 += 64) {
      const int s = s0 + lane;
      const bool valid = s < nslot;
      const int e = valid ? topk_idx[f0 + s] : 0;
      uint64_t peers = __ballot(valid);
      for (int b = 0; b < nbits; ++b) {
        const bool bit = (e >> b) & 1;
        const uint64_t bal = __ballot(bit);
        peers &= bit ? bal : ~bal;
      }
      const uint64_t lt = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
      const int rank = __popcll(peers & lt);
      const int leader = valid ? (__ffsll(static_cast<long long>(peers)) - 1) : 0;
      int base = 0;
      if (valid && lane == leader) base = atomicAdd(&ctr[e], __popcll(peers));
      base = __shfl(base, leader, 64);
      if (valid) {
        const int p = base + rank;
        perm[p] = static_cast<int32_t>(f0 + s);
        inv_perm[f0 + s] = p;
        pos[s] = p;
      }
    }
  }
  __syncthreads();
  if (x_q == nullptr) return;

  // gather: each token row is read once and written to its top_k destinations
  const int64_t chunks = hidden / 16;
  const int64_t work = static_cast<int64_t>(ntok) * chunks;
  for (int64_t w = threadIdx.x; w < work; w += kRouteThreads) {
    const int tt = static_cast<int>(w / chunks);
    const int64_t c = w - static_cast<int64_t>(tt) * chunks;
    const uint4 v = *reinterpret_cast<const uint4*>(x_q + static_cast<int64_t>(t0 + tt) * hidden + c * 16);
    for (int j = 0; j < top_k; ++j) {
      const int p = pos[tt * top_k + j];
      *reinterpret_cast<uint4*>(xp + static_cast<int64_t>(p) * hidden + c * 16) = v;
    }
  }
  if (block_scaled) {
    const int groups = static_cast<int>(hidden / kGroup);
    const int swork = ntok * groups;
    for (int w = threadIdx.x; w < swork; w += kRouteThreads) {
      const int tt = w / groups, g = w - tt * groups;
      const float sv = x_scale[static_cast<int64_t>(t0 + tt) * groups + g];
      for (int j = 0; j < top_k; ++j)
        xps_t[static_cast<int64_t>(g) * rows_total + pos[tt * top_k + j]] = sv;
    }
  }
}

// ---------------------------------------------------------------------------
// 4. requantisation of the bf16 intermediate
// ---------------------------------------------------------------------------
// 1x128 groups: one workgroup (256 threads) per row, one wave per group.
__global__ __launch_bounds__(256) void requant_group_kernel(const uint16_t* __restrict__ h,
                                                            int64_t rows, int inter,
                                                            uint8_t* __restrict__ hq,
                                                            float* __restrict__ hs_t) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t r = blockIdx.x;
  const int groups = inter / kGroup;
  for (int g = wave; g < groups; g += 4) {
    const int64_t base = r * inter + g * kGroup + lane * 2;
    const uint32_t pair = *reinterpret_cast<const uint32_t*>(h + base);
    const float a = bf16_bits_to_f32(pair & 0xffffu), b = bf16_bits_to_f32(pair >> 16);
    const float amax = wave_max(fmaxf(fabsf(a), fabsf(b)));
    const float s = scale_from_amax(amax);
    const uint32_t q = pack_e4m3x4(quot_e4m3(a, s), quot_e4m3(b, s), 0.0f, 0.0f) & 0xffffu;
    *reinterpret_cast<uint16_t*>(hq + base) = static_cast<uint16_t>(q);
    if (lane == 0) hs_t[static_cast<int64_t>(g) * rows + r] = s;
  }
}

// per-tensor: amax was accumulated by GEMM 1 over the bf16-rounded h, so s is
// the scale of a bf16 maximum and every x is a bf16 value: the division-free
// quotient (QuotScale) gives the bytes of x / s there, as the GEMM epilogues'
// self-check establishes for that domain.  One case lies outside it: an
// infinite x with a finite s (amax NaN, s = 1), where x / s is x (saturated by
// the conversion) and the remainder step would give NaN.  8 elements per
// 16-byte chunk; each thread issues its 4 chunks' loads (read once:
// non-temporal) before converting any, so 4 KiB per wave are in flight.
__global__ __launch_bounds__(256) void requant_tensor_kernel(const uint16_t* __restrict__ h,
                                                             int64_t n8, const float* amax,
                                                             uint8_t* __restrict__ hq,
                                                             float* __restrict__ hs) {
  constexpr int kU = 4;
  const float s = scale_from_amax(*amax);
  const QuotScale qs = quot_scale(s);
  const bool s_finite = !__builtin_isinf(s);
  if (blockIdx.x == 0 && threadIdx.x == 0) hs[0] = s;
  auto quot = [&](uint32_t bits) __attribute__((always_inline)) {
    const float x = bf16_bits_to_f32(bits);
    const float q = quot_e4m3(x, qs);
    return (s_finite && __builtin_isinf(x)) ? x : q;
  };
  auto convert = [&](uint4 v) __attribute__((always_inline)) {
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
    uint2 o;
    uint32_t* op = &o.x;
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const uint32_t p0 = w[q * 2], p1 = w[q * 2 + 1];
      op[q] = pack_e4m3x4(quot(p0 & 0xffffu), quot(p0 >> 16), quot(p1 & 0xffffu), quot(p1 >> 16));
    }
    return o;
  };
  const int64_t stride = static_cast<int64_t>(gridDim.x) * 256;
  int64_t i = blockIdx.x * 256ll + threadIdx.x;
  for (; i + (kU - 1) * stride < n8; i += kU * stride) {
    uint4 v[kU];
#pragma unroll
    for (int u = 0; u < kU; ++u) v[u] = ld_nt16(h + (i + u * stride) * 8);
#pragma unroll
    for (int u = 0; u < kU; ++u) reinterpret_cast<uint2*>(hq)[i + u * stride] = convert(v[u]);
  }
  for (; i < n8; i += stride) reinterpret_cast<uint2*>(hq)[i] = convert(ld_nt16(h + i * 8));
}

// ---------------------------------------------------------------------------
// 5. combine: out[t] = bf16(sum_j w[t,j] * y[inv_perm[t*k+j]]), one
//    workgroup per token, 8 columns (16 bytes) per thread and step (the
//    host sizes the workgroup so the row's 16-byte chunks divide evenly).  The
//    token's weights and y rows are staged in LDS once; the y loads of up to
//    8 slots are issued together, then summed in slot order j = 0 .. k-1.
//    Every y byte is read once and every out byte written once: non-temporal
//    loads and stores (181 vs 208 us on config 3).
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(512) void combine_kernel(const uint16_t* __restrict__ y,
                                                      const float* __restrict__ topk_w,
                                                      const int32_t* __restrict__ inv_perm,
                                                      int top_k, int hidden,
                                                      uint16_t* __restrict__ out) {
  __shared__ float s_w[kMaxTopK];
  __shared__ int32_t s_row[kMaxTopK];
  const int64_t t = blockIdx.x;
  if (threadIdx.x < top_k) {
    s_w[threadIdx.x] = topk_w[t * top_k + threadIdx.x];
    s_row[threadIdx.x] = inv_perm[t * top_k + threadIdx.x];
  }
  __syncthreads();
  const int cols8 = hidden / 8;
  for (int c = threadIdx.x; c < cols8; c += blockDim.x) {
    float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    for (int j0 = 0; j0 < top_k; j0 += 8) {
      uint4 v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u)
        if (j0 + u < top_k)
          v[u] = ld_nt16(y + static_cast<int64_t>(s_row[j0 + u]) * hidden + c * 8);
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        if (j0 + u < top_k) {
          const float w = s_w[j0 + u];
          const uint32_t wv[4] = {v[u].x, v[u].y, v[u].z, v[u].w};
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            acc[2 * q] = acc[2 * q] + w * bf16_bits_to_f32(wv[q] & 0xffffu);
            acc[2 * q + 1] = acc[2 * q + 1] + w * bf16_bits_to_f32(wv[q] >> 16);
          }
        }
      }
    }
    uint4 o;
    o.x = pack_bf16x2(acc[0], acc[1]);
    o.y = pack_bf16x2(acc[2], acc[3]);
    o.z = pack_bf16x2(acc[4], acc[5]);
    o.w = pack_bf16x2(acc[6], acc[7]);
    st_nt16(out + t * hidden + c * 8, o);
  }
}

// ---------------------------------------------------------------------------
// Self-check of the epilogues' requantisation quotient: quot_e4m3(x, qs)
// against the correctly rounded x / s for every input the GEMM epilogues can
// produce: x a bf16 value, s = scale_from_amax(amax) with amax a bf16 value
// >= |x|.  Both quotients scale exactly with powers of two, so the check
// enumerates mantissas and sampled exponents: blocks (ma, ea) with amax =
// (1 + ma/128) 2^ea, ea = -126, -119, ..., 126; threads mx; each thread tries
// x = +-(1 + mx/128) 2^(ea - g), g = 0 .. 40 (x <= amax, x normal), and, in
// blocks with y in 37 .. 63, bf16 subnormals and zeros x = +-mx 2^-133
// against amax with ea in [-126, -100]; blocks with y = 64, amax = +inf (a row
// whose h overflowed) against finite and infinite x.  counts[0] += cases,
// counts[1] += mismatches: e4m3 bytes that differ, or fp32 quotients that
// differ where |x / s| >= 2^-10 (signed zeros included; two NaNs agree).
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(128) void requant_quotient_check_kernel(int* __restrict__ counts) {
  const int ma = blockIdx.x, mx = threadIdx.x;
  if (blockIdx.y == 64) {
    // a row whose h overflowed: amax = +inf, s = +inf; x = +-(1 + mx/128) 2^e for
    // e = -126 + ma*2 (block ma < 127), or x = +-inf (block 127, thread 0)
    const QuotScale qs = quot_scale(scale_from_amax(__builtin_inff()));
    const float s = scale_from_amax(__builtin_inff());
    int cases = 0, bad = 0;
    if (ma < 127 || mx == 0) {
      const float x = ma < 127 ? __builtin_amdgcn_ldexpf(1.0f + mx / 128.0f, -126 + 2 * ma) : __builtin_inff();
#pragma unroll
      for (int sg = 0; sg < 2; ++sg) {
        const float xv = sg ? -x : x;
        const float qd = quot_e4m3(xv, s), qm = quot_e4m3(xv, qs);
        // both NaN (inf / inf; its sign is not specified), or the same bits
        bad += !((__builtin_isnan(qd) && __builtin_isnan(qm)) || __float_as_uint(qd) == __float_as_uint(qm));
        ++cases;
      }
    }
    atomicAdd(&counts[0], cases);
    atomicAdd(&counts[1], bad);
    return;
  }
  const bool sub = blockIdx.y >= 37;
  const int ea = sub ? -126 + static_cast<int>(blockIdx.y - 37) : -126 + 7 * static_cast<int>(blockIdx.y);
  const float amax = __builtin_amdgcn_ldexpf(1.0f + ma / 128.0f, ea);
  const float s = scale_from_amax(amax);
  const QuotScale qs = quot_scale(s);
  int cases = 0, bad = 0;
  for (int g = 0; g <= (sub ? 0 : 40); ++g) {
    float x;
    if (sub) {
      x = __builtin_amdgcn_ldexpf(static_cast<float>(mx), -133);  // mx = 0: +-0
    } else {
      if (ea - g < -126) break;
      if (g == 0 && mx > ma) continue;  // x <= amax
      x = __builtin_amdgcn_ldexpf(1.0f + mx / 128.0f, ea - g);
    }
#pragma unroll
    for (int sg = 0; sg < 2; ++sg) {
      const float xv = sg ? -x : x;
      const float qd = quot_e4m3(xv, s), qm = quot_e4m3(xv, qs);
      // the stored e4m3 bytes must agree, and the fp32 quotients too wherever
      // they can round to a nonzero e4m3 value
      const bool same_byte = (pack_e4m3x4(qd, 0.0f, 0.0f, 0.0f) & 0xffu) == (pack_e4m3x4(qm, 0.0f, 0.0f, 0.0f) & 0xffu);
      const bool same_bits = __float_as_uint(qd) == __float_as_uint(qm) || fabsf(qd) < 0.0009765625f;
      bad += !(same_byte && same_bits);
      ++cases;
    }
  }
  atomicAdd(&counts[0], cases);
  atomicAdd(&counts[1], bad);
}

// ---------------------------------------------------------------------------
// 6. quantisers (fp32 input) used to build e4m3 operands on the device
//
// All are one pass over HBM (4 bytes read, 1 written per value; the per-tensor
// one reads twice, the second time partly from the Infinity Cache), so they
// are built to keep enough 16-byte loads in flight: every thread issues its
// loads before it uses any.  x may be aligned to 4 bytes only and q to 1 (a
// view into a larger tensor): the vector types below say so, and the hardware
// takes such addresses at full width.  At 8192x7168 (5 bytes per value): groups
// 126 -> 49 us (2.3 -> 6.0 TB/s), blocks 88 -> 50 us (5.8 TB/s), MX 54 -> 50 us
// (5.9 TB/s), per-tensor 305 -> 95 us; what bounded them was a 512-byte wave load
// at a time, the IEEE division per value, and 16384 same-address atomics.
// ---------------------------------------------------------------------------
typedef float f32x4_u __attribute__((ext_vector_type(4), aligned(4)));
typedef uint32_t u32_u __attribute__((aligned(1)));

// Maximum over the row of 16 lanes, by DPP.  fmaxf skips NaNs.
__device__ __forceinline__ float row16_max(float v) {
  auto step = [&](auto ctrl) __attribute__((always_inline)) {
    v = fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(v), __float_as_int(v),
                                                            decltype(ctrl)::value, 0xf, 0xf, false)));
  };
  step(std::integral_constant<int, 0xB1>{});   // quad_perm [1,0,3,2]
  step(std::integral_constant<int, 0x4E>{});   // quad_perm [2,3,0,1]
  step(std::integral_constant<int, 0x141>{});  // row_half_mirror
  step(std::integral_constant<int, 0x140>{});  // row_mirror
  return v;
}

__device__ __forceinline__ float max_abs4(f32x4 v) {
  return fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w)));
}

// Four values / sc as e4m3 bytes.  Finite values take the division-free
// quotient (quot_e4m3 with QuotScale: the theorem named there holds for every fp32 x
// <= 448 sc with x / sc >= 2^-10, and below that both quotients round to 0) and
// the packed conversion; a NaN or an infinite scale keeps the division and the
// software conversion (NaN code 0x7f | sign).
__device__ __forceinline__ uint32_t quant4(f32x4 v, float sc, const QuotScale& qs) {
  const bool odd = __builtin_isunordered(v.x, v.y) || __builtin_isunordered(v.z, v.w) || __builtin_isinf(sc);
  if (__builtin_expect(odd, 0))
    return f32_to_e4m3(v.x / sc) | (f32_to_e4m3(v.y / sc) << 8) | (f32_to_e4m3(v.z / sc) << 16) |
           (f32_to_e4m3(v.w / sc) << 24);
  return pack_e4m3x4(quot_e4m3(v.x, qs), quot_e4m3(v.y, qs), quot_e4m3(v.z, qs), quot_e4m3(v.w, qs));
}

// 1x128 groups, row-major scales [R, C/128].  C is a multiple of 128, so x is
// a flat run of groups.  16 lanes per group, 8 values each (the scale's
// reciprocal is shared by 8 values, and the maximum stays inside a DPP row),
// two groups per lane row: four 16-byte loads in flight per thread.
constexpr int kQuantGroups = 32;  // groups per workgroup
__global__ __launch_bounds__(256) void quant_group_kernel(const float* __restrict__ x, int64_t groups,
                                                          uint8_t* __restrict__ q, float* __restrict__ s) {
  const int l = threadIdx.x & 15;
  const int64_t g0 = blockIdx.x * static_cast<int64_t>(kQuantGroups) + (threadIdx.x >> 4);
  f32x4 v[2][2];
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int64_t g = g0 + 16 * u;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      v[u][h] = f32x4{0.f, 0.f, 0.f, 0.f};
      if (g < groups)
        v[u][h] = __builtin_nontemporal_load(reinterpret_cast<const f32x4_u*>(x + g * kGroup + 64 * h + 4 * l));
    }
  }
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int64_t g = g0 + 16 * u;
    const float sc = scale_from_amax(row16_max(fmaxf(max_abs4(v[u][0]), max_abs4(v[u][1]))));
    const QuotScale qs = quot_scale(sc);
    if (g < groups) {
#pragma unroll
      for (int h = 0; h < 2; ++h)
        *reinterpret_cast<u32_u*>(q + g * kGroup + 64 * h + 4 * l) = quant4(v[u][h], sc, qs);
      if (l == 0) s[g] = sc;
    }
  }
}

// 128x128 blocks of [B, R, C]; one workgroup (256 threads) per block, the
// block held in registers (64 per thread) between the maximum and the
// conversion, so x is read once.
__global__ __launch_bounds__(256) void quant_block_kernel(const float* __restrict__ x, int64_t rows,
                                                          int64_t cols, uint8_t* __restrict__ q,
                                                          float* __restrict__ s) {
  __shared__ float red[4];
  const int64_t bc = cols / kGroup, br = rows / kGroup;
  const int64_t blk = blockIdx.x;
  const int64_t b = blk / (br * bc);
  const int64_t rem = blk - b * br * bc;
  const int64_t bi = rem / bc, bj = rem - bi * bc;
  const float* xb = x + (b * rows + bi * kGroup) * cols + bj * kGroup;
  uint8_t* qb = q + (b * rows + bi * kGroup) * cols + bj * kGroup;
  // thread: rows (tid/32) + 8*u, columns 4*(tid%32) .. +3
  const int cr = threadIdx.x >> 5, cc = (threadIdx.x & 31) * 4;
  f32x4 v[16];
#pragma unroll
  for (int u = 0; u < 16; ++u)
    v[u] = __builtin_nontemporal_load(
        reinterpret_cast<const f32x4_u*>(xb + static_cast<int64_t>(cr + 8 * u) * cols + cc));
  float m = 0.0f;
#pragma unroll
  for (int u = 0; u < 16; ++u) m = fmaxf(m, max_abs4(v[u]));
  m = wave_max(m);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
  __syncthreads();
  const float sc = scale_from_amax(fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3])));
  const QuotScale qs = quot_scale(sc);
#pragma unroll
  for (int u = 0; u < 16; ++u)
    *reinterpret_cast<u32_u*>(qb + static_cast<int64_t>(cr + 8 * u) * cols + cc) = quant4(v[u], sc, qs);
  if (threadIdx.x == 0) s[blk] = sc;
}

// Per-tensor: the maximum over all values, then the conversion.
constexpr int kAmaxUnroll = 4;  // 16-byte loads in flight per thread

// max |x| over n values, seen by a workgroup of THREADS threads that reads the
// 4-value chunks first, first + step, ...; the last n % 4 values go to the
// first chunk's owner.
template <int THREADS>
__device__ __forceinline__ float amax_range(const float* __restrict__ x, int64_t n, int64_t first, int64_t step) {
  const int64_t n4 = n / 4;
  float m = 0.0f;
  int64_t i = first;
  for (; i + (kAmaxUnroll - 1) * step < n4; i += kAmaxUnroll * step) {
    f32x4 v[kAmaxUnroll];
#pragma unroll
    for (int u = 0; u < kAmaxUnroll; ++u) v[u] = reinterpret_cast<const f32x4_u*>(x)[i + u * step];
#pragma unroll
    for (int u = 0; u < kAmaxUnroll; ++u) m = fmaxf(m, max_abs4(v[u]));
  }
  for (; i < n4; i += step) m = fmaxf(m, max_abs4(reinterpret_cast<const f32x4_u*>(x)[i]));
  if (first == 0)
    for (int64_t j = 4 * n4; j < n; ++j) m = fmaxf(m, fabsf(x[j]));
  __shared__ float red[THREADS / 64];
  m = wave_max(m);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < THREADS / 64; ++w) m = fmaxf(m, red[w]);
  return m;
}

// Chunks first, first + step, ... of x converted with scale sc.
__device__ __forceinline__ void quant_range(const float* __restrict__ x, int64_t n, int64_t first, int64_t step,
                                            float sc, uint8_t* __restrict__ q) {
  const QuotScale qs = quot_scale(sc);
  const int64_t n4 = n / 4;
  int64_t i = first;
  for (; i + (kAmaxUnroll - 1) * step < n4; i += kAmaxUnroll * step) {
    f32x4 v[kAmaxUnroll];
#pragma unroll
    for (int u = 0; u < kAmaxUnroll; ++u) v[u] = reinterpret_cast<const f32x4_u*>(x)[i + u * step];
#pragma unroll
    for (int u = 0; u < kAmaxUnroll; ++u) *reinterpret_cast<u32_u*>(q + 4 * (i + u * step)) = quant4(v[u], sc, qs);
  }
  for (; i < n4; i += step)
    *reinterpret_cast<u32_u*>(q + 4 * i) = quant4(reinterpret_cast<const f32x4_u*>(x)[i], sc, qs);
  if (first == 0)
    for (int64_t j = 4 * n4; j < n; ++j) q[j] = static_cast<uint8_t>(f32_to_e4m3(x[j] / sc));
}

// One atomic per workgroup at most: a workgroup whose maximum is not above the
// one already published skips it (the value only grows, so a stale read costs
// an atomic, not the result).
__global__ __launch_bounds__(256) void amax_kernel(const float* __restrict__ x, int64_t n, float* amax) {
  const float m = amax_range<256>(x, n, blockIdx.x * 256ll + threadIdx.x, static_cast<int64_t>(gridDim.x) * 256);
  if (threadIdx.x == 0 && m > __hip_atomic_load(amax, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
    atomicMax(reinterpret_cast<unsigned int*>(amax), __float_as_uint(m));
}

__global__ void fill_f32_kernel(float* p, float v) { *p = v; }

__global__ __launch_bounds__(256) void quant_tensor_kernel(const float* __restrict__ x, int64_t n,
                                                           const float* amax,
                                                           uint8_t* __restrict__ q,
                                                           float* __restrict__ s) {
  const float sc = scale_from_amax(*amax);
  if (blockIdx.x == 0 && threadIdx.x == 0) s[0] = sc;
  quant_range(x, n, blockIdx.x * 256ll + threadIdx.x, static_cast<int64_t>(gridDim.x) * 256, sc, q);
}

// Small tensors: one launch.  Every workgroup takes the maximum over the whole
// tensor (its XCD's L2 holds it) and converts its own share.
constexpr int64_t kQuantSmall = 1 << 17;  // values
__global__ __launch_bounds__(1024) void quant_tensor_small_kernel(const float* __restrict__ x, int64_t n,
                                                                  uint8_t* __restrict__ q, float* __restrict__ s) {
  const float sc = scale_from_amax(amax_range<1024>(x, n, threadIdx.x, 1024));
  if (blockIdx.x == 0 && threadIdx.x == 0) s[0] = sc;
  quant_range(x, n, blockIdx.x * 1024ll + threadIdx.x, static_cast<int64_t>(gridDim.x) * 1024, sc, q);
}

// ---------------------------------------------------------------------------
// 7. MX (e8m0 1x32) operands
// ---------------------------------------------------------------------------
// x viewed as [blocks, 32] (row-major [R, C] with C % 32 == 0): 8 lanes per
// block, 4 elements each.  s = biased exponent of amax = clamp(floor(log2 amax)
// + 127, 0, 254) -- exact for every finite amax (0 for zero or subnormal amax)
// -- and q = e4m3(x * 2^(127 - s)), an exact power-of-two scaling followed by
// one RNE conversion (|x * 2^(127-s)| < 2, so the saturating clamp never acts).
// Reference behaviour: 4_wave.cu:296-321, 368-373.
// Each workgroup owns 256 U quads; a thread's U loads are in flight together.  Up to
// kMxSmall values two loads, kept in the caches: fewer per thread spread a small
// tensor over more CUs (64x4096 1.9 us, four loads 2.2), and x was written just
// before it is quantised (1024x7168 with six inputs in turn 7.0 us, non-temporal
// 7.9).  Above, four non-temporal ones (4096x7168 in turn 23.7 us, else 26.9).
constexpr int64_t kMxSmall = 1 << 23;
template <int U, bool NT>
__global__ __launch_bounds__(256) void quant_mx_kernel(const float* __restrict__ x, int64_t blocks,
                                                       uint8_t* __restrict__ q, uint8_t* __restrict__ s) {
  const int64_t quads = blocks * 8;
  // quad i = lane i % 8 of block i / 8; the 8 lanes of a block sit in one DPP
  // row (i % 8 == threadIdx.x % 8) and are in or out of range together
  const int64_t i0 = blockIdx.x * static_cast<int64_t>(256 * U) + threadIdx.x;
  f32x4 v[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const f32x4_u* src = reinterpret_cast<const f32x4_u*>(x) + i0 + 256 * u;
    v[u] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (i0 + 256 * u < quads) v[u] = NT ? __builtin_nontemporal_load(src) : *src;
  }
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int64_t i = i0 + 256 * u;
    float m = max_abs4(v[u]);
    m = fmaxf(m, __shfl_xor(m, 1, kWave));
    m = fmaxf(m, __shfl_xor(m, 2, kWave));
    m = fmaxf(m, __shfl_xor(m, 4, kWave));
    const uint32_t e = min((__float_as_uint(m) >> 23) & 0xffu, 254u);
    const int sh = 127 - static_cast<int>(e);
    if (i < quads) {
      *reinterpret_cast<u32_u*>(q + 4 * i) =
          pack_e4m3x4(__builtin_amdgcn_ldexpf(v[u].x, sh), __builtin_amdgcn_ldexpf(v[u].y, sh),
                      __builtin_amdgcn_ldexpf(v[u].z, sh), __builtin_amdgcn_ldexpf(v[u].w, sh));
      if ((i & 7) == 0) s[i >> 3] = static_cast<uint8_t>(e);
    }
  }
}

// e8m0 s [R, C/32] -> packed words [C/128, R64] (R64 = R rounded up to 64):
// word (kt, p) byte g = s[64*(p/64) + 16*g + p%16][4*kt + (p%64)/16], 0 past
// row R.  One thread per word.  Same words as the reference's pack_scales_kernel
// + repack_scales_for_mfma_kernel (4_wave.cu:323-364) when R % 64 == 0.
__global__ __launch_bounds__(256) void mx_pack_scales_kernel(const uint8_t* __restrict__ s, int64_t rows,
                                                             int64_t kblocks, int64_t rows64,
                                                             uint32_t* __restrict__ packed,
                                                             int64_t words) {
  for (int64_t w = blockIdx.x * 256ll + threadIdx.x; w < words; w += static_cast<int64_t>(gridDim.x) * 256) {
    const int64_t kt = w / rows64, p = w - kt * rows64;
    const int64_t r0 = (p & ~63ll) + (p & 15);
    const int64_t kb = 4 * kt + ((p >> 4) & 3);
    uint32_t v = 0;
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int64_t r = r0 + 16 * g;
      if (r < rows) v |= static_cast<uint32_t>(s[r * kblocks + kb]) << (8 * g);
    }
    packed[w] = v;
  }
}

// Weight exponents e8m0 [E, nb, K/32] -> the grouped MX GEMM's words, per B
// tile: [E][nb/256][K/128][256], word p of (expert e, N tile nt, K step kt)
// holds in byte g the exponent of B-tile row R = 64*(p/64) + 16g + p%16 for K
// block 4kt + (p%64)/16.  B-tile row R is weight row nt*256 + R, or for the
// fused gate/up weights (gate_up = I) row nt*128 + 32*(R>>6) + (R&31) +
// ((R>>5)&1)*I: the row order of pack_weights_kernel's stage images.
__global__ __launch_bounds__(256) void mx_pack_weight_words_kernel(const uint8_t* __restrict__ s, int64_t nb,
                                                                   int K, int gate_up,
                                                                   uint32_t* __restrict__ out,
                                                                   int64_t words) {
  const int ks = K / 128, kb = K / 32;
  const int64_t ntile = nb / 256;
  for (int64_t w = blockIdx.x * 256ll + threadIdx.x; w < words; w += static_cast<int64_t>(gridDim.x) * 256) {
    const int pos = static_cast<int>(w & 255);
    const int64_t t = w >> 8;
    const int kt = static_cast<int>(t % ks);
    const int64_t tile = t / ks;
    const int64_t e = tile / ntile;
    const int nt = static_cast<int>(tile - e * ntile);
    const int blk = 4 * kt + ((pos >> 4) & 3);
    uint32_t v = 0;
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int R = (pos & ~63) + 16 * g + (pos & 15);
      const int64_t wrow = gate_up ? nt * 128 + 32 * (R >> 6) + (R & 31) + ((R >> 5) & 1) * gate_up
                                   : static_cast<int64_t>(nt) * 256 + R;
      v |= static_cast<uint32_t>(s[(e * nb + wrow) * kb + blk]) << (8 * g);
    }
    out[w] = v;
  }
}

// Activation exponents e8m0 [x_rows, K/32] -> tile-aligned words in expert
// order: [K/128][ws_rs], word m*256 + q of K step kt (M tile m in expert order,
// first row row0, `valid` rows) holds in byte g the exponent of tile row
// r = 64*(q/64) + 16g + q%16 -- output row row0 + r, read from x row
// gather[row0 + r] / gather_div (or row0 + r) -- for K block 4kt + (q%64)/16;
// 0 for r >= valid.
// One workgroup per M tile: the tile's expert is found once, its (gathered)
// rows' exponent bytes are copied into LDS as whole rows (4-byte loads along
// each row), and thread q then writes word q of every K step (consecutive
// threads, consecutive words).  K <= 16384: at most 512 bytes per row.
constexpr int kMxGatherMaxKb = 16384 / 32;
__global__ __launch_bounds__(256) void mx_gather_words_kernel(const uint8_t* __restrict__ s, int K,
                                                              const int32_t* __restrict__ gather, int gather_div,
                                                              const int32_t* __restrict__ offsets,
                                                              const int32_t* __restrict__ mtile_offsets,
                                                              int num_experts, int64_t ws_rs,
                                                              uint32_t* __restrict__ out) {
  extern __shared__ __attribute__((aligned(16))) uint8_t rows_s[];  // [256][kb] exponent bytes
  __shared__ int s_row0, s_valid;
  __shared__ int64_t xrow_s[256];  // x row of each tile row, -1 past `valid`
  const int kb = K / 32, ks = K / 128;
  const int n_mt = mtile_offsets[num_experts];
  const int tid = threadIdx.x;
  for (int m = blockIdx.x; m < n_mt; m += gridDim.x) {
    if (tid == 0) {
      int lo = 0, hi = num_experts;  // largest e with mtile_offsets[e] <= m
      while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (mtile_offsets[mid] <= m) lo = mid; else hi = mid;
      }
      const int row0 = offsets[lo] + (m - mtile_offsets[lo]) * 256;
      s_row0 = row0;
      s_valid = min(256, offsets[lo + 1] - row0);
    }
    __syncthreads();
    {
      const int row0 = s_row0, valid = s_valid;
      xrow_s[tid] = tid < valid ? (gather ? gather[row0 + tid] / gather_div : row0 + tid) : -1;
    }
    __syncthreads();
    // the rows' bytes in chunks of 16 (K a multiple of 512 and s 16-byte
    // aligned) or 4, up to 16 loads in flight per thread; rows past `valid`
    // read as zero bytes
    auto copy_rows = [&](auto chunk_tag) __attribute__((always_inline)) {
      using C = decltype(chunk_tag);
      constexpr int kC = sizeof(C);
      const int per_row = kb / kC, total = 256 * per_row;
      for (int base = 0; base < total; base += 256 * 16) {
        C v[16];
#pragma unroll
        for (int u = 0; u < 16; ++u) {
          const int i = base + u * 256 + tid;
          v[u] = C{};
          if (i < total) {
            const int r = i / per_row, c = i - r * per_row;
            const int64_t xr = xrow_s[r];
            if (xr >= 0) v[u] = reinterpret_cast<const C*>(s + xr * kb)[c];
          }
        }
#pragma unroll
        for (int u = 0; u < 16; ++u) {
          const int i = base + u * 256 + tid;
          if (i < total) reinterpret_cast<C*>(rows_s)[i] = v[u];
        }
      }
    };
    if (kb % 16 == 0 && (reinterpret_cast<uintptr_t>(s) & 15) == 0) copy_rows(uint4{}); else copy_rows(uint32_t{});
    __syncthreads();
    const int q = tid;
    const int rbase = (q & ~63) + (q & 15), bsub = (q >> 4) & 3;
    uint32_t* dst = out + static_cast<int64_t>(m) * 256 + q;
    for (int kt = 0; kt < ks; ++kt) {
      const int blk = 4 * kt + bsub;
      uint32_t v = 0;
#pragma unroll
      for (int g = 0; g < 4; ++g) v |= static_cast<uint32_t>(rows_s[(rbase + 16 * g) * kb + blk]) << (8 * g);
      dst[static_cast<int64_t>(kt) * ws_rs] = v;
    }
    __syncthreads();  // rows_s is rewritten for the next M tile
  }
}

}  // namespace hkmoe
