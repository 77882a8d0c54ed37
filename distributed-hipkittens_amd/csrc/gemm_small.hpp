// Dense FP8 GEMM for problems with too few 256x256 tiles to fill the chip (and
// too many rows for the strips of gemm_skinny.hpp): C[M,N] = (sa*sb) * A[M,K] .
// B[N,K]^T with per-tensor scales or MX exponents, bf16 or fp32 C.
//
// 128x128 output tiles, one non-persistent workgroup of 8 waves per tile, two
// waves per SIMD, each wave 64x32 outputs: 4x2 v_mfma_f32_16x16x128_f8f6f4 per
// K step, or (M32) two blocks of 32x32 outputs, each two
// v_mfma_f32_32x32x64_f8f6f4 (the two 64-byte halves of the K step).
// A K step is bounded by one wave's issue of fragment reads and DMA beside its
// MFMAs: each wave overlaps its own LDS fragment reads of step kt+1 with its MFMAs
// of step kt (two register sets of fragments), and the second wave of the SIMD fills
// what is left.  Against 4 waves of 64x64, one per SIMD, which read a quarter less
// from LDS (graph-replayed launches, one box, operands resident / rotating over 512 MB):
// 2048^3 12.7 -> 11.3 / 13.8 -> 13.7 us, 512x4096x4096 19.5 -> 16.8 / 21.4 -> 20.5,
// 1024x2048x7168 30.6 -> 26.8 / 34.6 -> 33.1.  A 4-deep LDS ring fed by buffer->LDS DMA keeps
// three K steps (96 KiB per CU) in flight (a fifth stage measured slower).  The
// 2048^3 GEMM (config 1) is 256 such tiles, one per CU, where the 256x256 kernel has
// 64.
#pragma once

#include "gemm_fp8.hpp"

namespace hkmoe {

constexpr int kSmTile = 128;                         // output tile edge
constexpr int kSmThreads = 512;                      // 8 waves, two per SIMD
constexpr int kSmStages = 4;                         // LDS ring depth (K steps)
constexpr int kSmAhead = kSmStages - 1;              // K steps in flight beyond the current one
constexpr int kSmOperandBytes = kSmTile * kBK;       // 16 KiB per operand per step
constexpr int kSmStageBytes = 2 * kSmOperandBytes;   // A then B
constexpr int kSmWordBytes = 2 * kSmTile * 4;           // MX: exponent words of A, then B
constexpr int sm_stage_bytes(bool mx) { return kSmStageBytes + (mx ? kSmWordBytes : 0); }
constexpr int sm_lds_bytes(bool mx) { return kSmStages * sm_stage_bytes(mx); }  // 128 KiB (132 KiB)
static_assert(sm_lds_bytes(true) <= 160 * 1024, "LDS budget");
static_assert(kSmTile * kSmTile * 2 <= kSmStageBytes, "the bf16 output tile is staged in one stage");

struct SmallGemmParams {
  const uint8_t* a;        // [M, K] e4m3
  const uint8_t* b;        // [N, K] e4m3
  void* c;                 // [M, N] bf16 or fp32
  const float* a_scale;    // optional per-tensor scales (MX: packed words [K/128][m64])
  const float* b_scale;    //                            (MX: packed words [K/128][N])
  int32_t m, n, k, m64;
  uint32_t a_bytes, b_bytes;  // buffer bounds (min(rows * K, 2^32 - 1))
  int32_t m_tiles, n_tiles;   // 128-row / 128-column tiles
  int32_t nbn;                // tile blocks per block row: ceil(n_tiles / 8)
};

// vmcnt wait leaving the newest n_newer stages (L loads each) of this wave in
// flight, then a barrier: every wave's loads of the older stages are in LDS.
template <int L>
__device__ __forceinline__ void small_wait_stage(int n_newer) {
  if (n_newer >= 3) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(3 * L) : "memory");
  else if (n_newer == 2) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(2 * L) : "memory");
  else if (n_newer == 1) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(L) : "memory");
  else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
}
static_assert(kSmAhead <= 4, "small_wait_stage covers at most 3 newer stages");

// MX: e8m0 exponents applied by the scaled 16x16x128 MFMA (read_operand's K
// order); a K step's words of the tile (64 per 64-row group of A and of B)
// ride in the stage, one 4-byte-per-lane DMA per wave.
template <bool F32OUT, bool M32, bool MX = false>
__global__ __launch_bounds__(kSmThreads, 2) void gemm_fp8_small(SmallGemmParams p) {
  static_assert(!(M32 && MX), "MX runs on the 16x16x128 MFMA");
  constexpr int kStg = sm_stage_bytes(MX);
  constexpr int kLoads = MX ? 5 : 4;  // vector-memory instructions per wave and step
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int l16 = lane & 15, lg = lane >> 4;
  const int wm = wave >> 2, wn = wave & 3;  // the wave's 64 rows and 32 columns
  const int fx = swz(l16);

  // Tile of this workgroup.  Workgroups are dispatched round-robin over the 8
  // XCDs (blockIdx % 8), so each XCD gets a contiguous run of virtual ids, and
  // a run of 32 ids is a block of 4 (M) x 8 (N) tiles sharing A rows and B
  // columns in that XCD's L2.  The grid is a whole number of blocks; ids past
  // the tile grid exit.
  const int g = gridDim.x;
  const int vid = (g & 7) == 0 ? (blockIdx.x & 7) * (g >> 3) + (blockIdx.x >> 3) : blockIdx.x;
  const int blk = vid >> 5, sl = vid & 31;
  const int mt = (blk / p.nbn) * 4 + (sl & 3), nt = (blk % p.nbn) * 8 + (sl >> 2);
  if (mt >= p.m_tiles || nt >= p.n_tiles) return;
  const int m0 = mt * kSmTile, n0 = nt * kSmTile;
  const int k_steps = p.k / kBK;

  // DMA: instruction i of wave w fills LDS rows 64i + 8w + lane/8 of an operand
  // tile; the lane fetches logical chunk (lane & 7) ^ swz(row), which lands
  // swizzled.  A rows past M repeat row M-1 (never stored).
  const int ld_row = 8 * wave + (lane >> 3);
  const int ld_chunk = (lane & 7) ^ swz(ld_row);
  const i32x4 a_srd = make_srd(p.a, p.a_bytes);
  const i32x4 b_srd = make_srd(p.b, p.b_bytes);
  int a_voff[2], b_voff[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int ra = min(m0 + 64 * i + ld_row, p.m - 1);
    a_voff[i] = buf_off(ra, p.k, ld_chunk * 16);
    b_voff[i] = buf_off(n0 + 64 * i + ld_row, p.k, ld_chunk * 16);
  }
  // MX: waves 0, 1 fetch the words of A's two 64-row groups (a group past the
  // padded rows repeats the last one: its rows are never stored), 2, 3 B's; 4-7
  // repeat them, so that every wave has the same number of loads in flight
  const int ww = wave & 3;
  const i32x4 w_srd = make_srd(ww < 2 ? p.a_scale : p.b_scale, 0xffffffffu);
  const int w_voff = ((ww < 2 ? min(m0 + 64 * ww, p.m64 - 64) : n0 + 64 * (ww - 2)) + lane) * 4;
  const int w_step = (ww < 2 ? p.m64 : p.n) * 4;
  auto issue = [&](int kt) __attribute__((always_inline)) {
    uint8_t* st = smem + (kt % kSmStages) * kStg;
    if constexpr (MX) load_lds_4B(w_srd, st + kSmStageBytes + ww * 256, w_voff, buf_off(kt, w_step, 0));
#pragma unroll
    for (int i = 0; i < 2; ++i) load_lds_16B(a_srd, st + (64 * i + 8 * wave) * kBK, a_voff[i], kt * kBK);
#pragma unroll
    for (int i = 0; i < 2; ++i)
      load_lds_16B(b_srd, st + kSmOperandBytes + (64 * i + 8 * wave) * kBK, b_voff[i], kt * kBK);
  };
  // The wave's fragments of step kt.  16x16x128: A sub-tiles (rows 64wm + 16i
  // + l16) and B fragments (columns 32wn + 16j + l16), K bytes 32lg .. +31.
  // M32: fragment 2b + h is 32-row block b (rows 64wm + 32b + l32 of A, 32wn +
  // l32 of B) and K half h: bytes 64h + 32g .. +31 (g = lane / 32), i.e.
  // the 32-byte chunk pair 2h + g of the row; the rows of a block start at a
  // multiple of 32, so the swizzle of row l32 is the lane constant f32.
  const int l32 = lane & 31, g32 = lane >> 5;
  const int f32 = swz(l32);
  struct Words {
    int a, b;
  };
  auto read = [&](int kt, i32x8 (&af)[4], i32x8 (&bf)[2], Words& w) __attribute__((always_inline)) {
    const uint8_t* st = smem + (kt % kSmStages) * kStg;
    if constexpr (MX) {
      const int32_t* words = reinterpret_cast<const int32_t*>(st + kSmStageBytes);
      w.a = words[wm * 64 + lane];
      w.b = words[kSmTile + (wn >> 1) * 64 + lane] >> (16 * (wn & 1));
    }
    if constexpr (M32) {
#pragma unroll
      for (int f = 0; f < 4; ++f) af[f] = read_frag(st, 64 * wm + 32 * (f >> 1) + l32, 2 * (f & 1) + g32, f32);
#pragma unroll
      for (int f = 0; f < 2; ++f) bf[f] = read_frag(st + kSmOperandBytes, 32 * wn + l32, 2 * f + g32, f32);
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) af[i] = read_operand<MX>(st, 64 * wm + 16 * i + l16, lg, fx);
#pragma unroll
      for (int j = 0; j < 2; ++j) bf[j] = read_operand<MX>(st + kSmOperandBytes, 32 * wn + 16 * j + l16, lg, fx);
    }
  };

  // accumulators: 16x16x128: acc[i][j] (4 values); M32: acc32[bi] (16 values)
  f32x4 acc[4][2];
  f32x16 acc32[2];
  if constexpr (M32) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc32[i][r] = 0.f;
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  auto mma = [&](const i32x8 (&af)[4], const i32x8 (&bf)[2], const Words& w) __attribute__((always_inline)) {
    if constexpr (MX) {
      auto sub = [&](auto u) __attribute__((always_inline)) {
        constexpr int U = decltype(u)::value;
        acc[U][0] = mfma_mx<0, U>(bf[0], af[U], acc[U][0], w.b, w.a);
        acc[U][1] = mfma_mx<1, U>(bf[1], af[U], acc[U][1], w.b, w.a);
      };
      sub(std::integral_constant<int, 0>{});
      sub(std::integral_constant<int, 1>{});
      sub(std::integral_constant<int, 2>{});
      sub(std::integral_constant<int, 3>{});
    } else if constexpr (M32) {
      // both K halves of the two blocks
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int i = 0; i < 2; ++i) acc32[i] = mfma_e4m3_32x32x64(bf[h], af[2 * i + h], acc32[i]);
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = mfma_e4m3_16x16x128(bf[j], af[i], acc[i][j]);
    }
  };

  // Prologue: steps 0 .. kSmAhead-1 in flight, step 0's fragments in registers.
  const int pre = min(kSmAhead, k_steps);
  for (int kt = 0; kt < pre; ++kt) issue(kt);
  small_wait_stage<kLoads>(pre - 1);
  i32x8 af0[4], bf0[2], af1[4], bf1[2];
  Words w0{}, w1{};
  read(0, af0, bf0, w0);

  // Step kt: DMA of step kt+kSmAhead into the slot of step kt-1 (read in
  // iteration kt-2, complete at iteration kt-1's barrier); wait for step kt+1;
  // read its fragments into the other register set while the MFMAs of step kt
  // run.
  auto step = [&](int kt, i32x8 (&ca)[4], i32x8 (&cb)[2], Words& cw, i32x8 (&na)[4], i32x8 (&nb)[2], Words& nw)
      __attribute__((always_inline)) {
    if (kt + kSmAhead < k_steps) issue(kt + kSmAhead);
    if (kt + 1 < k_steps) {
      small_wait_stage<kLoads>(min(kSmAhead - 1, k_steps - 1 - (kt + 1)));
      read(kt + 1, na, nb, nw);
    }
    // the reads stay ahead of the MFMAs (left behind them, the next step's
    // barrier, which waits for them, would expose their whole latency)
    __builtin_amdgcn_sched_barrier(0);
    mma(ca, cb, cw);
    __builtin_amdgcn_sched_barrier(0);
  };
  // Steady state, straight-line: every step issues a load and leaves kSmAhead-1
  // newer steps in flight.  (Written with the tail's conditions, the two
  // register sets got merged into one, which put each step's reads right
  // before its own MFMAs.)
  auto step_full = [&](int kt, i32x8 (&ca)[4], i32x8 (&cb)[2], Words& cw, i32x8 (&na)[4], i32x8 (&nb)[2], Words& nw)
      __attribute__((always_inline)) {
    issue(kt + kSmAhead);
    small_wait_stage<kLoads>(kSmAhead - 1);
    read(kt + 1, na, nb, nw);
    __builtin_amdgcn_sched_barrier(0);
    mma(ca, cb, cw);
    __builtin_amdgcn_sched_barrier(0);
  };
  int kt = 0;
  for (; kt + 1 + kSmAhead < k_steps; kt += 2) {
    step_full(kt, af0, bf0, w0, af1, bf1, w1);
    step_full(kt + 1, af1, bf1, w1, af0, bf0, w0);
  }
  for (; kt + 1 < k_steps; kt += 2) {
    step(kt, af0, bf0, w0, af1, bf1, w1);
    step(kt + 1, af1, bf1, w1, af0, bf0, w0);
  }
  if (kt < k_steps) step(kt, af0, bf0, w0, af1, bf1, w1);

  // ---- epilogue: lane holds row 64wm + 16i + l16, columns 32wn + 16j + 4lg .. +3
  // (M32: row 64wm + 32bi + l32, columns 32wn + 8q + 4g32 .. +3 in registers
  // 4q .. 4q+3 of acc32[bi])
  const float tens = MX ? 1.0f : (p.a_scale ? p.a_scale[0] : 1.0f) * (p.b_scale ? p.b_scale[0] : 1.0f);
  constexpr int kRowSteps = M32 ? 2 : 4, kColSteps = M32 ? 4 : 2;
  const int er = M32 ? l32 : l16;                     // row within a row step
  auto value = [&](int i, int j) __attribute__((always_inline)) -> f32x4 {  // row step i, 4 columns j
    if constexpr (M32)
      return f32x4{acc32[i][4 * j], acc32[i][4 * j + 1], acc32[i][4 * j + 2], acc32[i][4 * j + 3]};
    else
      return acc[i][j];
  };
  if constexpr (F32OUT) {
#pragma unroll
    for (int i = 0; i < kRowSteps; ++i) {
      const int r = m0 + 64 * wm + (64 / kRowSteps) * i + er;
      if (r < p.m) {
        float* dst = static_cast<float*>(p.c) + static_cast<int64_t>(r) * p.n + n0 + 32 * wn + 4 * (M32 ? g32 : lg);
#pragma unroll
        for (int j = 0; j < kColSteps; ++j) {
          const f32x4 v = value(i, j);
          *reinterpret_cast<float4*>(dst + (32 / kColSteps) * j) =
              float4{v.x * tens, v.y * tens, v.z * tens, v.w * tens};
        }
      }
    }
  } else {
    // staged in LDS (rows of 256 bytes = 16 chunks, chunk c of row r at slot
    // c ^ (r & 15)) and stored as 16-byte chunks covering whole rows
    __syncthreads();  // every wave is done with the ring
#pragma unroll
    for (int i = 0; i < kRowSteps; ++i) {
      const int r = 64 * wm + (64 / kRowSteps) * i + er;
#pragma unroll
      for (int j = 0; j < kColSteps; ++j) {
        const int c = 4 * wn + (M32 ? j : 2 * j + (lg >> 1)), half = M32 ? g32 : (lg & 1);
        const f32x4 a = value(i, j);
        uint2 v;
        v.x = pack_bf16x2(a.x * tens, a.y * tens);
        v.y = pack_bf16x2(a.z * tens, a.w * tens);
        *reinterpret_cast<uint2*>(smem + r * 256 + ((c ^ (r & 15)) << 4) + half * 8) = v;
      }
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kSmTile * 16 / kSmThreads; ++u) {
      const int idx = tid + kSmThreads * u, r = idx >> 4, c = idx & 15;
      if (m0 + r < p.m) {
        const uint4 v = *reinterpret_cast<const uint4*>(smem + r * 256 + ((c ^ (r & 15)) << 4));
        *reinterpret_cast<uint4*>(static_cast<uint16_t*>(p.c) + static_cast<int64_t>(m0 + r) * p.n + n0 + c * 8) = v;
      }
    }
  }
}

}  // namespace hkmoe
