// Dense FP8 GEMM for few rows of A (or few output tiles): C[M,N] = A[M,K] .
// B[N,K]^T, per-tensor scales or MX exponents, bf16 or fp32 C.
//
// With a few dozen rows the product is one pass over B, and what bounds it is
// how many CUs pull on HBM and how much each can have in flight: 128x128 (or
// 256x256) tiles leave most CUs idle and walk K serially (17x8192x2048: 64
// workgroups of 16 steps, 11.9 us for 16.8 MB).  Here a workgroup owns a strip
// of 16 NF columns and up to 16 MF rows, and its NW waves split K: wave w takes
// the 128-wide K steps w, w + NW, ..., so the workgroup reads runs of NW whole
// lines of each row at a time.  Every wave streams its own steps through its
// own LDS ring (buffer->LDS DMA, D steps deep, whole 128-byte lines), so there
// is no barrier in the K loop; the partial tiles meet in LDS once, at the end,
// and are summed in wave order (deterministic).
//
// The operands go through LDS although no wave shares them: a load straight
// into the MFMA's operand order touches 16 rows of 64 bytes, and a CU then gets
// 30-40 GB/s whether the lines come from L2 or HBM, less than half of what the
// same loads give on whole lines.
#pragma once

#include "gemm_fp8.hpp"

namespace hkmoe {

struct SkinnyParams {
  const uint8_t* a;  // [M, K] e4m3
  const uint8_t* b;  // [N, K] e4m3
  void* c;           // [M, N] bf16 or fp32
  const float* a_scale;  // optional per-tensor scales (MX: packed words [K/128][m64])
  const float* b_scale;  //                            (MX: packed words [K/128][N])
  int32_t m, n, k, m64;
  int32_t strips;    // N / (16 NF)
  int32_t m_blocks;  // ceil(M / (16 MF))
};

constexpr int kSkMaxLds = 160 * 1024;
constexpr int sk_step_bytes(int mf, int nf, bool mx) { return (mf + nf) * 2048 + (mx ? 512 : 0); }
// ring depth: the steps that fit (one workgroup per CU), 2 to 5 for the strips in use
constexpr int sk_depth(int mf, int nf, int nw, bool mx) { return kSkMaxLds / (sk_step_bytes(mf, nf, mx) * nw); }
constexpr int sk_ring_bytes(int mf, int nf, int nw, bool mx) {
  return sk_depth(mf, nf, nw, mx) * nw * sk_step_bytes(mf, nf, mx);
}
constexpr int sk_part_bytes(int mf, int nf, int nw) { return nw * 16 * mf * (16 * nf + 4) * 4; }
constexpr int sk_lds_bytes(int mf, int nf, int nw, bool mx) {
  return sk_ring_bytes(mf, nf, nw, mx) > sk_part_bytes(mf, nf, nw) ? sk_ring_bytes(mf, nf, nw, mx)
                                                                   : sk_part_bytes(mf, nf, nw);
}

// One operand fragment from a 16-row ring tile (chunks at a_lo / a_hi +
// OFF), complete on return: the compiler would wait for every DMA in flight
// before an LDS read that it can see.
template <int OFF>
__device__ __forceinline__ void sk_frag(uint32_t a_lo, uint32_t a_hi, i32x8& f) {
  i32x4 lo, hi;
  asm volatile("ds_read_b128 %0, %2 offset:%4\n\tds_read_b128 %1, %3 offset:%4\n\ts_waitcnt lgkmcnt(0)"
               : "=&v"(lo), "=&v"(hi)
               : "v"(a_lo), "v"(a_hi), "i"(OFF));
  f.lo = lo;
  f.hi = hi;
}
// Two fragments, one wait.
template <int OFF>
__device__ __forceinline__ void sk_frag2(uint32_t a_lo, uint32_t a_hi, i32x8& f, i32x8& g) {
  i32x4 lo, hi, lo2, hi2;
  asm volatile(
      "ds_read_b128 %0, %4 offset:%6\n\tds_read_b128 %1, %5 offset:%6\n\t"
      "ds_read_b128 %2, %4 offset:%7\n\tds_read_b128 %3, %5 offset:%7\n\ts_waitcnt lgkmcnt(0)"
      : "=&v"(lo), "=&v"(hi), "=&v"(lo2), "=&v"(hi2)
      : "v"(a_lo), "v"(a_hi), "i"(OFF), "i"(OFF + 2048));
  f.lo = lo;
  f.hi = hi;
  g.lo = lo2;
  g.hi = hi2;
}
__device__ __forceinline__ void sk_words(uint32_t a, int& x, int& y) {
  asm volatile("ds_read_b32 %0, %2\n\tds_read_b32 %1, %2 offset:256\n\ts_waitcnt lgkmcnt(0)"
               : "=&v"(x), "=&v"(y)
               : "v"(a));
}

// One 16-row fragment's MFMAs against the strip's NF B fragments.  MX: A's
// exponent byte U of sa, B's bytes 0 .. NF-1 of sb.
template <int NF, bool MX, int U>
__device__ __forceinline__ void skinny_mma(f32x4 (&acc)[NF], const i32x8& a, const i32x8 (&b)[NF], int sa, int sb) {
  if constexpr (MX) {
    acc[0] = mfma_mx<0, U>(b[0], a, acc[0], sb, sa);
    if constexpr (NF > 1) acc[1] = mfma_mx<1, U>(b[1], a, acc[1], sb, sa);
    if constexpr (NF > 2) {
      acc[2] = mfma_mx<2, U>(b[2], a, acc[2], sb, sa);
      acc[3] = mfma_mx<3, U>(b[3], a, acc[3], sb, sa);
    }
  } else {
#pragma unroll
    for (int j = 0; j < NF; ++j) acc[j] = mfma_e4m3_16x16x128(b[j], a, acc[j]);
  }
}

template <int MF, int NF, int NW, bool MX, bool F32OUT>
__global__ __launch_bounds__(NW * 64, 1) void gemm_fp8_skinny(SkinnyParams p) {
  static_assert((MF == 1 || MF == 2 || MF == 4) && (NF == 1 || NF == 2 || NF == 4), "tile");
  constexpr int kRows = 16 * MF, kCols = 16 * NF;
  constexpr int kStep = sk_step_bytes(MF, NF, MX);
  constexpr int D = sk_depth(MF, NF, NW, MX);
  constexpr int kLoads = 2 * (MF + NF) + (MX ? 2 : 0);  // DMA instructions per step
  static_assert(D >= 2 && kLoads * (D - 1) <= 63, "ring depth, vmcnt range");
  constexpr int kLd = kCols + 4;  // padded partial-tile row (floats)
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63, l16 = lane & 15, lg = lane >> 4;
  // The M blocks of a strip run side by side on one XCD (workgroups go
  // round-robin over the 8), so B comes from HBM once: eight strips at a time,
  // M blocks next, and the remaining strips (fewer than 8) one M block after
  // the other.
  const int whole = p.strips & ~7, g = blockIdx.x;
  int mb, strip;
  if (g < whole * p.m_blocks) {
    const int q = g >> 3;
    mb = q % p.m_blocks;
    strip = (q / p.m_blocks) * 8 + (g & 7);
  } else {
    const int r = g - whole * p.m_blocks;
    mb = r / (p.strips - whole);
    strip = whole + r % (p.strips - whole);
  }
  const int n0 = strip * kCols, m0 = mb * kRows;
  const int k_steps = p.k / kBK;
  const int mine = (k_steps - wave + NW - 1) / NW;  // this wave's steps (0: none)

  const i32x4 a_srd = make_srd(p.a, static_cast<uint32_t>(p.m) * static_cast<uint32_t>(p.k));
  const i32x4 b_srd = make_srd(p.b, static_cast<uint32_t>(p.n) * static_cast<uint32_t>(p.k));
  // DMA instruction i of an operand fills its ring rows 8i .. 8i+7; the lane
  // fetches the chunk that lands swizzled (chunk c of row r at c ^ swz(r)).
  // Rows of A past M repeat row M - 1 (never stored).
  const int ld_row = lane >> 3;
  int a_off[2 * MF], b_off[2 * NF];
#pragma unroll
  for (int i = 0; i < 2 * MF; ++i)
    a_off[i] = buf_off(min(m0 + 8 * i + ld_row, p.m - 1), p.k, ((lane & 7) ^ swz(8 * i + ld_row)) * 16);
#pragma unroll
  for (int j = 0; j < 2 * NF; ++j)
    b_off[j] = buf_off(n0 + 8 * j + ld_row, p.k, ((lane & 7) ^ swz(8 * j + ld_row)) * 16);
  // MX words: word (kt, 64*(row/64) + lane) holds in byte g the exponent of row
  // 64*(row/64) + 16g + l16 for K block lg
  const i32x4 sa_srd = make_srd(p.a_scale, 0xffffffffu), sb_srd = make_srd(p.b_scale, 0xffffffffu);
  const int sa_off = MX ? ((m0 & ~63) + lane) * 4 : 0, sb_off = MX ? ((n0 & ~63) + lane) * 4 : 0;
  const int sa_sh = 8 * ((m0 & 63) >> 4), sb_sh = 8 * ((n0 & 63) >> 4);
  const float tens = MX ? 1.0f : (p.a_scale ? p.a_scale[0] : 1.0f) * (p.b_scale ? p.b_scale[0] : 1.0f);

  f32x4 acc[MF][NF];
#pragma unroll
  for (int i = 0; i < MF; ++i)
#pragma unroll
    for (int j = 0; j < NF; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  uint8_t* ring = smem + wave * D * kStep;
  // Step i of this wave into its slot.  Steps past the last one go through
  // empty descriptors (no memory traffic), so the loads in flight stay a
  // constant count.
  auto issue = [&](int i, int slot) __attribute__((always_inline)) {
    const bool in = i < mine;
    const int kt = wave + NW * i;
    const int ko = in ? kt * kBK : 0;
    uint8_t* st = ring + slot * kStep;
    i32x4 as = a_srd, bs = b_srd;
    as.z = in ? as.z : 0;
    bs.z = in ? bs.z : 0;
#pragma unroll
    for (int j = 0; j < 2 * NF; ++j) load_lds_16B(bs, st + (2 * MF + j) * 1024, b_off[j], ko);
#pragma unroll
    for (int u = 0; u < 2 * MF; ++u) load_lds_16B(as, st + u * 1024, a_off[u], ko);
    if constexpr (MX) {
      i32x4 ss = sa_srd, sw = sb_srd;
      ss.z = in ? ss.z : 0;
      sw.z = in ? sw.z : 0;
      load_lds_4B(ss, st + (MF + NF) * 2048, sa_off, in ? buf_off(kt, p.m64 * 4, 0) : 0);
      load_lds_4B(sw, st + (MF + NF) * 2048 + 256, sb_off, in ? buf_off(kt, p.n * 4, 0) : 0);
    }
  };
  const int x = swz(l16);
  const uint32_t ring_a = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(ring));
  const uint32_t lo_off = l16 * kBK + ((lg ^ x) << 4), hi_off = l16 * kBK + (((lg + 4) ^ x) << 4);
  // The scaled MFMA's K order (chunks lg and lg + 4 of a row); any order common
  // to both operands serves the unscaled one.
  auto step = [&](int i, int slot) __attribute__((always_inline)) {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kLoads * (D - 1)) : "memory");
    const uint32_t lo = ring_a + slot * kStep + lo_off, hi = ring_a + slot * kStep + hi_off;
    i32x8 a[MF], b[NF];
    int sa = 0, sb = 0;
    if constexpr (MF == 1) {
      sk_frag<0>(lo, hi, a[0]);
    } else {
      sk_frag2<0>(lo, hi, a[0], a[1]);
      if constexpr (MF == 4) sk_frag2<4096>(lo, hi, a[2], a[3]);
    }
    if constexpr (NF == 1) {
      sk_frag<MF * 2048>(lo, hi, b[0]);
    } else {
      sk_frag2<MF * 2048>(lo, hi, b[0], b[1]);
      if constexpr (NF == 4) sk_frag2<(MF + 2) * 2048>(lo, hi, b[2], b[3]);
    }
    if constexpr (MX) {
      sk_words(ring_a + slot * kStep + (MF + NF) * 2048 + lane * 4, sa, sb);
      sa >>= sa_sh;
      sb >>= sb_sh;
    }
    issue(i + D, slot);  // this wave has read the slot
    __builtin_amdgcn_sched_barrier(0);
    skinny_mma<NF, MX, 0>(acc[0], a[0], b, sa, sb);
    if constexpr (MF > 1) skinny_mma<NF, MX, 1>(acc[1], a[1], b, sa, sb);
    if constexpr (MF > 2) {
      skinny_mma<NF, MX, 2>(acc[2], a[2], b, sa, sb);
      skinny_mma<NF, MX, 3>(acc[3], a[3], b, sa, sb);
    }
  };
#pragma unroll
  for (int u = 0; u < D; ++u) issue(u, u);
  int slot = 0;
  for (int i = 0; i < mine; ++i) {
    step(i, slot);
    slot = slot == D - 1 ? 0 : slot + 1;
  }
  // every wave's DMA has landed before the partial tiles overwrite the rings
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  float* part = reinterpret_cast<float*>(smem);
  // lane holds row 16i + l16, columns 16j + 4lg .. +3 of its wave's partial tile
#pragma unroll
  for (int i = 0; i < MF; ++i)
#pragma unroll
    for (int j = 0; j < NF; ++j)
      *reinterpret_cast<f32x4*>(part + (wave * kRows + 16 * i + l16) * kLd + 16 * j + 4 * lg) = acc[i][j];
  __syncthreads();
  for (int idx = tid; idx < kRows * kCols / 4; idx += NW * 64) {
    const int r = idx / (kCols / 4), cc = (idx % (kCols / 4)) * 4;
    if (m0 + r >= p.m) continue;
    f32x4 s = *reinterpret_cast<const f32x4*>(part + r * kLd + cc);
#pragma unroll
    for (int w = 1; w < NW; ++w) s += *reinterpret_cast<const f32x4*>(part + (w * kRows + r) * kLd + cc);
    const int64_t at = static_cast<int64_t>(m0 + r) * p.n + n0 + cc;
    if constexpr (F32OUT) {
      *reinterpret_cast<float4*>(static_cast<float*>(p.c) + at) = float4{s.x * tens, s.y * tens, s.z * tens, s.w * tens};
    } else {
      *reinterpret_cast<uint2*>(static_cast<uint16_t*>(p.c) + at) =
          uint2{pack_bf16x2(s.x * tens, s.y * tens), pack_bf16x2(s.z * tens, s.w * tens)};
    }
  }
}

}  // namespace hkmoe
