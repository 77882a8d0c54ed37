// Narrow grouped GEMM for small expert segments (at most 64 rows), with
// per-tensor, block or MX scales, gfx950.
//
// A segment of <= 64 rows against a 256-row weight panel does 2*64*256*K
// FLOPs for 256*K weight bytes: it is bound by streaming the weights from HBM,
// not by the MFMA.  The 256x256 persistent kernel (gemm_fp8.hpp) keeps only
// two K steps of weights in flight per CU and needs the whole CU's LDS for
// them, so such tiles run at HBM latency.  This kernel streams the weights
// straight into VGPRs instead, P K steps ahead (P * 4 KiB per wave, 256 KiB
// per CU at P = 8), so a few dozen CUs can pull HBM bandwidth while the other
// CUs run the compute-bound 256x256 tiles of the large experts (the host
// launches the two kernels on two streams).
//
//  * work item: (narrow segment m, N tile nt of 256 rows, or a half or quarter
//    of one).  Alone on the chip workgroup b starts on item b, and the items past the
//    grid come from an atomic counter; while the list also holds 256x256
//    tiles all come from the counter and only narrow_active workgroups take items,
//    the first ones to start (a second counter), while the others exit at once and
//    leave their CUs to the 256x256 kernel.  Segment m is entry first + m of the
//    M-tile list (the narrow experts are listed last).
//  * NW waves (8, or 4 / 2 for half / quarter tiles); wave w owns 32 weight rows =
//    two 16-row fragments:
//      gate/up GEMM: gate rows 16w..16w+15 of the tile's 128 and the matching
//                    up rows (h columns 16w..16w+15);
//      plain GEMM:   rows 32w..32w+31 of the 256.
//    Each lane loads its fragment rows' 32 K bytes per step with two 16-byte
//    buffer loads per fragment, in the register order read_frag (MX: read_frag_mx)
//    produces from LDS: the MFMA operands, the accumulation (MFMA chain, or block
//    products folded in with their scales) and the epilogue are those of the
//    256x256 kernel, so both kernels give the same bits.
//  * activations: the waves DMA the segment's rows, 8 per instruction (rows past
//    the segment repeat its last one; eight past it cost no traffic), into an LDS
//    ring of P+1 stages, P steps ahead like the weights; one barrier per K step.
//    An item's activation scales (MX: its rows' own exponent bytes, one dword per
//    row and step) and block scales for all its K steps are DMA'd into one of two
//    LDS buffers once, when the item is decoded (at least P steps before its
//    first step); MX weight exponents come as one dword per lane and step.
//  * every wave issues the same number kVm of vector-memory instructions per K
//    step, so "step kt has landed" is vmcnt(kVm*(P-1)) (other loads only add to
//    the count, so the wait can only be longer); after the last item the loads
//    continue on that item's first steps (valid addresses, never read), so the
//    count never changes.
//  * a group of P unrolled steps never straddles two items: the loads of an item's
//    last group are the next item's first P steps, and where P does not divide
//    the K steps the last group's missing steps are empty (PAD).
//  * the compiler must not wait for the prefetch window by itself: LDS
//    accesses and the item decode's scalar loads are inline asm with their own
//    lgkmcnt waits (it would otherwise wait for every buffer->LDS DMA before an
//    LDS access, and for pending stores before a scalar load), and the next
//    item's gathered row indices reach LDS by a DMA issued a group before they
//    are read.
#pragma once

#include "gemm_fp8.hpp"

namespace hkmoe {

constexpr int kNarrowRows = 64;
// Geometry of one instantiation: NW waves per workgroup (each two 16-row weight
// fragments, so a workgroup covers 32 NW of a tile's 256 weight rows), segments
// of at most ROWS rows, prefetch depth P, scales SC.
template <Scale SC, int P, int NW, int ROWS>
struct NarrowGeo {
  static constexpr int kThreads = NW * 64;
  static constexpr int kSub = 8 / NW;                       // work items per 256-row tile
  static constexpr int kStage = ROWS * kBK;                 // one ring stage: A rows
  static constexpr int kADma = ROWS / 8 / NW;               // A-row DMA instructions per wave and step
  static constexpr int kVm = kADma + 4 + (SC == Scale::kMX ? 1 : 0);  // vector-memory instructions per step
  // K steps whose scales fit an item's LDS buffer (per-tensor scales: no limit)
  static constexpr int kMaxSteps = SC == Scale::kBlock && P == 8 ? 64 : 128;
  // per-item scales, two buffers (current / next item): [K step][ROWS]
  // activation scales (MX: exponent dwords), then block scales: per wave [2
  // block rows][K step] weight scales
  static constexpr int kWsOff = kMaxSteps * ROWS * 4;
  static constexpr int kScaleBuf =
      SC == Scale::kTensor ? 0 : kWsOff + (SC == Scale::kBlock ? NW * 2 * kMaxSteps * 4 : 0);
  static constexpr int kCtLd = NW * 16 + 8;                 // staged h row (bf16)
  static constexpr int kCtOff = (P + 1) * kStage;
  static constexpr int kGidxOff = kCtOff + ROWS * kCtLd * 2;  // per-wave gathered row indices
  static constexpr int kQOff = kGidxOff + NW * 256;           // published item index
  static constexpr int kScaleOff = kQOff + 256;
  static constexpr int kLds = kScaleOff + 2 * kScaleBuf;
  static_assert(kLds <= 160 * 1024, "LDS budget");
  static_assert(kADma >= 1 && kVm * (P - 1) <= 63, "vmcnt range");
};

extern "C" __device__ i32x4 hk_raw_buffer_load_v4i32(i32x4 rsrc, int voffset, int soffset,
                                                     int aux) __asm("llvm.amdgcn.raw.buffer.load.v4i32");
extern "C" __device__ int hk_raw_buffer_load_i32(i32x4 rsrc, int voffset, int soffset,
                                                 int aux) __asm("llvm.amdgcn.raw.buffer.load.i32");

// a[idx] for a wave-uniform idx through the scalar cache, complete on return.
// Only for data written before the kernel started.
__device__ __forceinline__ int sload_i32(const int32_t* a, int idx) {
  const i32x4 srd = make_srd(a, 0xffffffffu);
  const int off = __builtin_amdgcn_readfirstlane(idx * 4);
  int v;
  asm volatile("s_buffer_load_dword %0, %1, %2\n\ts_waitcnt lgkmcnt(0)" : "=&s"(v) : "s"(srd), "s"(off));
  return v;
}

template <int N>
__device__ __forceinline__ void wait_vm_barrier() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

// LDS accesses of the narrow kernel are written as inline asm with their own
// lgkmcnt waits; outputs are early-clobber ("=&"), since a load's destination
// is written after later instructions of the same block have read their
// address registers.  The compiler cannot tell the ring slots apart, so before any
// LDS access it can see it would wait for every buffer->LDS DMA still in
// flight, i.e. for the whole prefetch window.
__device__ __forceinline__ uint32_t lds_addr(const void* p) {
  return static_cast<uint32_t>(reinterpret_cast<uintptr_t>(p));
}

// One A fragment (two 16-byte chunks at a_lo / a_hi + OFF) and its row scale
// (a_sc + SOFF), complete on return.
template <int OFF, int SOFF>
__device__ __forceinline__ void lds_frag(uint32_t a_lo, uint32_t a_hi, uint32_t a_sc, i32x8& f, float& sc) {
  i32x4 lo, hi;
  asm volatile(
      "ds_read_b128 %0, %3 offset:%6\n\t"
      "ds_read_b128 %1, %4 offset:%6\n\t"
      "ds_read_b32 %2, %5 offset:%7\n\t"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(lo), "=&v"(hi), "=&v"(sc)
      : "v"(a_lo), "v"(a_hi), "v"(a_sc), "i"(OFF), "i"(SOFF));
  f.lo = lo;
  f.hi = hi;
}

// the same fragment without a scale
template <int OFF>
__device__ __forceinline__ void lds_frag(uint32_t a_lo, uint32_t a_hi, i32x8& f) {
  i32x4 lo, hi;
  asm volatile("ds_read_b128 %0, %2 offset:%4\n\tds_read_b128 %1, %3 offset:%4\n\ts_waitcnt lgkmcnt(0)"
               : "=&v"(lo), "=&v"(hi)
               : "v"(a_lo), "v"(a_hi), "i"(OFF));
  f.lo = lo;
  f.hi = hi;
}

// the dwords at a and a + OFF (an item's two weight-scale rows at one K step)
template <int OFF>
__device__ __forceinline__ float2 lds_read_w2(uint32_t a) {
  float x, y;
  asm volatile("ds_read_b32 %0, %2\n\tds_read_b32 %1, %2 offset:%3\n\ts_waitcnt lgkmcnt(0)"
               : "=&v"(x), "=&v"(y)
               : "v"(a), "i"(OFF));
  return float2{x, y};
}

__device__ __forceinline__ int lds_read_i32(uint32_t a) {
  int v;
  asm volatile("ds_read_b32 %0, %1\n\ts_waitcnt lgkmcnt(0)" : "=&v"(v) : "v"(a));
  return v;
}

__device__ __forceinline__ void lds_write_i32(uint32_t a, int v) {
  asm volatile("ds_write_b32 %0, %1" ::"v"(a), "v"(v) : "memory");
}

__device__ __forceinline__ void lds_write_b64(uint32_t a, uint2 v) {
  asm volatile("ds_write_b64 %0, %1" ::"v"(a), "v"(v) : "memory");
}

// 16 bytes at a, complete on return
__device__ __forceinline__ uint4 lds_read_u4(uint32_t a) {
  uint4 v;
  asm volatile("ds_read_b128 %0, %1\n\ts_waitcnt lgkmcnt(0)" : "=&v"(v) : "v"(a));
  return v;
}

// LDS writes done, then the workgroup barrier (no vmcnt: DMA stays in flight)
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// PAD: K steps need not be a multiple of P (the last group's missing steps are
// empty: nothing loaded, nothing computed).
template <Epi EPI, Scale SC, int P, int NW, int ROWS, bool PAD>
__global__ __launch_bounds__(NW * 64, 2) void gemm_fp8_narrow(GemmParams p) {
  using G = NarrowGeo<SC, P, NW, ROWS>;
  constexpr bool kBlockSc = SC == Scale::kBlock, kMX = SC == Scale::kMX;
  constexpr bool kSilu = EPI != Epi::kStoreBf16;
  static_assert(EPI == Epi::kStoreBf16 || EPI == (kBlockSc ? Epi::kSiluQuant : kMX ? Epi::kSiluMx : Epi::kSiluBf16),
                "narrow epilogues");
  static_assert(!(kBlockSc && kSilu) || NW == 8, "a 1x128 group's maximum spans the tile's 8 waves");
  static_assert(P == 4 || P == 8, "prefetch depth");
  constexpr int kT = G::kThreads;
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
  uint16_t* ct = reinterpret_cast<uint16_t*>(smem + G::kCtOff);
  int32_t* gidx = reinterpret_cast<int32_t*>(smem + G::kGidxOff);

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int l16 = lane & 15;
  const int lg = lane >> 4;
  const int fx = swz(l16);

  const int k_steps = p.K / kBK;
  const int groups = (k_steps + P - 1) / P;  // the last one may run past k_steps: empty steps
  const int total_mt = sload_i32(p.mtile_offsets, p.num_experts);
  const int n_narrow = sload_i32(p.narrow_cnt, 0);
  const int first = total_mt - n_narrow;
  const int per_seg = p.n_tiles * G::kSub;
  const int n_items = n_narrow * per_seg;
  // beside 256x256 tiles only narrow_active workgroups take items (the others
  // exit and leave their CUs to the 256x256 kernel); alone, all of them do
  if (n_items <= 0) return;
  int32_t* const item_ctr = p.tile_ctr;  // zeroed item counter; p.tile_ctr[2]: active slots
  int* s_q = reinterpret_cast<int*>(smem + G::kQOff);  // published item index

  // this wave's two fragment rows: tile-local in the item's part of the tile
  // (row R; fragment R/16 of the packed block) and relative to the item's
  // first weight row
  int frag_r[2], frag_w[2];
  if constexpr (kSilu) {
    frag_r[0] = 64 * (wave >> 1) + 16 * (wave & 1) + l16;  // gate row 16w + l16 of the part
    frag_r[1] = frag_r[0] + 32;                             // its up row
    frag_w[0] = 16 * wave + l16;
    frag_w[1] = 16 * wave + l16 + p.n_out;                  // up half starts at I
  } else {
    frag_r[0] = 32 * wave + l16;
    frag_r[1] = 32 * wave + 16 + l16;
    frag_w[0] = frag_r[0];
    frag_w[1] = frag_r[1];
  }
  int ld_row[G::kADma];                                     // A rows this lane DMAs
#pragma unroll
  for (int i = 0; i < G::kADma; ++i) ld_row[i] = 8 * (wave + NW * i) + (lane >> 3);
  const i32x4 a_srd = make_srd(p.a, p.a_bytes);
  const i32x4 as_srd = make_srd(p.a_scale, 0xffffffffu);
  const i32x4 g_srd = make_srd(p.a_gather, 0xffffffffu);
  const int64_t kb_per_expert = static_cast<int64_t>(p.nb / kGroup) * k_steps;
  const float tens_a = SC == Scale::kTensor ? __int_as_float(sload_i32(reinterpret_cast<const int32_t*>(p.a_scale), 0)) : 1.0f;

  // K bytes of a lane's two 16-byte register halves: chunks 2lg, 2lg + 1 of the
  // 128, or in the scaled MFMA's order lg, lg + 4
  const int c_lo = kMX ? lg : 2 * lg, c_hi = kMX ? lg + 4 : 2 * lg + 1;
  // Lane-constant weight offsets within a K step: packed layout, the
  // contiguous 1 KiB register halves of the fragment (chunk c of row r in half
  // c & 1, lane slot 16 (c >> 1) + r; whole 128-byte lines); row-major, the
  // weight row (relative to the item's first row, which goes into the descriptor).
  int wvoff[4];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    if (p.b_packed) {
      const int f = frag_r[j] >> 4;
      wvoff[2 * j] = (2 * f + (c_lo & 1)) * 1024 + (16 * (c_lo >> 1) + l16) * 16;
      wvoff[2 * j + 1] = (2 * f + (c_hi & 1)) * 1024 + (16 * (c_hi >> 1) + l16) * 16;
    } else {
      wvoff[2 * j] = buf_off(frag_w[j], p.K, c_lo * 16);
      wvoff[2 * j + 1] = buf_off(frag_w[j], p.K, c_hi * 16);
    }
  }
  // lane-constant LDS offsets within a ring stage: A fragment chunks of row
  // l16 (fragment i adds 2 KiB), its row scale (fragment i adds 64 bytes), and
  // this wave's two weight scales
  const uint32_t smem_base = lds_addr(smem);
  const uint32_t lo_off = l16 * kBK + ((c_lo ^ fx) << 4);
  const uint32_t hi_off = l16 * kBK + ((c_hi ^ fx) << 4);
  const uint32_t scale_base = smem_base + G::kScaleOff;
  const uint32_t sa_lane = l16 * 4;                              // + buffer + kt*ROWS*4 + 64*i
  const uint32_t sb_wave = G::kWsOff + wave * 2 * G::kMaxSteps * 4;  // + buffer + h*4*kMaxSteps + kt*4
  const uint32_t gidx_wave = lds_addr(gidx) + 256 * wave;
  const uint32_t q_addr = lds_addr(s_q);
  const int kstride = p.b_packed ? (p.nb / kBN) * kTileBytes : kBK;

  // per-item state of the load side: uniform descriptors (weights; block scales
  // or MX words of the weights), and the lane's A-row and A-scale offsets
  struct Load {
    i32x4 wsrd, ssrd;
    int a_voff[G::kADma], as_voff, valid;
  };
  // per-item state of the compute side; col0: first output column (of the h
  // columns for the SiLU epilogues); mnat: M tile in expert order (MX); buf:
  // which scale buffer holds its scales
  struct Item {
    int row0, valid, nt, col0, mnat, mf, buf;
    float tens;
  };
  auto uniform4 = [](const i32x4& v) __attribute__((always_inline)) {
    i32x4 r;
    r.x = __builtin_amdgcn_readfirstlane(v.x);
    r.y = __builtin_amdgcn_readfirstlane(v.y);
    r.z = __builtin_amdgcn_readfirstlane(v.z);
    r.w = __builtin_amdgcn_readfirstlane(v.w);
    return r;
  };

  // uniform part of item `it` (scalar loads); with a row gather, the DMA of
  // the segment's gathered row indices into this wave's LDS slot
  auto decode_head = [&](int it, Load& L, Item& C) {
    const int m = it / per_seg;
    const int r = it - m * per_seg;
    const int nt = r / G::kSub, sub = r - nt * G::kSub;
    const int entry = first + m;
    const int e = sload_i32(p.mtile_list, 2 * entry);
    const int row0 = sload_i32(p.mtile_list, 2 * entry + 1);
    const int valid = min(ROWS, sload_i32(p.offsets, e + 1) - row0);
    C.row0 = row0;
    C.valid = valid;
    C.nt = nt;
    C.col0 = kSilu ? nt * 128 + sub * NW * 16 : nt * kBN + sub * NW * 32;
    C.mf = (valid + 15) >> 4;
    C.mnat = kMX ? sload_i32(p.mtile_offsets, e) : 0;
    C.tens = SC == Scale::kTensor ? tens_a * __int_as_float(sload_i32(reinterpret_cast<const int32_t*>(p.b_scale), e)) : 1.0f;
    if (p.b_packed) {
      const int64_t skip = static_cast<int64_t>(nt) * kTileBytes + sub * (NW * 4096);
      L.wsrd = make_srd(p.b + static_cast<int64_t>(e) * p.nb * p.K + skip,
                        static_cast<uint32_t>(static_cast<int64_t>(p.nb) * p.K - skip));
    } else {
      L.wsrd = make_srd(p.b + (static_cast<int64_t>(e) * p.nb + C.col0) * p.K,
                        static_cast<uint32_t>(p.nb - C.col0) * p.K);
    }
    if constexpr (kBlockSc) {
      const int nb0 = kSilu ? nt : 2 * nt + ((sub * NW + wave) >> 2);
      L.ssrd = make_srd(p.b_scale + e * kb_per_expert + static_cast<int64_t>(nb0) * k_steps,
                        static_cast<uint32_t>((kb_per_expert - static_cast<int64_t>(nb0) * k_steps) * 4));
    } else if constexpr (kMX) {
      // words of this wave's 64-row group of B tile (e, nt): 1 KiB per K step
      L.ssrd = make_srd(p.b_scale + ((static_cast<int64_t>(e) * (p.nb / kBN) + nt) * k_steps) * 256 +
                            64 * ((sub * NW + wave) >> 1),
                        static_cast<uint32_t>(k_steps) * 1024u - 256u * ((sub * NW + wave) >> 1));
    } else {
      L.ssrd = L.wsrd;  // unused
    }
    if (p.a_gather) load_lds_4B(g_srd, gidx + 64 * wave, (row0 + min(lane, valid - 1)) * 4, 0);
  };
  // lane offsets of item C, once its gathered row indices are in LDS
  auto decode_tail = [&](Load& L, const Item& C) {
    L.valid = C.valid;
    const int rs = min(lane % ROWS, C.valid - 1);
    int ts = C.row0 + rs;
    if (p.a_gather && SC != Scale::kTensor) ts = lds_read_i32(gidx_wave + 4 * rs) / p.gather_div;
#pragma unroll
    for (int i = 0; i < G::kADma; ++i) {
      const int ra = min(ld_row[i], C.valid - 1);
      const int ta = p.a_gather ? lds_read_i32(gidx_wave + 4 * ra) / p.gather_div : C.row0 + ra;
      L.a_voff[i] = buf_off(ta, p.K, ((lane & 7) ^ swz(ld_row[i])) * 16);
    }
    // MX, second GEMM: GEMM 1 left the segment's exponents in its M tile's words
    if (kMX && !kSilu) ts = C.mnat * kBM + rs;
    L.as_voff = SC != Scale::kTensor ? static_cast<int>(ts * p.as_rs) * 4 : 0;
  };

  // all K steps' activation scales of item C into its buffer (64 / ROWS steps
  // per instruction, dealt out to the waves), and block scales of its weights
  // (lane l: K block l of the first, gate, and of the second, up block row)
  auto stage_scales = [&](const Load& L, const Item& C) {
    if constexpr (SC == Scale::kTensor) return;
    constexpr int kPer = 64 / ROWS;
    uint8_t* sb = smem + G::kScaleOff + C.buf * G::kScaleBuf;
    for (int kt = wave * kPer; kt < k_steps; kt += NW * kPer) {
      const int my = min(kt + lane / ROWS, k_steps - 1) - kt;
      load_lds_4B(as_srd, sb + kt * (ROWS * 4), L.as_voff + my * static_cast<int>(p.as_ks) * 4,
                  static_cast<int>(kt * p.as_ks) * 4);
    }
    if constexpr (kBlockSc) {
      const i32x4 ssrd = uniform4(L.ssrd);
      uint8_t* wsb = sb + G::kWsOff + wave * 2 * G::kMaxSteps * 4;
#pragma unroll
      for (int k0 = 0; k0 < G::kMaxSteps; k0 += 64) {
        if (k0 >= k_steps) break;
        const int v0 = min(k0 + lane, k_steps - 1) * 4;
        load_lds_4B(ssrd, wsb + k0 * 4, v0, 0);
        load_lds_4B(ssrd, wsb + (G::kMaxSteps + k0) * 4, v0 + (kSilu ? (p.n_out / kGroup) * k_steps * 4 : 0), 0);
      }
    }
  };

  // the loads of K step kt into ring slot `slot` and weight registers wr (MX:
  // and its exponent words ws).  Steps past the last one go through empty
  // descriptors: no memory traffic, and the count of loads in flight holds.
  auto issue = [&](const Load& L, int kt, int slot, i32x8 (&wr)[2], int& ws) {
    // descriptors and K offsets are wave-uniform: keep them in SGPRs (a
    // descriptor in VGPRs would turn every load into a waterfall loop)
    i32x4 srd = uniform4(L.wsrd), asrd = a_srd;
    const int ktu = __builtin_amdgcn_readfirstlane(kt);
    const bool in = !PAD || ktu < k_steps;
    srd.z = in ? srd.z : 0;
    asrd.z = in ? asrd.z : 0;
    const int ko = in ? ktu : 0;
    uint8_t* st = smem + __builtin_amdgcn_readfirstlane(slot) * G::kStage;
#pragma unroll
    for (int i = 0; i < G::kADma; ++i) {
      // eight rows past the segment's end: no traffic either (zeros, never stored)
      i32x4 rows = asrd;
      rows.z = 8 * (wave + NW * i) < L.valid ? rows.z : 0;
      load_lds_16B(rows, st + 8 * (wave + NW * i) * kBK, L.a_voff[i], ko * kBK);
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      // weights are read once: non-temporal loads keep them from displacing
      // the 256x256 kernel's operand panels in the XCD's L2
      wr[j].lo = hk_raw_buffer_load_v4i32(srd, wvoff[2 * j], ko * kstride, kAuxNT);
      wr[j].hi = hk_raw_buffer_load_v4i32(srd, wvoff[2 * j + 1], ko * kstride, kAuxNT);
    }
    if constexpr (kMX) {
      i32x4 ssrd = uniform4(L.ssrd);
      ssrd.z = in ? ssrd.z : 0;
      ws = hk_raw_buffer_load_i32(ssrd, lane * 4, ko * 1024, 0);
    }
  };

  // ---- first item --------------------------------------------------------
  // Alone on the chip, workgroup b starts on item b and takes the items past
  // the grid from one atomic counter (none where the grid covers them all: a
  // same-address atomic costs 10 ns, and 1024 workgroups fetching two indices
  // each had spent 20 us).  Beside 256x256 tiles all items come from the counter
  // and only narrow_active workgroups take any: the first ones to start (an atomic
  // slot counter), wherever the hardware placed them; later ones exit and leave
  // their CUs to the 256x256 kernel.  Thread 0 fetches the index after next as
  // soon as it publishes one; its result is first needed an item later.
  const bool limited = first > 0 && p.narrow_active > 0;
  const int dealt = limited ? 0 : static_cast<int>(gridDim.x);  // items given out by position
  auto fetch = [&]() -> int { return dealt >= n_items ? n_items : dealt + atomicAdd(item_ctr, 1); };
  int nxt = 0;
  if (tid == 0) {
    int it0 = n_items;  // "no item": exit
    if (!limited) {
      it0 = blockIdx.x;
      nxt = fetch();
    } else if (atomicAdd(item_ctr + 2, 1) < p.narrow_active) {
      it0 = fetch();
      nxt = fetch();
    }
    lds_write_i32(q_addr, it0);
  }
  lds_barrier();
  const int it_first = __builtin_amdgcn_readfirstlane(lds_read_i32(q_addr));
  lds_barrier();  // every wave has read the slot before it is rewritten
  if (it_first >= n_items) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    return;
  }
  Load L, Ln;
  Item C, Cn;
  C.buf = 0;
  float amax = 0.0f;  // kSiluBf16: this lane's running max |h|
  decode_head(it_first, L, C);
  if (p.a_gather) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // own gather DMA
  decode_tail(L, C);
  stage_scales(L, C);
  i32x8 wbuf[P][2];
  int wexp[P];
#pragma unroll
  for (int s = 0; s < P; ++s) {
    wexp[s] = 0;
    issue(L, s, s, wbuf[s], wexp[s]);
  }

  // The next item is decoded at the first step of group `dgroup`, at least P
  // steps before its first loads are issued (in the last group) when an item
  // has two or more groups; its gathered row indices have landed by then.
  const int dgroup = groups >= 2 ? groups - 2 : 0;
  int cp_slot = 0;  // ring slot of the step being computed
  bool have_next = false;

  while (true) {
    constexpr int MF = ROWS / 16;
    const int mf = C.mf;
    f32x4 acc[MF][2];
#pragma unroll
    for (int i = 0; i < MF; ++i) {
      acc[i][0] = f32x4{0.f, 0.f, 0.f, 0.f};
      acc[i][1] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    for (int g = 0; g < groups; ++g) {
      const bool last_group = (g == groups - 1);
      if (g == dgroup && tid == 0) lds_write_i32(q_addr, nxt);  // read after the barrier below
#pragma unroll
      for (int s = 0; s < P; ++s) {
        const int kt = g * P + s;
        // scheduling barriers keep each step's MFMAs and loads inside the step,
        // so the operands of one step are live at a time
        __builtin_amdgcn_sched_barrier(0);
        wait_vm_barrier<G::kVm * (P - 1)>();
        __builtin_amdgcn_sched_barrier(0);
        if (s == 0 && g == dgroup) {
          const int it = __builtin_amdgcn_readfirstlane(lds_read_i32(q_addr));
          have_next = it < n_items;
          if (have_next) {
            Cn.buf = C.buf ^ 1;
            decode_head(it, Ln, Cn);
            if (tid == 0) nxt = fetch();
          } else {
            Ln = L;
            Cn = C;
          }
        }
        if (s == 0 && last_group && have_next) {
          // a single-group item decodes and reads its indices in one step
          if (groups == 1 && p.a_gather) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
          decode_tail(Ln, Cn);
          stage_scales(Ln, Cn);
        }
        const uint32_t st = smem_base + __builtin_amdgcn_readfirstlane(cp_slot) * G::kStage;
        const uint32_t sbuf = scale_base + C.buf * G::kScaleBuf;
        const uint32_t sa_addr = sbuf + kt * (ROWS * 4) + sa_lane;
        // fragment i (rows 16i..16i+15) only while the segment reaches it
        auto frag_step = [&](auto i_tag, float sb0, float sb1, int sbx) {
          constexpr int i = decltype(i_tag)::value;
          i32x8 af;
          if constexpr (kBlockSc) {
            // MFMAs from zero folded in with the block's scale product, in the
            // 256x256 kernel's arithmetic (fold_block)
            float sa_cur;
            lds_frag<2048 * i, 64 * i>(st + lo_off, st + hi_off, sa_addr, af, sa_cur);
            const float f0 = sa_cur * sb0;
            const float f1 = kSilu ? sa_cur * sb1 : f0;
            const f32x4 p0 = mfma_e4m3_16x16x128(wbuf[s][0], af, f32x4{0.f, 0.f, 0.f, 0.f});
            const f32x4 p1 = mfma_e4m3_16x16x128(wbuf[s][1], af, f32x4{0.f, 0.f, 0.f, 0.f});
            fold_block(acc[i][0], p0, f0);
            fold_block(acc[i][1], p1, f1);
          } else if constexpr (kMX) {
            float sa_bits;  // the row's four exponents of this K step: byte lg is K block lg
            lds_frag<2048 * i, 64 * i>(st + lo_off, st + hi_off, sa_addr, af, sa_bits);
            const int sa = static_cast<int>(__float_as_uint(sa_bits) >> (8 * lg));
            acc[i][0] = mfma_mx<0, 0>(wbuf[s][0], af, acc[i][0], sbx, sa);
            acc[i][1] = mfma_mx<kSilu ? 2 : 1, 0>(wbuf[s][1], af, acc[i][1], sbx, sa);
          } else {
            lds_frag<2048 * i>(st + lo_off, st + hi_off, af);
            acc[i][0] = mfma_e4m3_16x16x128(wbuf[s][0], af, acc[i][0]);
            acc[i][1] = mfma_e4m3_16x16x128(wbuf[s][1], af, acc[i][1]);
          }
          // each fragment's products are folded before the next fragment's LDS
          // reads (an empty volatile asm that takes the accumulators): the
          // kernel's VGPRs hold the weight prefetch window, and MFMA
          // temporaries sunk past the next fragments would spill it
          asm volatile("" : "+v"(acc[i][0]), "+v"(acc[i][1]));
        };
        if (!PAD || kt < k_steps) {
          float2 sbv = float2{0.f, 0.f};  // gate / only block, up block
          if constexpr (kBlockSc) sbv = lds_read_w2<G::kMaxSteps * 4>(sbuf + sb_wave + kt * 4);
          // MX: bytes of this wave's fragments in its 64-row group's words
          const int sbx = static_cast<int>(static_cast<uint32_t>(wexp[s]) >> ((kSilu ? 8 : 16) * (wave & 1)));
          frag_step(std::integral_constant<int, 0>{}, sbv.x, sbv.y, sbx);
          if constexpr (MF > 1) {
            if (mf > 1) frag_step(std::integral_constant<int, 1>{}, sbv.x, sbv.y, sbx);
            if (mf > 2) frag_step(std::integral_constant<int, 2>{}, sbv.x, sbv.y, sbx);
            if (mf > 3) frag_step(std::integral_constant<int, 3>{}, sbv.x, sbv.y, sbx);
          }
        }
        __builtin_amdgcn_sched_barrier(0);
        // loads P steps ahead: this item's step kt+P, or the next item's step s
        const int ld_slot = cp_slot == 0 ? P : cp_slot - 1;
        Load LL;
        LL.wsrd = last_group ? Ln.wsrd : L.wsrd;
        LL.ssrd = last_group ? Ln.ssrd : L.ssrd;
        LL.as_voff = 0;
        LL.valid = __builtin_amdgcn_readfirstlane(last_group ? Ln.valid : L.valid);
#pragma unroll
        for (int i = 0; i < G::kADma; ++i) LL.a_voff[i] = last_group ? Ln.a_voff[i] : L.a_voff[i];
        issue(LL, last_group ? s : kt + P, ld_slot, wbuf[s], wexp[s]);
        cp_slot = cp_slot == P ? 0 : cp_slot + 1;
      }
    }

    // ---- epilogue (the next item's first P steps are in flight) ----------
    // block-scaled and MX accumulators hold the scaled sums
    if constexpr (!kSilu) {
      const float tens = SC == Scale::kTensor ? C.tens : 1.0f;
#pragma unroll
      for (int i = 0; i < MF; ++i) {
        const int r = 16 * i + l16;
        if (i < mf && r < C.valid) {
          uint16_t* yrow = static_cast<uint16_t*>(p.c) + static_cast<int64_t>(C.row0 + r) * p.n_out +
                           C.col0 + 32 * wave + 4 * lg;
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            uint2 v;
            if constexpr (SC == Scale::kTensor) {
              v.x = pack_bf16x2(acc[i][j][0] * tens, acc[i][j][1] * tens);
              v.y = pack_bf16x2(acc[i][j][2] * tens, acc[i][j][3] * tens);
            } else {
              v.x = pack_bf16x2(acc[i][j][0], acc[i][j][1]);
              v.y = pack_bf16x2(acc[i][j][2], acc[i][j][3]);
            }
            st_nt8(yrow + 16 * j, v);  // not read again by this kernel
          }
        }
      }
    } else if constexpr (EPI == Epi::kSiluBf16) {
      // h = bf16(SiLU(gate) * up) and its running maximum
#pragma unroll
      for (int i = 0; i < MF; ++i) {
        const int r = 16 * i + l16;
        if (i < mf && r < C.valid) {
          float hv[4];
#pragma unroll
          for (int q = 0; q < 4; ++q) hv[q] = silu(acc[i][0][q] * C.tens) * (acc[i][1][q] * C.tens);
          const uint2 v = uint2{pack_bf16x2(hv[0], hv[1]), pack_bf16x2(hv[2], hv[3])};
          *reinterpret_cast<uint2*>(static_cast<uint16_t*>(p.c) + static_cast<int64_t>(C.row0 + r) * p.n_out +
                                    C.col0 + 16 * wave + 4 * lg) = v;
          amax = fmaxf(amax, fmaxf(fmaxf(fabsf(bf16_bits_to_f32(v.x & 0xffffu)), fabsf(bf16_bits_to_f32(v.x >> 16))),
                                   fmaxf(fabsf(bf16_bits_to_f32(v.y & 0xffffu)), fabsf(bf16_bits_to_f32(v.y >> 16)))));
        }
      }
    } else {
      // h = bf16(SiLU(gate) * up) staged in LDS, then each row's columns (one
      // 1x128 group, or MX: blocks of 32) requantised to e4m3 with their scale
#pragma unroll
      for (int i = 0; i < MF; ++i) {
        if (i >= mf) break;
        float hv[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) hv[q] = silu(acc[i][0][q]) * acc[i][1][q];
        uint2 v;
        v.x = pack_bf16x2(hv[0], hv[1]);
        v.y = pack_bf16x2(hv[2], hv[3]);
        lds_write_b64(lds_addr(ct + (16 * i + l16) * G::kCtLd + 16 * wave + 4 * lg), v);
      }
      lds_barrier();
      // 2 NW lanes per row, 8 columns each, the maxima by shuffles among the
      // 16 (MX: 4) lanes of a group; a 10-row segment keeps 160 lanes busy
      // instead of 20.
      constexpr int kLanes = 2 * NW;
      for (int base = 0; base < kLanes * C.valid; base += kT) {
        const int idx = base + tid, r = idx / kLanes, q = idx % kLanes;
        const bool live = r < C.valid;
        uint4 hv = uint4{0u, 0u, 0u, 0u};
        if (live) hv = lds_read_u4(lds_addr(ct + r * G::kCtLd + q * 8));
        const uint32_t w[4] = {hv.x, hv.y, hv.z, hv.w};
        float m = 0.0f;
#pragma unroll
        for (int u = 0; u < 4; ++u)
          m = fmaxf(m, fmaxf(fabsf(bf16_bits_to_f32(w[u] & 0xffffu)), fabsf(bf16_bits_to_f32(w[u] >> 16))));
#pragma unroll
        for (int o = 1; o < (kMX ? 4 : 16); o <<= 1) m = fmaxf(m, __shfl_xor(m, o, 64));
        if (live) {
          uint8_t* dst = static_cast<uint8_t*>(p.c) + static_cast<int64_t>(C.row0 + r) * p.n_out + C.col0 + q * 8;
          uint32_t qw[2];
          if constexpr (kMX) {
            // the quant_mx_kernel rule; the exponents go into this M tile's
            // words as one dword per row and K step (nt) of the next GEMM, the
            // order in which its narrow form reads them
            const uint32_t eb = min((__float_as_uint(m) >> 23) & 0xffu, 254u);
            const int sh = 127 - static_cast<int>(eb);
            auto qv = [&](uint32_t h) { return __builtin_amdgcn_ldexpf(bf16_bits_to_f32(h), sh); };
#pragma unroll
            for (int h2 = 0; h2 < 2; ++h2)
              qw[h2] = pack_e4m3x4(qv(w[2 * h2] & 0xffffu), qv(w[2 * h2] >> 16), qv(w[2 * h2 + 1] & 0xffffu),
                                   qv(w[2 * h2 + 1] >> 16));
            if ((q & 3) == 0) {
              const int64_t word = static_cast<int64_t>(C.nt) * p.cs_rs + static_cast<int64_t>(C.mnat) * kBM + r;
              reinterpret_cast<uint8_t*>(p.c_scale)[word * 4 + ((C.col0 & 127) >> 5) + (q >> 2)] =
                  static_cast<uint8_t>(eb);
            }
          } else {
            const float sc = scale_from_amax(m);
            const QuotScale qs = quot_scale(sc);
#pragma unroll
            for (int h2 = 0; h2 < 2; ++h2) {
              const uint32_t lo = w[2 * h2], hi = w[2 * h2 + 1];
              qw[h2] = pack_e4m3x4(quot_e4m3(bf16_bits_to_f32(lo & 0xffffu), qs),
                                   quot_e4m3(bf16_bits_to_f32(lo >> 16), qs),
                                   quot_e4m3(bf16_bits_to_f32(hi & 0xffffu), qs),
                                   quot_e4m3(bf16_bits_to_f32(hi >> 16), qs));
            }
            if (q == 0) p.c_scale[static_cast<int64_t>(C.nt) * p.rows + C.row0 + r] = sc;
          }
          st_nt8(dst, uint2{qw[0], qw[1]});
        }
      }
      // the staging tile is next written after at least P more barriers
    }
    if (!have_next) break;
    L = Ln;
    C = Cn;
  }
  // the re-loads issued after the last item land before the workgroup ends
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  if constexpr (EPI == Epi::kSiluBf16) {
    // one atomic per workgroup: the waves' maxima meet in LDS
    lds_barrier();
    amax = wave_max(amax);
    if (lane == 0) lds_write_i32(q_addr + 4 * wave, __float_as_int(amax));
    lds_barrier();
    if (tid == 0) {
      for (int w = 1; w < NW; ++w) amax = fmaxf(amax, __int_as_float(lds_read_i32(q_addr + 4 * w)));
      atomicMax(reinterpret_cast<unsigned int*>(p.amax), __float_as_uint(amax));
    }
  }
}

}  // namespace hkmoe
