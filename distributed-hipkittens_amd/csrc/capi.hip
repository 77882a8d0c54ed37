// C ABI of the gfx950 FP8 MoE path (declarations: include/hkmoe.h).
//
// Host code: argument validation (before any launch), launch configuration,
// workspace carving and stream-ordered enqueueing.  No host synchronisation and
// no allocation happens in any entry point: callers own every buffer, as with
// the reference's dispatch functions (include/pyutils/pyutils.cuh:54-71,
// kernels/cdna3/.../256_256_64_32.cpp:202-206).
#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <string>

#include "../../include/hkmoe.h"
#include "gemm_fp8.hpp"
#include "gemm_narrow.hpp"
#include "gemm_skinny.hpp"
#include "gemm_small.hpp"
#include "moe_kernels.hpp"

#include <atomic>
#include <cstdlib>
#include <mutex>
#include <vector>

using namespace hkmoe;

namespace {

thread_local std::string g_last_error;

int fail(int code, const char* fmt, ...) __attribute__((format(printf, 2, 3)));
int fail(int code, const char* fmt, ...) {
  char buf[512];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof(buf), fmt, ap);
  va_end(ap);
  g_last_error = buf;
  return code;
}

int check_launch(const char* what) {
  const hipError_t err = hipGetLastError();
  if (err != hipSuccess) return fail(HKMOE_ERR_HIP, "%s: %s", what, hipGetErrorString(err));
  return HKMOE_OK;
}

// ---------------------------------------------------------------------------
// Kernel timing of the layer entry points (hkmoe_kernel_timing).  While it is
// on, each kernel a layer call enqueues is launched by hipExtLaunchKernelGGL
// with a pair of library-owned events that take that dispatch's own start and
// end timestamps: no marker packet goes between the kernels, so the timed
// calls keep the untimed schedule, but for routing of at most kSmallTok tokens
// (three kernels instead of one, each with a time of its own).  One set of events per call, in a ring of
// `calls` sets; t_slot is the set of the call being enqueued (-1: untimed) and
// t_role the kernel role about to be launched.
// ---------------------------------------------------------------------------
struct KernelTiming {
  int calls = 0;                 // ring size, 0: off
  int next = 0;                  // next call's set
  int device = -1;
  std::vector<hipEvent_t> ev;    // [calls][HKMOE_TIMING_ROLES][2]
  std::vector<uint8_t> used;     // [calls][HKMOE_TIMING_ROLES]
  std::vector<int> first, last;  // [calls]: roles of the call's first and last launch
};
KernelTiming g_timing;
std::mutex g_timing_mu;
thread_local int t_slot = -1;
thread_local int t_role = -1;

// The events of the launch about to be made (false: launch untimed).
bool timing_events(hipEvent_t* start, hipEvent_t* stop) {
  if (t_slot < 0 || t_role < 0 || t_role >= HKMOE_TIMING_ROLES) return false;
  const size_t i = static_cast<size_t>(t_slot) * HKMOE_TIMING_ROLES + t_role;
  *start = g_timing.ev[2 * i];
  *stop = g_timing.ev[2 * i + 1];
  g_timing.used[i] = 1;
  if (g_timing.first[t_slot] < 0) g_timing.first[t_slot] = t_role;
  g_timing.last[t_slot] = t_role;
  return true;
}

// Every kernel of the layer entry points goes through here.
template <typename... Kargs, typename... Args>
void hk_launch(void (*kern)(Kargs...), dim3 grid, dim3 block, uint32_t lds, hipStream_t stream, Args... args) {
  hipEvent_t a, b;
  if (timing_events(&a, &b))
    hipExtLaunchKernelGGL(kern, grid, block, lds, stream, a, b, 0u, static_cast<Kargs>(args)...);
  else
    hipLaunchKernelGGL(kern, grid, block, lds, stream, static_cast<Kargs>(args)...);
}

// Marks the launches of one layer call as timed (a set of the ring) for its
// lifetime; does nothing while timing is off or on another device.  A timed
// call holds the timing mutex until it has enqueued its last launch, so
// timing_events never sees the ring replaced by a concurrent
// hkmoe_kernel_timing, and timed calls from several host threads take their
// sets one after the other.
struct TimedCall {
  bool on = false;
  std::unique_lock<std::mutex> lk;
  TimedCall() : lk(g_timing_mu) {
    int dev = -1;
    if (g_timing.calls <= 0 || hipGetDevice(&dev) != hipSuccess || dev != g_timing.device) {
      lk.unlock();
      return;
    }
    t_slot = g_timing.next;
    g_timing.next = (g_timing.next + 1) % g_timing.calls;
    std::fill_n(g_timing.used.begin() + static_cast<size_t>(t_slot) * HKMOE_TIMING_ROLES, HKMOE_TIMING_ROLES, 0);
    g_timing.first[t_slot] = g_timing.last[t_slot] = -1;
    on = true;
  }
  ~TimedCall() {
    if (on) t_slot = -1;
    t_role = -1;
  }
};

#define HK_REQUIRE(cond, ...)                                 \
  do {                                                        \
    if (!(cond)) return fail(HKMOE_ERR_INVALID_ARGUMENT, __VA_ARGS__); \
  } while (0)

#define HK_TRY(expr)               \
  do {                             \
    const int _rc = (expr);        \
    if (_rc != HKMOE_OK) return _rc; \
  } while (0)

constexpr int kMaxDevices = 64;

int device_cus() {
  static int cus[kMaxDevices] = {0};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return 256;
  if (cus[dev] == 0) {
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0)
      n = 256;
    cus[dev] = n;
  }
  return cus[dev];
}

int env_int(const char* name, int dflt) {
  const char* v = std::getenv(name);
  return (v && *v) ? std::atoi(v) : dflt;
}

size_t align256(size_t x) { return (x + 255) & ~static_cast<size_t>(255); }

int route_blocks(int64_t t) { return static_cast<int>((t + kRouteTok - 1) / kRouteTok); }

template <Epi EPI, Scale SC>
int launch_gemm(GemmParams p, hipStream_t stream, int grid_override = 0) {
  p.a_bytes = static_cast<uint32_t>(std::min<int64_t>(p.a_rows * p.K, 0xffffffffll));
  static bool attr_set[kMaxDevices] = {false};
  int dev = 0;
  (void)hipGetDevice(&dev);
  auto kern = gemm_fp8_persistent<EPI, SC>;
  if (dev >= 0 && dev < kMaxDevices && !attr_set[dev]) {
    const hipError_t err = hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                               hipFuncAttributeMaxDynamicSharedMemorySize, kLdsBytes);
    if (err != hipSuccess) return fail(HKMOE_ERR_HIP, "hipFuncSetAttribute: %s", hipGetErrorString(err));
    attr_set[dev] = true;
  }
  const int grid = grid_override > 0 ? grid_override : device_cus();
  hk_launch(kern, dim3(grid), dim3(kThreads), kLdsBytes, stream, p);
  return check_launch("gemm_fp8_persistent");
}

// MFMA shape of the 128x128-tile dense kernel (hkmoe_set_dense_mfma): 16 or 32.
// 32x32x64 is the default from the time of four waves per workgroup, where it was
// 4-7% faster.  On the eight waves of today the two are within 1-4%, 16x16x128 ahead
// (bf16 output, rotating operand copies, graph-replayed launches, best of three
// interleaved rounds on one box: 2048^3 13.3 / 13.7 us, 1024x4096x4096 21.6 / 22.2,
// 4096x2048x1024 17.0 / 17.1).
std::atomic<int> g_dense_mfma{32};

// The dense GEMM on 128x128 tiles (gemm_small.hpp): one workgroup per tile,
// the grid a whole number of 4x8 tile blocks.
template <bool F32OUT, bool M32, bool MX>
int launch_gemm_small(const SmallGemmParams& p, hipStream_t stream) {
  static bool attr_set[kMaxDevices] = {false};
  int dev = 0;
  (void)hipGetDevice(&dev);
  auto kern = gemm_fp8_small<F32OUT, M32, MX>;
  constexpr int lds = sm_lds_bytes(MX);
  if (dev >= 0 && dev < kMaxDevices && !attr_set[dev]) {
    const hipError_t err = hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                               hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (err != hipSuccess) return fail(HKMOE_ERR_HIP, "hipFuncSetAttribute: %s", hipGetErrorString(err));
    attr_set[dev] = true;
  }
  const int grid = ((p.m_tiles + 3) / 4) * p.nbn * 32;
  hipLaunchKernelGGL(kern, dim3(grid), dim3(kSmThreads), lds, stream, p);
  return check_launch("gemm_fp8_small");
}

template <int MF, int NF, int NW, bool MX, bool F32OUT>
int launch_gemm_skinny(const SkinnyParams& p, hipStream_t stream) {
  static bool attr_set[kMaxDevices] = {false};
  int dev = 0;
  (void)hipGetDevice(&dev);
  auto kern = gemm_fp8_skinny<MF, NF, NW, MX, F32OUT>;
  constexpr int lds = sk_lds_bytes(MF, NF, NW, MX);
  if (dev >= 0 && dev < kMaxDevices && !attr_set[dev]) {
    const hipError_t err = hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                               hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (err != hipSuccess) return fail(HKMOE_ERR_HIP, "hipFuncSetAttribute: %s", hipGetErrorString(err));
    attr_set[dev] = true;
  }
  const int64_t grid = static_cast<int64_t>(p.strips) * p.m_blocks;
  hipLaunchKernelGGL(kern, dim3(static_cast<unsigned>(grid)), dim3(NW * 64), lds, stream, p);
  return check_launch("gemm_fp8_skinny");
}
template <int MF, int NF, int NW, bool MX>
int launch_gemm_skinny(SkinnyParams p, bool f32out, hipStream_t stream) {
  p.strips = p.n / (16 * NF);
  p.m_blocks = (p.m + 16 * MF - 1) / (16 * MF);
  return f32out ? launch_gemm_skinny<MF, NF, NW, MX, true>(p, stream) : launch_gemm_skinny<MF, NF, NW, MX, false>(p, stream);
}

// Estimated times (us) of the dense kernels, from which the dense GEMM picks one:
// rounds of workgroups over the CUs x (ramp + K steps x time per step), or B's
// stream from HBM where that is longer (a tenth of the compute term breaks ties
// there).  The constants are fits to graph-replayed launches over rotating operand
// copies: on 1040 shapes (M = 1 .. 12000, N = 256 .. 16384, K = 128 .. 14336, both outputs
// and modes) the pick costs 0.8% over the best kernel on average; with one K step up to
// 30% (1 us), else 17%.
//   split-K strips against 128x128 tiles: 128x2048x8192 9.3 / 29.5 us, 128x8192x1024
//     6.4 / 7.0, 512x2048x2048 8.2 / 10.4 (and losing: 512x4096x4096 20.8 / 17.3)
//   128x128 against 256x256 tiles: 2048^3 13.9 / 25.6 us, 2048x4096x4096 40.8 / 48.1
//     (MX 44.8 / 52.5), 4096^3 79 / 51, 2048x8192x1024 28.3 / 21.2
// MX: the scaled MFMA's steps take longer in every kernel.
enum class DenseKernel { kStrip11, kStrip21, kStrip12, kStrip22, kStrip24, kStrip44, kTile128, kTile256 };

// Tile blocks of the dense 256x256 kernel: 2^b M tiles x 32 / 2^b N tiles, one
// block per XCD and round.  4 x 8 unless another shape needs fewer rounds: a
// block wider than N (or taller than M) leaves workgroups idle (12878x1024x1664,
// 51 x 4 tiles, fp32 out: 48.5 us in 4 x 8 blocks, whose right half is empty,
// 30.8 in 8 x 4).
int dense_block_log2(int64_t m, int64_t n, int64_t* rounds) {
  const uint64_t mt = (m + kBM - 1) / kBM, nt = n / kBN;
  int best = 2;
  uint64_t best_r = UINT64_MAX;
  for (int b : {2, 3, 1, 4, 5, 0}) {
    const uint64_t blocks = ((mt + (1u << b) - 1) >> b) * ((nt + (32u >> b) - 1) >> (5 - b));
    if ((blocks + 7) / 8 < best_r) best = b, best_r = (blocks + 7) / 8;
  }
  *rounds = static_cast<int64_t>(best_r);
  return best;
}

DenseKernel pick_dense(int64_t m, int64_t n, int64_t k, bool f32out, bool mx) {
  const double ks = static_cast<double>(k / kBK), cus = device_cus(), nk = static_cast<double>(n) * k;
  const uint64_t um = m, un = n, ncu = device_cus();
  DenseKernel best = DenseKernel::kTile256;
  double best_t = 0;
  auto offer = [&](DenseKernel kern, double compute, double hbm) {
    const double t = std::max(compute, hbm) + 0.1 * compute;
    if (kern == DenseKernel::kTile256 || t < best_t) best = kern, best_t = t;
  };
  {
    const double tiles = static_cast<double>((m + kBM - 1) / kBM) * (n / kBN);
    auto step = [&](double t) {  // per step, t tiles in the round
      return t <= cus / 4 ? (mx ? 1.12 : 0.95) : t <= cus / 2 ? (mx ? 1.27 : 1.13) : (mx ? 1.45 : 1.3);
    };
    int64_t rounds;
    (void)dense_block_log2(m, n, &rounds);
    const double full = static_cast<double>(rounds - 1), ramp = f32out ? 10 : 4.5;
    const double last = rounds == 1 ? tiles : std::max(1.0, std::min(cus, tiles - full * cus));
    offer(DenseKernel::kTile256, 5.4 + full * (ramp + ks * step(cus)) + ramp + ks * step(last), 0);
  }
  {
    // M tiles in fours: the workgroups that a 4x8 block has past M exit at once, but they
    // take their turns in the dispatch, and the live ones share a part of the CUs
    // (65x11264x2048, 88 live ones: 24 us, as two rounds would)
    const uint64_t mt = (um + kSmTile - 1) / kSmTile, nt = un / kSmTile, tiles = (mt + 3) / 4 * 4 * nt;
    const double full = static_cast<double>(tiles / ncu), part = static_cast<double>(tiles % ncu);
    const double live = std::min(part, static_cast<double>(mt * nt));  // of the last round
    const double busy = mx ? 0.58 : 0.52, idle = mx ? 0.51 : 0.40;  // per step, chip full / half full
    const double ramp = f32out ? 4.0 : 2.6;
    offer(DenseKernel::kTile128,
          1.75 + full * (ramp + ks * busy) + (part > 0 ? ramp + ks * (live <= cus / 2 ? idle : busy) : 0), 3 + nk / 2.0e6);
  }
  const struct {
    DenseKernel kern;
    int rows_log2, cols_log2, waves_log2;
    double ramp, step;
  } strips[] = {{DenseKernel::kStrip11, 4, 4, 3, 1.6, 0.055}, {DenseKernel::kStrip21, 5, 4, 3, 1.7, 0.075},
                {DenseKernel::kStrip12, 4, 5, 3, 1.7, 0.075}, {DenseKernel::kStrip22, 5, 5, 3, 1.85, 0.085},
                {DenseKernel::kStrip24, 5, 6, 2, 2.4, 0.13},  {DenseKernel::kStrip44, 6, 6, 2, 3.1, 0.215}};
  for (const auto& c : strips) {
    const uint64_t wgs = ((um + (1u << c.rows_log2) - 1) >> c.rows_log2) * (un >> c.cols_log2);
    const double rounds = static_cast<double>((wgs + ncu - 1) / ncu);
    const double steps = static_cast<double>(((k / kBK + (1 << c.waves_log2) - 1) >> c.waves_log2) << c.waves_log2);
    offer(c.kern, (mx ? 1.6 : 1.3) + rounds * (c.ramp + steps * c.step * (mx ? 1.1 : 1.0)), 3 + nk / 5.5e6);
  }
  return best;
}

// The dense GEMM (a, b, c and shapes checked by the caller).  MX: scale_a and
// scale_b are the packed exponent words.
template <bool MX>
int launch_dense(const void* a, const void* b, void* c, int64_t m, int64_t n, int64_t k, const float* scale_a,
                 const float* scale_b, int out_dtype, hipStream_t s) {
  const bool f32out = out_dtype == HKMOE_F32;
  const int32_t m64 = static_cast<int32_t>((m + 63) / 64 * 64);
  const DenseKernel kern = pick_dense(m, n, k, f32out, MX);
  if (kern < DenseKernel::kTile128) {
    SkinnyParams q{};
    q.a = static_cast<const uint8_t*>(a);
    q.b = static_cast<const uint8_t*>(b);
    q.c = c;
    q.a_scale = scale_a;
    q.b_scale = scale_b;
    q.m = static_cast<int32_t>(m);
    q.n = static_cast<int32_t>(n);
    q.k = static_cast<int32_t>(k);
    q.m64 = m64;
    switch (kern) {
      case DenseKernel::kStrip11: return launch_gemm_skinny<1, 1, 8, MX>(q, f32out, s);
      case DenseKernel::kStrip21: return launch_gemm_skinny<2, 1, 8, MX>(q, f32out, s);
      case DenseKernel::kStrip12: return launch_gemm_skinny<1, 2, 8, MX>(q, f32out, s);
      case DenseKernel::kStrip22: return launch_gemm_skinny<2, 2, 8, MX>(q, f32out, s);
      case DenseKernel::kStrip24: return launch_gemm_skinny<2, 4, 4, MX>(q, f32out, s);
      default: return launch_gemm_skinny<4, 4, 4, MX>(q, f32out, s);
    }
  }
  if (kern == DenseKernel::kTile128) {
    SmallGemmParams q{};
    q.a = static_cast<const uint8_t*>(a);
    q.b = static_cast<const uint8_t*>(b);
    q.c = c;
    q.a_scale = scale_a;
    q.b_scale = scale_b;
    q.m = static_cast<int32_t>(m);
    q.n = static_cast<int32_t>(n);
    q.k = static_cast<int32_t>(k);
    q.m64 = m64;
    q.a_bytes = static_cast<uint32_t>(std::min<int64_t>(m * k, 0xffffffffll));
    q.b_bytes = static_cast<uint32_t>(std::min<int64_t>(n * k, 0xffffffffll));
    q.m_tiles = static_cast<int32_t>((m + kSmTile - 1) / kSmTile);
    q.n_tiles = static_cast<int32_t>(n / kSmTile);
    q.nbn = (q.n_tiles + 7) / 8;
    if constexpr (MX) {
      return f32out ? launch_gemm_small<true, false, true>(q, s) : launch_gemm_small<false, false, true>(q, s);
    } else {
      if (g_dense_mfma.load() == 32)
        return f32out ? launch_gemm_small<true, true, false>(q, s) : launch_gemm_small<false, true, false>(q, s);
      return f32out ? launch_gemm_small<true, false, false>(q, s) : launch_gemm_small<false, false, false>(q, s);
    }
  }
  GemmParams p{};
  p.a = static_cast<const uint8_t*>(a);
  p.b = static_cast<const uint8_t*>(b);
  p.c = c;
  p.a_scale = scale_a;
  p.b_scale = scale_b;
  p.rows = m;
  p.a_rows = m;
  p.as_rs = m64;  // MX words per K step
  p.num_experts = 1;
  p.K = static_cast<int32_t>(k);
  p.nb = static_cast<int32_t>(n);
  p.n_out = static_cast<int32_t>(n);
  p.n_tiles = static_cast<int32_t>(n / kBN);
  int64_t rounds;
  p.blk_m_log2 = dense_block_log2(m, n, &rounds);
  constexpr Scale kSc = MX ? Scale::kMX : Scale::kTensor;
  return f32out ? launch_gemm<Epi::kStoreF32, kSc>(p, s) : launch_gemm<Epi::kStoreBf16, kSc>(p, s);
}

template <Epi EPI, Scale SC, int P, int NW, int ROWS, bool PAD>
int launch_narrow_v(const GemmParams& p, hipStream_t stream, int grid) {
  static bool attr_set[kMaxDevices] = {false};
  int dev = 0;
  (void)hipGetDevice(&dev);
  auto kern = gemm_fp8_narrow<EPI, SC, P, NW, ROWS, PAD>;
  using G = NarrowGeo<SC, P, NW, ROWS>;
  if (dev >= 0 && dev < kMaxDevices && !attr_set[dev]) {
    const hipError_t err = hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                               hipFuncAttributeMaxDynamicSharedMemorySize, G::kLds);
    if (err != hipSuccess) return fail(HKMOE_ERR_HIP, "hipFuncSetAttribute: %s", hipGetErrorString(err));
    attr_set[dev] = true;
  }
  hk_launch(kern, dim3(grid), dim3(G::kThreads), G::kLds, stream, p);
  return check_launch("gemm_fp8_narrow");
}

// Prefetch depth: 8 K steps where they divide the step count (and, with block
// scales, an item's scales fit beside that ring: 64 steps), else 4, the last
// group padded with empty steps.
template <Epi EPI, Scale SC, int NW, int ROWS>
int launch_narrow_p(const GemmParams& p, hipStream_t stream, int grid) {
  const int k_steps = p.K / kBK;
  if (k_steps % 8 == 0 && k_steps <= NarrowGeo<SC, 8, NW, ROWS>::kMaxSteps)
    return launch_narrow_v<EPI, SC, 8, NW, ROWS, false>(p, stream, grid);
  return launch_narrow_v<EPI, SC, 4, NW, ROWS, true>(p, stream, grid);
}

// How the narrow path shares a grouped GEMM.  count: device count of narrow M
// tiles (null: no narrow path, the 256x256 kernel takes every tile).  active ==
// 0: the 256x256 kernel on the other tiles; yield_from > 0 leaves CUs >=
// yield_from to the narrow kernel when it has work, < 0 is the late-join launch
// of `grid` workgroups.  active > 0: the narrow kernel on exactly the narrow
// tiles, on `grid` workgroups, `active` of them while 256x256 tiles exist;
// max_rows > 0: nothing runs beside it, and no segment has more rows.
struct NarrowPart {
  const int32_t* count = nullptr;
  int yield_from = 0, active = 0, grid = 0;
  int64_t max_rows = 0;
};

template <Epi EPI, Scale SC>
int launch_narrow(GemmParams p, hipStream_t stream, const NarrowPart& part) {
  p.a_bytes = static_cast<uint32_t>(std::min<int64_t>(p.a_rows * p.K, 0xffffffffll));
  const int grid = part.grid > 0 ? part.grid : part.active;
  if constexpr (EPI != Epi::kSiluQuant) {
    // Alone on the chip, items of half a tile (4 waves): finer last rounds, and
    // twice the items for shapes with fewer tiles than CUs.  Layer, 8 / 4 waves:
    // E=128 H=4096 I=1536 MX T=48 388 / 368 us, E=8 H=4096 I=14336 per-tensor T=29 264 /
    // 246 us.  With at most 16 rows per segment and no more than half a CU per tile, quarters
    // (2 waves, four workgroups per CU): E=128 T=1 second GEMM 24.6 -> 12.8 us; with more
    // tiles their fixed cost per item loses (T=4 49 / 41 us).
    const int64_t tiles = std::min<int64_t>(p.num_experts, p.rows) * p.n_tiles;  // at most
    if (part.max_rows > 0 && part.max_rows <= 16 && tiles <= grid / 2)
      return launch_narrow_p<EPI, SC, 2, 16>(p, stream, 4 * grid);
    if (part.max_rows > 0) return launch_narrow_p<EPI, SC, 4, kNarrowRows>(p, stream, grid);
  }
  return launch_narrow_p<EPI, SC, 8, kNarrowRows>(p, stream, grid);
}

// Narrow path settings, read once from the environment:
//   HKMOE_NARROW_CUS   workgroups (CUs) of the narrow kernels, 0 = off (default 64)
//   HKMOE_NARROW_MAX   largest expert (rows) the narrow kernel takes, <= 64 (default 64)
//   HKMOE_NARROW_SHARE 1: the first wide GEMM leaves those CUs to the narrow
//                      kernel while it has work; 0: it keeps them (default 1).  A
//                      wide GEMM that keeps every CU takes them first, and the
//                      narrow kernel then mostly runs after it.
// hkmoe_set_narrow overrides them.
struct NarrowConfig {
  int cus, max_rows, share;
};
std::mutex g_narrow_mu;
NarrowConfig& narrow_config_ref() {
  static NarrowConfig cfg = [] {
    NarrowConfig c;
    c.cus = std::max(0, env_int("HKMOE_NARROW_CUS", 64));
    c.max_rows = std::min(kNarrowRows, std::max(0, env_int("HKMOE_NARROW_MAX", kNarrowRows)));
    c.share = std::min(2, std::max(0, env_int("HKMOE_NARROW_SHARE", 1)));
    return c;
  }();
  return cfg;
}
NarrowConfig narrow_config() {
  std::lock_guard<std::mutex> g(g_narrow_mu);
  return narrow_config_ref();
}

// Tile blocks of the grouped GEMMs: 2^b M tiles x 32 / 2^b N tiles share an
// XCD's L2.  2^b = HKMOE_BLOCK_M1 (GEMM 1) / HKMOE_BLOCK_M2 (GEMM 2) from the
// environment (1, 2, 4, 8, 16 or 32; read once; other values give the
// default), default 2 M tiles x 16 N tiles: a block then spans one or two
// experts, whose N tiles share the A rows.  A measurement knob for the L2-miss
// traffic of other block shapes.
int block_m_log2(int gemm) {
  static const int b1 = [] {
    const int m = env_int("HKMOE_BLOCK_M1", 2);
    for (int t = 0; t <= 5; ++t)
      if (m == (1 << t)) return t;
    return 1;
  }();
  static const int b2 = [] {
    const int m = env_int("HKMOE_BLOCK_M2", 2);
    for (int t = 0; t <= 5; ++t)
      if (m == (1 << t)) return t;
    return 1;
  }();
  return gemm == 1 ? b1 : b2;
}

// Per-device auxiliary stream (default priority, non-blocking) and fork/join
// events of the one-call layer.  Created on the first call that is not being
// captured into a graph.  g_aux_mu guards g_aux from that creation on and keeps
// the fork/join sequences of concurrent host threads from interleaving on the shared
// events: a call takes it before it looks at g_aux and holds it until it has
// enqueued its join.
struct AuxStreams {
  hipStream_t aux = nullptr;
  hipEvent_t fork = nullptr, join = nullptr;
};
std::mutex g_aux_mu;
AuxStreams g_aux[kMaxDevices];

// The current device's auxiliary stream (null: none); the caller holds g_aux_mu.
int get_aux(hipStream_t main_stream, AuxStreams** out) {
  *out = nullptr;
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return HKMOE_OK;
  AuxStreams& a = g_aux[dev];
  if (a.aux == nullptr) {
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(main_stream, &st) != hipSuccess || st != hipStreamCaptureStatusNone)
      return HKMOE_OK;  // no set-up under capture: this call runs without the narrow path
    AuxStreams n;
    if (hipStreamCreateWithFlags(&n.aux, hipStreamNonBlocking) != hipSuccess ||
        hipEventCreateWithFlags(&n.fork, hipEventDisableTiming) != hipSuccess ||
        hipEventCreateWithFlags(&n.join, hipEventDisableTiming) != hipSuccess) {
      if (n.fork) (void)hipEventDestroy(n.fork);
      if (n.aux) (void)hipStreamDestroy(n.aux);
      (void)hipGetLastError();  // reported here, not by a later launch
      return fail(HKMOE_ERR_HIP, "moe_forward: cannot create the auxiliary stream / events");
    }
    a = n;
  }
  *out = &a;
  return HKMOE_OK;
}

// The allocation-free layer's workspace: one array per device, created with
// the code object, held until the process ends.  In host code `scratch` names
// a host-side stand-in: its device address (different on every GPU) comes from
// hipGetSymbolAddress, looked up once per device on the first call with that
// device current, and only that address is passed to kernels.
constexpr size_t kScratchBytes = HKMOE_NOALLOC_SCRATCH_BYTES;
static __device__ __align__(256) uint8_t scratch[kScratchBytes];
std::mutex g_scratch_mu;
void* g_scratch_ptr[kMaxDevices] = {};

int scratch_ptr(void** out) {
  *out = nullptr;
  int dev = 0;
  const hipError_t gerr = hipGetDevice(&dev);
  if (gerr != hipSuccess || dev < 0 || dev >= kMaxDevices)
    return fail(HKMOE_ERR_HIP, "moe_forward_noalloc: no usable current device (%s)", hipGetErrorString(gerr));
  std::lock_guard<std::mutex> g(g_scratch_mu);
  if (g_scratch_ptr[dev] == nullptr) {
    void* p = nullptr;
    const hipError_t err = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (err != hipSuccess || p == nullptr)
      return fail(HKMOE_ERR_HIP, "moe_forward_noalloc: hipGetSymbolAddress(scratch) on device %d: %s", dev,
                  hipGetErrorString(err));
    if ((reinterpret_cast<uintptr_t>(p) & 255) != 0)
      return fail(HKMOE_ERR_HIP, "moe_forward_noalloc: scratch of device %d is not 256-byte aligned", dev);
    g_scratch_ptr[dev] = p;
  }
  *out = g_scratch_ptr[dev];
  return HKMOE_OK;
}

// K step counts that hkmoe_grouped_gemm{1,2}_part take for part 1.
bool narrow_part_steps(int k_steps) { return k_steps % 2 == 0 && k_steps <= 64; }

// Workgroups the narrow kernels may take while 256x256 tiles exist: at most
// three quarters of the CUs, so the first 256x256 GEMM keeps at least a quarter
// of them whatever hkmoe_set_narrow asked for.
int narrow_cus_limit(int cus) { return std::min(cus, device_cus() - device_cus() / 4); }

// Joins the auxiliary stream back into the caller's stream when it goes out of
// scope, unless disarmed: every exit path after the fork (errors included)
// leaves the caller's stream ordered after the narrow kernels, which read and
// write the workspace, and a capture with the auxiliary stream joined.
struct AuxJoin {
  AuxStreams* a;
  hipStream_t s;
  bool armed = true;
  ~AuxJoin() {
    if (armed) {
      (void)hipEventRecord(a->join, a->aux);
      (void)hipStreamWaitEvent(s, a->join, 0);
    }
  }
};

int launch_expert_offsets(const int32_t* block_counts, int64_t num_tokens, int32_t num_experts,
                          int32_t* counts, int32_t* offsets, int32_t* block_base,
                          int32_t* mtile_offsets, int32_t* mtile_list, float* amax_reset,
                          int32_t* tile_counters, int narrow_max, const NarrowRule& rule, int32_t* narrow_info,
                          hipStream_t stream) {
  const int nblk = route_blocks(num_tokens);
  // few routing blocks: expert_offsets_kernel also does the block scan (one
  // launch instead of two; ~6 us less on a decode step's critical path)
  const bool fuse = nblk <= kOffFuseBlocks;
  if (!fuse) {
    const bool timed = t_role == HKMOE_TIMING_OFFSETS;
    if (timed) t_role = HKMOE_TIMING_BLOCK_SCAN;
    hk_launch(expert_block_scan_kernel, dim3((num_experts + kOffExperts - 1) / kOffExperts),
              dim3(kScanThreads), 0, stream, block_counts, nblk, num_experts, counts, block_base);
    HK_TRY(check_launch("expert_block_scan_kernel"));
    if (timed) t_role = HKMOE_TIMING_OFFSETS;
  }
  hk_launch(expert_offsets_kernel, dim3(1), dim3(kScanThreads), 0, stream, num_experts, counts, offsets,
            mtile_offsets, mtile_list, kBM, amax_reset, tile_counters, narrow_max, rule, narrow_info,
            block_counts, fuse ? nblk : -1, block_base);
  return check_launch("expert_offsets_kernel");
}


}  // namespace

extern "C" {

int hkmoe_version(void) { return 200; }

int hkmoe_set_narrow(int32_t cus, int32_t max_rows, int32_t wide_share) {
  HK_REQUIRE(cus >= 0 && cus <= 4096, "set_narrow: cus=%d outside [0, 4096]", cus);
  HK_REQUIRE(max_rows >= 0 && max_rows <= kNarrowRows, "set_narrow: max_rows=%d outside [0, %d]", max_rows,
             kNarrowRows);
  HK_REQUIRE(wide_share >= 0 && wide_share <= 2, "set_narrow: wide_share=%d outside [0, 2]", wide_share);
  std::lock_guard<std::mutex> g(g_narrow_mu);
  NarrowConfig& c = narrow_config_ref();
  c.cus = cus;
  c.max_rows = max_rows;
  c.share = wide_share;
  return HKMOE_OK;
}

int hkmoe_get_narrow(int32_t* cus, int32_t* max_rows, int32_t* wide_share) {
  HK_REQUIRE(cus && max_rows && wide_share, "get_narrow: null pointer");
  const NarrowConfig c = narrow_config();
  *cus = c.cus;
  *max_rows = c.max_rows;
  *wide_share = c.share;
  return HKMOE_OK;
}

const char* hkmoe_last_error(void) { return g_last_error.c_str(); }

int hkmoe_set_dense_mfma(int32_t shape) {
  HK_REQUIRE(shape == 16 || shape == 32, "set_dense_mfma: shape=%d must be 16 or 32", shape);
  g_dense_mfma.store(shape);
  return HKMOE_OK;
}

int hkmoe_get_dense_mfma(void) { return g_dense_mfma.load(); }

int hkmoe_gemm_fp8(const void* a, const void* b, void* c, int64_t m, int64_t n, int64_t k,
                   const float* scale_a, const float* scale_b, int out_dtype, hkmoe_stream_t stream) {
  HK_REQUIRE(b && (m == 0 || (a && c)), "gemm_fp8: null tensor pointer");
  HK_REQUIRE(m >= 0 && n > 0 && k > 0, "gemm_fp8: bad shape M=%lld N=%lld K=%lld", (long long)m,
             (long long)n, (long long)k);
  HK_REQUIRE(k % 128 == 0, "gemm_fp8: K=%lld must be a multiple of 128", (long long)k);
  HK_REQUIRE(n % kBN == 0, "gemm_fp8: N=%lld must be a multiple of 256", (long long)n);
  HK_REQUIRE(k <= (1 << 20) && n * k < (1ll << 32) && m * k < (1ll << 32) && m < (1ll << 31),
             "gemm_fp8: operand too large for 32-bit buffer offsets (M*K and N*K must be < 2^32)");
  HK_REQUIRE(out_dtype == HKMOE_BF16 || out_dtype == HKMOE_F32, "gemm_fp8: bad out_dtype %d", out_dtype);
  if (m == 0) return HKMOE_OK;
  return launch_dense<false>(a, b, c, m, n, k, scale_a, scale_b, out_dtype, static_cast<hipStream_t>(stream));
}

int hkmoe_route_blocks(int64_t num_tokens) { return route_blocks(num_tokens); }

int hkmoe_route_topk(const float* logits, int64_t num_tokens, int32_t num_experts, int32_t top_k,
                     int32_t* topk_idx, float* topk_w, int32_t* block_counts, hkmoe_stream_t stream) {
  HK_REQUIRE(num_tokens == 0 || (logits && topk_idx && topk_w && block_counts), "route_topk: null pointer");
  HK_REQUIRE(num_tokens >= 0 && num_tokens < (1ll << 31) / kMaxTopK, "route_topk: bad T=%lld",
             (long long)num_tokens);
  HK_REQUIRE(num_experts >= 1 && num_experts <= kMaxExperts, "route_topk: E=%d outside [1, %d]",
             num_experts, kMaxExperts);
  HK_REQUIRE(top_k >= 1 && top_k <= num_experts && top_k <= kMaxTopK,
             "route_topk: top_k=%d outside [1, min(E, %d)]", top_k, kMaxTopK);
  if (num_tokens == 0) return HKMOE_OK;
  const int per_lane = (num_experts + 15) / 16;  // experts per lane of a token's 16-lane row
  auto kern = per_lane <= 1 ? route_topk_kernel<1> : per_lane <= 2 ? route_topk_kernel<2>
            : per_lane <= 4 ? route_topk_kernel<4> : per_lane <= 8 ? route_topk_kernel<8>
            : per_lane <= 16 ? route_topk_kernel<16> : per_lane <= 32 ? route_topk_kernel<32>
                             : route_topk_kernel<64>;
  hk_launch(kern, dim3(route_blocks(num_tokens)), dim3(kTopkThreads), 0, static_cast<hipStream_t>(stream), logits,
            static_cast<int>(num_tokens), num_experts, top_k, topk_idx, topk_w, block_counts);
  return check_launch("route_topk_kernel");
}

int hkmoe_expert_offsets(const int32_t* block_counts, int64_t num_tokens, int32_t num_experts,
                         int32_t* counts, int32_t* offsets, int32_t* block_base,
                         int32_t* mtile_offsets, int32_t* mtile_list, float* amax_reset,
                         int32_t* tile_counters, hkmoe_stream_t stream) {
  HK_REQUIRE(counts && offsets && mtile_offsets && (num_tokens == 0 || block_base), "expert_offsets: null pointer");
  HK_REQUIRE(num_experts >= 1 && num_experts <= kMaxExperts, "expert_offsets: E=%d outside [1, %d]",
             num_experts, kMaxExperts);
  HK_REQUIRE(num_tokens >= 0, "expert_offsets: bad T");
  HK_REQUIRE(num_tokens == 0 || block_counts, "expert_offsets: null block_counts");
  return launch_expert_offsets(block_counts, num_tokens, num_experts, counts, offsets, block_base,
                               mtile_offsets, mtile_list, amax_reset, tile_counters, 0, NarrowRule{}, nullptr,
                               static_cast<hipStream_t>(stream));
}

int hkmoe_expert_offsets_narrow(const int32_t* block_counts, int64_t num_tokens, int32_t num_experts,
                                int32_t* counts, int32_t* offsets, int32_t* block_base,
                                int32_t* mtile_offsets, int32_t* mtile_list, float* amax_reset,
                                int32_t* tile_counters, int32_t narrow_max, int32_t* narrow_info,
                                hkmoe_stream_t stream) {
  HK_REQUIRE(counts && offsets && mtile_offsets && mtile_list && narrow_info && (num_tokens == 0 || block_base),
             "expert_offsets_narrow: null pointer");
  HK_REQUIRE(num_experts >= 1 && num_experts <= kMaxExperts, "expert_offsets_narrow: E=%d outside [1, %d]",
             num_experts, kMaxExperts);
  HK_REQUIRE(num_tokens >= 0, "expert_offsets_narrow: bad T");
  HK_REQUIRE(num_tokens == 0 || block_counts, "expert_offsets_narrow: null block_counts");
  HK_REQUIRE(narrow_max >= 0 && narrow_max <= kNarrowRows, "expert_offsets_narrow: narrow_max=%d outside [0, %d]",
             narrow_max, kNarrowRows);
  return launch_expert_offsets(block_counts, num_tokens, num_experts, counts, offsets, block_base,
                               mtile_offsets, mtile_list, amax_reset, tile_counters, narrow_max, NarrowRule{},
                               narrow_info,
                               static_cast<hipStream_t>(stream));
}

int hkmoe_scatter(const int32_t* topk_idx, int64_t num_tokens, int32_t num_experts, int32_t top_k,
                  const int32_t* offsets, const int32_t* block_base, int32_t* perm, int32_t* inv_perm,
                  const void* x_q, const float* x_scale, int64_t hidden, int scale_mode, void* xp,
                  float* xp_scale_t, hkmoe_stream_t stream) {
  HK_REQUIRE(num_tokens == 0 || (topk_idx && offsets && block_base && perm && inv_perm), "scatter: null pointer");
  HK_REQUIRE(num_experts >= 1 && num_experts <= kMaxExperts, "scatter: E=%d outside [1, %d]",
             num_experts, kMaxExperts);
  HK_REQUIRE(top_k >= 1 && top_k <= num_experts && top_k <= kMaxTopK, "scatter: bad top_k=%d", top_k);
  HK_REQUIRE(num_tokens >= 0, "scatter: bad T");
  HK_REQUIRE(scale_mode == HKMOE_SCALE_TENSOR || scale_mode == HKMOE_SCALE_BLOCK,
             "scatter: bad scale_mode %d", scale_mode);
  if (x_q != nullptr) {
    HK_REQUIRE(xp != nullptr, "scatter: x_q given without xp");
    HK_REQUIRE(hidden > 0 && hidden % 16 == 0, "scatter: hidden=%lld must be a multiple of 16",
               (long long)hidden);
    if (scale_mode == HKMOE_SCALE_BLOCK) {
      HK_REQUIRE(hidden % kGroup == 0, "scatter: hidden must be a multiple of 128 for block scales");
      HK_REQUIRE(x_scale && xp_scale_t, "scatter: block scales need x_scale and xp_scale_t");
    }
  }
  if (num_tokens == 0) return HKMOE_OK;
  hk_launch(scatter_kernel, dim3(route_blocks(num_tokens)), dim3(kRouteThreads), 0,
                     static_cast<hipStream_t>(stream), topk_idx, static_cast<int>(num_tokens),
                     num_experts, top_k, offsets, block_base, perm, inv_perm,
                     static_cast<const uint8_t*>(x_q), x_scale, hidden,
                     scale_mode == HKMOE_SCALE_BLOCK ? 1 : 0, static_cast<uint8_t*>(xp), xp_scale_t,
                     num_tokens * top_k);
  return check_launch("scatter_kernel");
}

static int grouped_gemm1_impl(const void* x, const float* x_scale, const int32_t* gather,
                              int32_t gather_div, int64_t x_rows, const void* w13, const float* w13_scale,
                              const int32_t* offsets, const int32_t* mtile_offsets,
                              const int32_t* mtile_list, int64_t rows,
                              int32_t num_experts, int32_t hidden, int32_t inter, int scale_mode,
                              int w_layout, int out_format, void* h, float* h_aux,
                              int32_t* tile_counters, hkmoe_stream_t stream,
                              const NarrowPart& part) {
  HK_REQUIRE(w13 && w13_scale && offsets && mtile_offsets, "grouped_gemm1: null pointer");
  HK_REQUIRE(rows == 0 || (x && x_scale && h), "grouped_gemm1: null pointer");
  HK_REQUIRE(num_experts >= 1 && num_experts <= kMaxExperts, "grouped_gemm1: bad E=%d", num_experts);
  HK_REQUIRE(hidden > 0 && hidden % kGroup == 0 && hidden <= kGroup * kMaxKBlocks,
             "grouped_gemm1: hidden=%d must be a multiple of 128 and <= %d", hidden, kGroup * kMaxKBlocks);
  HK_REQUIRE(inter > 0 && inter % 128 == 0, "grouped_gemm1: inter=%d must be a multiple of 128", inter);
  HK_REQUIRE(rows >= 0 && rows < (1ll << 31), "grouped_gemm1: bad rows");
  HK_REQUIRE(x_rows >= (rows > 0 ? 1 : 0) && x_rows * hidden < (1ll << 32), "grouped_gemm1: x_rows=%lld out of range",
             (long long)x_rows);
  HK_REQUIRE(gather == nullptr || gather_div >= 1, "grouped_gemm1: gather_div must be >= 1");
  HK_REQUIRE(gather != nullptr || x_rows >= rows, "grouped_gemm1: x has fewer rows than rows");
  HK_REQUIRE(2ll * inter * hidden < (1ll << 32), "grouped_gemm1: expert weight too large");
  HK_REQUIRE(scale_mode == HKMOE_SCALE_TENSOR || scale_mode == HKMOE_SCALE_BLOCK,
             "grouped_gemm1: bad scale_mode %d", scale_mode);
  HK_REQUIRE(w_layout == HKMOE_W_ROWS || w_layout == HKMOE_W_PACKED, "grouped_gemm1: bad w_layout %d",
             w_layout);
  HK_REQUIRE(out_format == HKMOE_BF16 || (out_format == HKMOE_E4M3 && scale_mode == HKMOE_SCALE_BLOCK),
             "grouped_gemm1: out_format %d not supported with scale_mode %d", out_format, scale_mode);
  HK_REQUIRE(out_format != HKMOE_E4M3 || rows == 0 || h_aux != nullptr, "grouped_gemm1: e4m3 output needs h_aux scales");
  if (rows == 0) return HKMOE_OK;
  GemmParams p{};
  p.a = static_cast<const uint8_t*>(x);
  p.a_gather = gather;
  p.gather_div = gather ? gather_div : 1;
  p.b = static_cast<const uint8_t*>(w13);
  p.c = h;
  p.a_scale = x_scale;
  p.b_scale = w13_scale;
  p.offsets = offsets;
  p.mtile_offsets = mtile_offsets;
  p.rows = rows;
  p.a_rows = x_rows;
  p.as_rs = hidden / kGroup;  // x_scale is row-major [x_rows, H/128]
  p.as_ks = 1;
  p.num_experts = num_experts;
  p.K = hidden;
  p.nb = 2 * inter;
  p.n_out = inter;
  p.n_tiles = inter / 128;
  p.b_packed = w_layout == HKMOE_W_PACKED;
  p.mtile_list = mtile_list;
  p.blk_m_log2 = block_m_log2(1);  // 2 x 16 tile blocks by default
  p.tile_ctr = tile_counters;
  p.narrow_cnt = part.count;
  p.yield_from = part.yield_from;
  p.narrow_active = part.active;
  auto s = static_cast<hipStream_t>(stream);
  if (part.active > 0) {
    if (part.count == nullptr || mtile_list == nullptr || tile_counters == nullptr ||
        (scale_mode == HKMOE_SCALE_BLOCK && out_format != HKMOE_E4M3))
      return fail(HKMOE_ERR_INVALID_ARGUMENT, "grouped_gemm1: the narrow kernel needs the M-tile list, an item "
                                              "counter and, with block scales, e4m3 output");
    if (scale_mode == HKMOE_SCALE_TENSOR) {
      p.amax = h_aux;
      return launch_narrow<Epi::kSiluBf16, Scale::kTensor>(p, s, part);
    }
    p.c_scale = h_aux;
    return launch_narrow<Epi::kSiluQuant, Scale::kBlock>(p, s, part);
  }
  if (scale_mode == HKMOE_SCALE_TENSOR) {
    p.amax = h_aux;
    return launch_gemm<Epi::kSiluBf16, Scale::kTensor>(p, s);
  }
  if (out_format == HKMOE_E4M3) {
    p.c_scale = h_aux;
    return launch_gemm<Epi::kSiluQuant, Scale::kBlock>(p, s, part.yield_from < 0 ? part.grid : 0);
  }
  return launch_gemm<Epi::kSiluBf16, Scale::kBlock>(p, s);
}

int hkmoe_grouped_gemm1(const void* x, const float* x_scale, const int32_t* gather,
                        int32_t gather_div, int64_t x_rows, const void* w13, const float* w13_scale,
                        const int32_t* offsets, const int32_t* mtile_offsets,
                        const int32_t* mtile_list, int64_t rows,
                        int32_t num_experts, int32_t hidden, int32_t inter, int scale_mode,
                        int w_layout, int out_format, void* h, float* h_aux,
                        int32_t* tile_counters, hkmoe_stream_t stream) {
  return grouped_gemm1_impl(x, x_scale, gather, gather_div, x_rows, w13, w13_scale, offsets,
                            mtile_offsets, mtile_list, rows, num_experts, hidden, inter, scale_mode,
                            w_layout, out_format, h, h_aux, tile_counters, stream, NarrowPart{});
}

int hkmoe_requant(const void* h, int64_t rows, int32_t inter, int scale_mode, const float* amax,
                  void* hq, float* hs, hkmoe_stream_t stream) {
  HK_REQUIRE(inter > 0 && inter % 128 == 0, "requant: inter=%d must be a multiple of 128", inter);
  HK_REQUIRE(rows >= 0, "requant: bad rows");
  // rows == 0: h and hq are empty; block scales hs too, a tensor scale is still written
  HK_REQUIRE(rows == 0 || (h && hq), "requant: null pointer");
  HK_REQUIRE(hs || (rows == 0 && scale_mode == HKMOE_SCALE_BLOCK), "requant: null pointer");
  auto s = static_cast<hipStream_t>(stream);
  if (scale_mode == HKMOE_SCALE_BLOCK) {
    if (rows == 0) return HKMOE_OK;
    HK_REQUIRE(rows < (1ll << 31), "requant: too many rows");
    hk_launch(requant_group_kernel, dim3(static_cast<unsigned>(rows)), dim3(256), 0, s,
                       static_cast<const uint16_t*>(h), rows, inter, static_cast<uint8_t*>(hq), hs);
    return check_launch("requant_group_kernel");
  }
  HK_REQUIRE(scale_mode == HKMOE_SCALE_TENSOR, "requant: bad scale_mode %d", scale_mode);
  HK_REQUIRE(amax != nullptr, "requant: per-tensor mode needs amax");
  const int64_t n8 = rows * inter / 8;
  const int grid = static_cast<int>(std::min<int64_t>(std::max<int64_t>(1, (n8 + 255) / 256), 4 * 1024));
  hk_launch(requant_tensor_kernel, dim3(grid), dim3(256), 0, s,
                     static_cast<const uint16_t*>(h), n8, amax, static_cast<uint8_t*>(hq), hs);
  return check_launch("requant_tensor_kernel");
}

static int grouped_gemm2_impl(const void* hq, const float* hs, const void* w2, const float* w2_scale,
                              const int32_t* offsets, const int32_t* mtile_offsets,
                              const int32_t* mtile_list, int64_t rows,
                              int32_t num_experts, int32_t hidden, int32_t inter, int scale_mode,
                              int w_layout, void* y, int32_t* tile_counters, hkmoe_stream_t stream,
                              const NarrowPart& part) {
  HK_REQUIRE(w2 && w2_scale && offsets && mtile_offsets, "grouped_gemm2: null pointer");
  HK_REQUIRE(rows == 0 || (hq && hs && y), "grouped_gemm2: null pointer");
  HK_REQUIRE(num_experts >= 1 && num_experts <= kMaxExperts, "grouped_gemm2: bad E=%d", num_experts);
  HK_REQUIRE(hidden > 0 && hidden % kBN == 0, "grouped_gemm2: hidden=%d must be a multiple of 256", hidden);
  HK_REQUIRE(inter > 0 && inter % kGroup == 0 && inter <= kGroup * kMaxKBlocks,
             "grouped_gemm2: inter=%d must be a multiple of 128 and <= %d", inter, kGroup * kMaxKBlocks);
  HK_REQUIRE(rows >= 0 && rows < (1ll << 31), "grouped_gemm2: bad rows");
  HK_REQUIRE(rows * inter < (1ll << 32), "grouped_gemm2: rows*inter must be < 2^32 (32-bit buffer offsets into hq)");
  HK_REQUIRE(static_cast<int64_t>(hidden) * inter < (1ll << 32), "grouped_gemm2: expert weight too large");
  HK_REQUIRE(scale_mode == HKMOE_SCALE_TENSOR || scale_mode == HKMOE_SCALE_BLOCK,
             "grouped_gemm2: bad scale_mode %d", scale_mode);
  HK_REQUIRE(w_layout == HKMOE_W_ROWS || w_layout == HKMOE_W_PACKED, "grouped_gemm2: bad w_layout %d",
             w_layout);
  if (rows == 0) return HKMOE_OK;
  GemmParams p{};
  p.a = static_cast<const uint8_t*>(hq);
  p.b = static_cast<const uint8_t*>(w2);
  p.c = y;
  p.a_scale = hs;
  p.b_scale = w2_scale;
  p.offsets = offsets;
  p.mtile_offsets = mtile_offsets;
  p.rows = rows;
  p.a_rows = rows;
  p.as_rs = 1;  // group scales are transposed [I/128, rows]
  p.as_ks = rows;
  p.num_experts = num_experts;
  p.K = inter;
  p.nb = hidden;
  p.n_out = hidden;
  p.n_tiles = hidden / kBN;
  p.b_packed = w_layout == HKMOE_W_PACKED;
  p.mtile_list = mtile_list;
  p.blk_m_log2 = block_m_log2(2);  // 2 x 16 tile blocks by default
  p.tile_ctr = tile_counters;
  p.narrow_cnt = part.count;
  p.yield_from = part.yield_from;
  p.narrow_active = part.active;
  auto s = static_cast<hipStream_t>(stream);
  if (part.active > 0) {
    if (part.count == nullptr || mtile_list == nullptr || tile_counters == nullptr)
      return fail(HKMOE_ERR_INVALID_ARGUMENT, "grouped_gemm2: the narrow kernel needs the M-tile list and an "
                                              "item counter");
    return scale_mode == HKMOE_SCALE_BLOCK ? launch_narrow<Epi::kStoreBf16, Scale::kBlock>(p, s, part)
                                           : launch_narrow<Epi::kStoreBf16, Scale::kTensor>(p, s, part);
  }
  return scale_mode == HKMOE_SCALE_BLOCK ? launch_gemm<Epi::kStoreBf16, Scale::kBlock>(p, s)
                                         : launch_gemm<Epi::kStoreBf16, Scale::kTensor>(p, s);
}

int hkmoe_grouped_gemm2(const void* hq, const float* hs, const void* w2, const float* w2_scale,
                        const int32_t* offsets, const int32_t* mtile_offsets,
                        const int32_t* mtile_list, int64_t rows,
                        int32_t num_experts, int32_t hidden, int32_t inter, int scale_mode,
                        int w_layout, void* y, int32_t* tile_counters, hkmoe_stream_t stream) {
  return grouped_gemm2_impl(hq, hs, w2, w2_scale, offsets, mtile_offsets, mtile_list, rows, num_experts,
                            hidden, inter, scale_mode, w_layout, y, tile_counters, stream, NarrowPart{});
}

int hkmoe_grouped_gemm1_part(const void* x, const float* x_scale, const int32_t* gather,
                             int32_t gather_div, int64_t x_rows, const void* w13, const float* w13_scale,
                             const int32_t* offsets, const int32_t* mtile_offsets,
                             const int32_t* mtile_list, int64_t rows, int32_t num_experts, int32_t hidden,
                             int32_t inter, int w_layout, void* hq, float* hs, int32_t* tile_counters,
                             const int32_t* narrow_info, int32_t part, int32_t grid, hkmoe_stream_t stream) {
  HK_REQUIRE(narrow_info && mtile_list, "grouped_gemm1_part: needs narrow_info and mtile_list");
  HK_REQUIRE(part == 0 || part == 1, "grouped_gemm1_part: part=%d must be 0 (wide) or 1 (narrow)", part);
  HK_REQUIRE(grid >= 0 && grid <= 65536, "grouped_gemm1_part: bad grid %d", grid);
  HK_REQUIRE(part == 0 || narrow_part_steps(hidden / kBK),
             "grouped_gemm1_part: the narrow kernel needs an even number of at most 64 128-wide K steps (H=%d)", hidden);
  if (part == 1) {
    // the narrow kernel's item counter: narrow_info[1], zeroed by hkmoe_expert_offsets_narrow
    return grouped_gemm1_impl(x, x_scale, gather, gather_div, x_rows, w13, w13_scale, offsets, mtile_offsets,
                              mtile_list, rows, num_experts, hidden, inter, HKMOE_SCALE_BLOCK, w_layout,
                              HKMOE_E4M3, hq, hs, const_cast<int32_t*>(narrow_info) + 1, stream,
                              NarrowPart{narrow_info, 0, grid > 0 ? grid : device_cus(), device_cus()});
  }
  return grouped_gemm1_impl(x, x_scale, gather, gather_div, x_rows, w13, w13_scale, offsets, mtile_offsets,
                            mtile_list, rows, num_experts, hidden, inter, HKMOE_SCALE_BLOCK, w_layout, HKMOE_E4M3,
                            hq, hs, tile_counters, stream, NarrowPart{narrow_info, grid});
}

int hkmoe_grouped_gemm2_part(const void* hq, const float* hs, const void* w2, const float* w2_scale,
                             const int32_t* offsets, const int32_t* mtile_offsets, const int32_t* mtile_list,
                             int64_t rows, int32_t num_experts, int32_t hidden, int32_t inter, int w_layout,
                             void* y, int32_t* tile_counters, const int32_t* narrow_info, int32_t part,
                             int32_t grid, hkmoe_stream_t stream) {
  HK_REQUIRE(narrow_info && mtile_list, "grouped_gemm2_part: needs narrow_info and mtile_list");
  HK_REQUIRE(part == 0 || part == 1, "grouped_gemm2_part: part=%d must be 0 (wide) or 1 (narrow)", part);
  HK_REQUIRE(grid >= 0 && grid <= 65536, "grouped_gemm2_part: bad grid %d", grid);
  HK_REQUIRE(part == 0 || narrow_part_steps(inter / kBK),
             "grouped_gemm2_part: the narrow kernel needs an even number of at most 64 128-wide K steps (I=%d)", inter);
  // the narrow kernel's item counter: narrow_info[2], zeroed by hkmoe_expert_offsets_narrow
  return grouped_gemm2_impl(hq, hs, w2, w2_scale, offsets, mtile_offsets, mtile_list, rows, num_experts, hidden,
                            inter, HKMOE_SCALE_BLOCK, w_layout, y,
                            part == 1 ? const_cast<int32_t*>(narrow_info) + 2 : tile_counters, stream,
                            part == 0 ? NarrowPart{narrow_info, grid}
                                      : NarrowPart{narrow_info, 0, grid > 0 ? grid : device_cus(), device_cus()});
}

int hkmoe_pack_weights(const void* w, int64_t num_experts, int64_t n, int64_t k, int32_t gate_up,
                       void* packed, hkmoe_stream_t stream) {
  HK_REQUIRE(w && packed, "pack_weights: null pointer");
  HK_REQUIRE(w != packed, "pack_weights: in-place packing is not supported");
  HK_REQUIRE(num_experts >= 0 && n > 0 && n % kBN == 0 && k > 0 && k % kBK == 0,
             "pack_weights: N=%lld must be a multiple of 256 and K=%lld of 128", (long long)n,
             (long long)k);
  HK_REQUIRE(n * k < (1ll << 32) && k <= kBK * kMaxKBlocks, "pack_weights: expert weight too large");
  HK_REQUIRE(gate_up == 0 || (gate_up > 0 && n == 2ll * gate_up),
             "pack_weights: gate_up=%d must be 0 or N/2", gate_up);
  const int64_t chunks = num_experts * n * k / 16;
  if (chunks == 0) return HKMOE_OK;
  const int grid = static_cast<int>(std::min<int64_t>((chunks + 255) / 256, 8 * 1024));
  hipLaunchKernelGGL(pack_weights_kernel, dim3(grid), dim3(256), 0, static_cast<hipStream_t>(stream),
                     static_cast<const uint8_t*>(w), n, static_cast<int>(k), gate_up,
                     static_cast<uint8_t*>(packed), chunks);
  return check_launch("pack_weights_kernel");
}

int hkmoe_requant_quotient_check(int32_t* counts, hkmoe_stream_t stream) {
  HK_REQUIRE(counts, "requant_quotient_check: null pointer");
  hipLaunchKernelGGL(requant_quotient_check_kernel, dim3(128, 37 + 27 + 1), dim3(128), 0,
                     static_cast<hipStream_t>(stream), counts);
  return check_launch("requant_quotient_check_kernel");
}

int hkmoe_combine(const void* y, const float* topk_w, const int32_t* inv_perm, int64_t num_tokens,
                  int32_t top_k, int32_t hidden, void* out, hkmoe_stream_t stream) {
  HK_REQUIRE(num_tokens == 0 || (y && topk_w && inv_perm && out), "combine: null pointer");
  HK_REQUIRE(top_k >= 1 && top_k <= kMaxTopK, "combine: bad top_k=%d", top_k);
  HK_REQUIRE(hidden > 0 && hidden % 8 == 0, "combine: hidden=%d must be a multiple of 8", hidden);
  HK_REQUIRE(num_tokens >= 0 && num_tokens < (1ll << 31), "combine: bad T");
  if (num_tokens == 0) return HKMOE_OK;
  // the largest multiple of 64 threads (<= 512) that divides the row's 16-byte
  // chunks, so no workgroup ends on a partly idle pass (H = 7168: 448 threads
  // and two passes instead of 256 and a half-empty fourth); 256 otherwise
  const int chunks = hidden / 8;
  int threads = 256;
  for (int t = 512; t >= 64; t -= 64)
    if (chunks % t == 0) {
      threads = t;
      break;
    }
  hk_launch(combine_kernel, dim3(static_cast<unsigned>(num_tokens)), dim3(threads), 0,
                     static_cast<hipStream_t>(stream), static_cast<const uint16_t*>(y), topk_w,
                     inv_perm, top_k, hidden, static_cast<uint16_t*>(out));
  return check_launch("combine_kernel");
}

// ---------------------------------------------------------------------------
// whole layer
// ---------------------------------------------------------------------------
namespace {
struct MoeWorkspace {
  int32_t* topk_idx;
  float* topk_w;
  int32_t* block_counts;
  int32_t* block_base;
  int32_t* counts;
  int32_t* offsets;
  int32_t* mtile_offsets;
  int32_t* mtile_list;  // [M tiles][2], at most ceil(T*k/256) + E tiles
  float* amax;
  int32_t* tile_ctr;  // HKMOE_TILE_COUNTERS
  int32_t* narrow_info;  // [0] narrow M tiles, [1] / [2] narrow item counters of GEMM 1 / 2,
                         // [3] / [4] their active-slot counters
  int32_t* perm;
  int32_t* inv_perm;
  uint16_t* h;   // per-tensor mode only: bf16 intermediate before requantisation
  uint8_t* hq;
  float* hs;     // block: group scales; MX: packed e8m0 words of hq [I/128][ws]
  uint32_t* xw;  // MX only: packed e8m0 words of the gathered x rows [H/128][ws]
  uint16_t* y;
  size_t bytes;
};

// Words per K step of the tile-aligned MX exponent layouts: every M tile
// (at most ceil(rows/256) + E of them) owns 256 words.
int64_t mx_words_per_step(int64_t rows, int32_t e) { return ((rows + kBM - 1) / kBM + e) * kBM; }

MoeWorkspace carve(uint8_t* base, int64_t t, int32_t e, int32_t k, int32_t hidden, int32_t inter,
                   int mode) {
  const bool block = mode == HKMOE_SCALE_BLOCK, mx = mode == HKMOE_SCALE_MX;
  MoeWorkspace w{};
  size_t off = 0;
  const int64_t r = t * k;
  const int64_t nblk = route_blocks(t);
  auto take = [&](size_t bytes) -> uint8_t* {
    uint8_t* p = base ? base + off : nullptr;
    off += align256(bytes);
    return p;
  };
  w.topk_idx = reinterpret_cast<int32_t*>(take(r * 4));
  w.topk_w = reinterpret_cast<float*>(take(r * 4));
  w.block_counts = reinterpret_cast<int32_t*>(take(nblk * e * 4));
  w.block_base = reinterpret_cast<int32_t*>(take(nblk * e * 4));
  w.counts = reinterpret_cast<int32_t*>(take(e * 4));
  w.offsets = reinterpret_cast<int32_t*>(take((e + 1) * 4));
  w.mtile_offsets = reinterpret_cast<int32_t*>(take((e + 1) * 4));
  w.mtile_list = reinterpret_cast<int32_t*>(take(((r + kBM - 1) / kBM + e) * 8));
  w.amax = reinterpret_cast<float*>(take(4));
  w.tile_ctr = reinterpret_cast<int32_t*>(take(HKMOE_TILE_COUNTERS * 4));
  w.narrow_info = reinterpret_cast<int32_t*>(take((1 + kNarrowCounters) * 4));  // HKMOE_NARROW_INFO ints
  w.perm = reinterpret_cast<int32_t*>(take(r * 4));
  w.inv_perm = reinterpret_cast<int32_t*>(take(r * 4));
  const int64_t ws = mx_words_per_step(r, e);
  w.h = (block || mx) ? nullptr : reinterpret_cast<uint16_t*>(take(r * inter * 2));
  w.hq = take(r * inter);
  w.hs = reinterpret_cast<float*>(take(block ? r * (inter / kGroup) * 4 : mx ? (inter / kGroup) * ws * 4 : 4));
  w.xw = mx ? reinterpret_cast<uint32_t*>(take((hidden / kGroup) * ws * 4)) : nullptr;
  w.y = reinterpret_cast<uint16_t*>(take(r * hidden * 2));
  w.bytes = off;
  return w;
}
}  // namespace

size_t hkmoe_moe_workspace_size(int64_t num_tokens, int32_t num_experts, int32_t top_k,
                                int32_t hidden, int32_t inter, int scale_mode) {
  if (num_tokens < 0 || num_experts < 1 || top_k < 1 || hidden < 1 || inter < 1) return 0;
  if (scale_mode != HKMOE_SCALE_TENSOR && scale_mode != HKMOE_SCALE_BLOCK && scale_mode != HKMOE_SCALE_MX)
    return 0;
  return carve(nullptr, num_tokens, num_experts, top_k, hidden, inter, scale_mode).bytes;
}

// Which schedule the layer's experts take.  Experts of at most
// HKMOE_NARROW_MAX rows go to the weight-streaming narrow kernels, in one of two ways:
//   seq: up to 2*max_rows rows per expert on average (T*k <= 2*E*max_rows) the
//     small experts' weight stream dominates: the narrow kernels run on `stream`
//     after the 256x256 ones, each on every CU, without the fork to the auxiliary stream and the join
//     back (about 20 us of cross-stream latency).  Measured on the block-scaled config-3
//     shape (H=7168, I=2048, E=256, k=8): T=512 / 1024 / 2048 / 4096 run 26 / 21 /
//     13 / 4% faster on one stream, T=6144 / 8192 10 / 8% slower;
//   aux: on the library's auxiliary stream, beside the 256x256 kernels of the
//     larger experts on `stream`.  Not with per-tensor scales, whose
//     requantisation between the GEMMs needs both parts of GEMM 1.
struct NarrowPlan {
  NarrowConfig cfg{};
  bool seq = false;
  NarrowRule rule;  // beside larger experts (narrow_limit); not met, the 256x256 kernels take all
  AuxStreams* aux = nullptr;
  std::unique_lock<std::mutex> lock;  // of g_aux_mu, held with aux until the join is enqueued
  bool on() const { return seq || aux != nullptr; }
};

// aux_ok: the layer may use the auxiliary stream (else layers that need it run
// the 256x256 kernels alone).  tuned: block scales and at most 64 K steps, an even
// number, in both GEMMs; the lines above were measured there.  For the rest
// (per-tensor and MX scales, other step counts) the 256x256 kernels lose less to
// small experts, and with experts of both kinds each kernel's start and tail cost
// 30 us or so.  They take the narrow path
//   with at most max_rows tokens (every expert is narrow): E=8 H=4096 I=14336
//     per-tensor T=29 326 -> 245 us, E=128 H=4096 I=1536 MX T=48 453 -> 358 us.
//     Row-major weights, which the narrow kernel reads at 5.0-5.4 TB/s, only up to
//     kRowMajorBytes of them (T=64 above: 498 -> 482 us; the 256x256 kernels reach
//     5.9 on more: E=256 H=7168 I=2048 T=40 1376, narrow 1505 us);
//   and with packed weights of at least 256 experts
//     where no expert has more rows (the device decides): E=256 H=7168 I=2048
//       per-tensor uniform T=700 1959 -> 1718 us, H=2048 I=768 MX T=400 320 -> 256,
//       E=1024 H=1024 I=512 MX T=900 580 -> 383; 0.49 to 0.99 of the 256x256 kernels'
//       time over 432 such batches;
//     and beside larger experts, where the small ones pay (mixed_rule): on one stream
//       if they save more than the second start and tail of each GEMM cost.  One saves
//       0.25 us and 0.015 us per MB of its weights, less 0.002 us and 0.0004 us per MB
//       for each row (per-tensor 0.36, 0.006, 0 and 0.0006): at 50-60 rows the narrow kernel
//       gains little over a 256x256 tile.  MX T=4500: E=256 H=7168 I=2048 skewed, 118 small ones,
//       2365 -> 2265 us; E=512 H=2048 I=512 uniform, 121 of 60 rows, would go 513 -> 553.
//       On two streams at least 100 (108 to 147 gained 2-9%, whatever their size).
//       Over 1224 batches (E = 256-1024, experts of 1.6-47 MB, T = 65-8192, uniform and
//       skewed) those sent here took 1.02 of the 256x256 kernels' time at most; one
//       number of small experts for all layers, 112, lost up to 9% on 87 of them.
//       MX and block scales run on one stream up to kMixedSeqRows rows per expert (T=5000
//       2580 -> 2482 us, on two 2654), on two above (T=6500 3175 -> 2786, on one 3034).
//     Where neither holds, the empty narrow GEMMs take 4-6 us (on two streams 12).  Nothing
//     is launched where not all experts can be small and more than half would have to pay.
//   Fewer experts stay with the 256x256 kernels: uniform batches of E=128 and 192 would
//     gain 10-15%, but small layers would pay those 4-6 us on every skewed one.
static NarrowRule mixed_rule(int64_t expert_bytes, bool tensor, bool one_stream) {
  if (!one_stream) return NarrowRule{100, 1, 0};
  const double mb = 1e-6 * static_cast<double>(expert_bytes);
  auto ns = [](double v) { return static_cast<int32_t>(v + 0.5); };
  return tensor ? NarrowRule{40000, ns(360 + 6 * mb), ns(0.6 * mb)}
                : NarrowRule{60000, ns(250 + 15 * mb), ns(2 + 0.4 * mb)};
}
constexpr int64_t kMixedSeqRows = 176, kMixedTensorRows = 256;
constexpr int64_t kRowMajorBytes = 2500000000;
struct NarrowCall {
  int64_t tokens, rows;
  int32_t experts;
  int64_t expert_bytes;  // both weights of one expert
  bool tuned, tensor, packed, aux_ok;
};
static int plan_narrow(const NarrowCall& c, hipStream_t s, NarrowPlan* plan) {
  plan->cfg = narrow_config();
  const int64_t max_rows = plan->cfg.max_rows;
  if (plan->cfg.cus <= 0 || max_rows <= 0) return HKMOE_OK;
  if (c.tuned) {
    plan->seq = c.tokens <= max_rows || c.rows <= 2 * c.experts * max_rows;
  } else if (c.tokens <= max_rows) {
    plan->seq = c.packed || std::min<int64_t>(c.rows, c.experts) * c.expert_bytes <= kRowMajorBytes;
    if (!plan->seq) return HKMOE_OK;
  } else {
    if (c.experts < 256 || !c.packed) return HKMOE_OK;
    plan->seq = c.rows <= c.experts * (c.tensor ? kMixedTensorRows : kMixedSeqRows);
    plan->rule = mixed_rule(c.expert_bytes, c.tensor, plan->seq);
    if (plan->seq && c.rows > c.experts * max_rows &&
        static_cast<int64_t>(c.experts) * plan->rule.per_expert < 2ll * plan->rule.need) {
      plan->seq = false;
      return HKMOE_OK;
    }
  }
  if (plan->seq || !c.aux_ok) return HKMOE_OK;
  plan->lock = std::unique_lock<std::mutex>(g_aux_mu);
  const int rc = get_aux(s, &plan->aux);
  if (plan->aux == nullptr) plan->lock.unlock();
  return rc;
}

// Routing, permutation, both grouped GEMMs and the combine, enqueued by `plan`.
// gemm1 / gemm2(part, counters, stream) launch one grouped GEMM; prep() what the
// 256x256 kernel of GEMM 1 needs beyond the routing tables; mid() what comes between
// the GEMMs.
extern "C++" {
// route_topk, expert_offsets and scatter of at most kSmallTok tokens in one launch.
static int launch_route_small(const float* logits, const MoeWorkspace& w, int64_t num_tokens, int32_t num_experts,
                              int32_t top_k, int narrow_max, const NarrowRule& rule, int32_t* narrow_info,
                              hipStream_t s) {
  const int per_lane = (num_experts + 15) / 16;  // experts per lane of a token's 16-lane row
  auto kern = per_lane <= 1 ? route_small_kernel<1> : per_lane <= 2 ? route_small_kernel<2>
            : per_lane <= 4 ? route_small_kernel<4> : per_lane <= 8 ? route_small_kernel<8>
            : per_lane <= 16 ? route_small_kernel<16> : per_lane <= 32 ? route_small_kernel<32>
                             : route_small_kernel<64>;
  hk_launch(kern, dim3(1), dim3(kScanThreads), 0, s, logits, static_cast<int>(num_tokens), num_experts, top_k,
            w.topk_idx, w.topk_w, w.counts, w.offsets, w.mtile_offsets, w.mtile_list, kBM, w.amax, w.tile_ctr,
            narrow_max, rule, narrow_info, w.perm, w.inv_perm);
  return check_launch("route_small_kernel");
}

template <typename Prep, typename G1, typename Mid, typename G2>
int moe_enqueue(const float* logits, const MoeWorkspace& w, int64_t num_tokens, int32_t num_experts, int32_t top_k,
                int32_t hidden, void* out, hipStream_t s, NarrowPlan& plan, Prep prep, G1 gemm1, Mid mid, G2 gemm2) {
  const NarrowConfig& nc = plan.cfg;
  const int cus = device_cus();
  TimedCall timed_call;
  t_role = HKMOE_TIMING_ROUTE;
  // (a timed call takes the three steps apart, so that each has a time of its own)
  if (num_tokens <= kSmallTok && !timed_call.on) {
    HK_TRY(launch_route_small(logits, w, num_tokens, num_experts, top_k, plan.on() ? nc.max_rows : 0,
                              plan.rule, plan.on() ? w.narrow_info : nullptr, s));
  } else {
    HK_TRY(hkmoe_route_topk(logits, num_tokens, num_experts, top_k, w.topk_idx, w.topk_w, w.block_counts, s));
    t_role = HKMOE_TIMING_OFFSETS;
    HK_TRY(launch_expert_offsets(w.block_counts, num_tokens, num_experts, w.counts, w.offsets, w.block_base,
                                 w.mtile_offsets, w.mtile_list, w.amax, w.tile_ctr, plan.on() ? nc.max_rows : 0,
                                 plan.rule, plan.on() ? w.narrow_info : nullptr, s));
    t_role = HKMOE_TIMING_SCATTER;
    HK_TRY(hkmoe_scatter(w.topk_idx, num_tokens, num_experts, top_k, w.offsets, w.block_base, w.perm, w.inv_perm,
                         nullptr, nullptr, hidden, HKMOE_SCALE_TENSOR, nullptr, nullptr, s));
  }
  if (plan.seq) {
    // each 256x256 GEMM keeps every CU and skips the narrow experts' tiles; each
    // narrow GEMM then runs its items on every CU.  A token's k experts are
    // distinct, so no expert has more than T rows: with T <= max_rows every
    // expert is narrow, and the 256x256 GEMMs, which would find no tile, are not
    // launched.
    const bool wide = num_tokens > nc.max_rows;
    const NarrowPart skip{w.narrow_info}, narrow{w.narrow_info, 0, cus, cus, std::min<int64_t>(num_tokens, nc.max_rows)};
    if (wide) {
      HK_TRY(prep());
      t_role = HKMOE_TIMING_GEMM1;
      HK_TRY(gemm1(skip, w.tile_ctr, s));
    }
    t_role = HKMOE_TIMING_GEMM1_NARROW;
    HK_TRY(gemm1(narrow, w.narrow_info + 1, s));
    HK_TRY(mid());
    t_role = HKMOE_TIMING_GEMM2;
    if (wide) HK_TRY(gemm2(skip, w.tile_ctr + 8, s));
    t_role = HKMOE_TIMING_GEMM2_NARROW;
    HK_TRY(gemm2(narrow, w.narrow_info + 2, s));
  } else if (AuxStreams* aux = plan.aux) {
    // fork: both GEMMs of the narrow experts on the auxiliary stream, enqueued
    // first so that their workgroups find free CUs; join before the combine
    // (prep() first: beside the narrow kernels its few workgroups would wait for
    // CUs, 69 against 12 us for the MX words, and the 256x256 GEMM 1 with them)
    HK_TRY(prep());
    const int ncus = narrow_cus_limit(nc.cus);
    // Which workgroups work is decided on the device from narrow_info: with
    // experts of both kinds the narrow kernels use ncus workgroups and (share)
    // the first 256x256 GEMM leaves them those CUs; with one kind only, that
    // kind gets every CU it was launched on.
    if (hipEventRecord(aux->fork, s) != hipSuccess)
      return fail(HKMOE_ERR_HIP, "moe_forward: fork event failed");
    const int yield_from = nc.share ? cus - ncus : 0;  // >= device_cus() / 4
    if (hipStreamWaitEvent(aux->aux, aux->fork, 0) != hipSuccess)
      return fail(HKMOE_ERR_HIP, "moe_forward: fork to the auxiliary stream failed");
    AuxJoin guard{aux, s};
    // the narrow kernels launch one workgroup per CU: beside 256x256 tiles the
    // first ncus to start take items, else all of them (decode-like shapes)
    const NarrowPart narrow{w.narrow_info, 0, ncus, cus};
    t_role = HKMOE_TIMING_GEMM1_NARROW;
    HK_TRY(gemm1(narrow, w.narrow_info + 1, aux->aux));
    t_role = HKMOE_TIMING_GEMM2_NARROW;
    HK_TRY(gemm2(narrow, w.narrow_info + 2, aux->aux));
    // share == 2: once the narrow GEMMs are done, their CUs join the first 256x256
    // GEMM's tile queues (a second launch of it on the auxiliary stream, which
    // takes whatever tiles are left); the second 256x256 GEMM then waits for both.
    const bool late_join = nc.share == 2;
    t_role = HKMOE_TIMING_GEMM1_JOIN;
    if (late_join) HK_TRY(gemm1(NarrowPart{w.narrow_info, -1, 0, ncus}, w.tile_ctr, aux->aux));
    if (hipEventRecord(aux->join, aux->aux) != hipSuccess)
      return fail(HKMOE_ERR_HIP, "moe_forward: join event failed");
    t_role = HKMOE_TIMING_GEMM1;
    HK_TRY(gemm1(NarrowPart{w.narrow_info, yield_from}, w.tile_ctr, s));
    if (late_join && hipStreamWaitEvent(s, aux->join, 0) != hipSuccess)
      return fail(HKMOE_ERR_HIP, "moe_forward: join of the auxiliary stream failed");
    t_role = HKMOE_TIMING_GEMM2;
    HK_TRY(gemm2(NarrowPart{w.narrow_info}, w.tile_ctr + 8, s));
    if (!late_join && hipStreamWaitEvent(s, aux->join, 0) != hipSuccess)
      return fail(HKMOE_ERR_HIP, "moe_forward: join of the auxiliary stream failed");
    guard.armed = false;  // joined above
    plan.lock.unlock();
  } else {
    HK_TRY(prep());
    t_role = HKMOE_TIMING_GEMM1;
    HK_TRY(gemm1(NarrowPart{}, w.tile_ctr, s));
    HK_TRY(mid());
    t_role = HKMOE_TIMING_GEMM2;
    HK_TRY(gemm2(NarrowPart{}, w.tile_ctr + 8, s));
  }
  t_role = HKMOE_TIMING_COMBINE;
  return hkmoe_combine(w.y, w.topk_w, w.inv_perm, num_tokens, top_k, hidden, out, s);
}
}  // extern "C++"

// The layer; aux_ok: the narrow path may fork to the library's auxiliary
// stream (else every kernel runs on `stream`: the one-stream narrow schedule
// where it applies, otherwise the 256x256 kernels alone).
static int moe_forward_impl(const void* x_q, const float* x_scale, const float* logits, const void* w13,
                            const float* w13_scale, const void* w2, const float* w2_scale,
                            int64_t num_tokens, int32_t num_experts, int32_t top_k, int32_t hidden,
                            int32_t inter, int scale_mode, int w_layout, void* out, void* workspace,
                            size_t workspace_bytes, hkmoe_stream_t stream, bool aux_ok) {
  // with no tokens the activations, the output and the workspace may be empty
  // (null); the weights and shapes are checked either way
  HK_REQUIRE(w13 && w13_scale && w2 && w2_scale, "moe_forward: null pointer");
  HK_REQUIRE(num_tokens == 0 || (x_q && x_scale && logits && out), "moe_forward: null pointer");
  HK_REQUIRE(scale_mode == HKMOE_SCALE_TENSOR || scale_mode == HKMOE_SCALE_BLOCK,
             "moe_forward: bad scale_mode %d", scale_mode);
  HK_REQUIRE(w_layout == HKMOE_W_ROWS || w_layout == HKMOE_W_PACKED, "moe_forward: bad w_layout %d",
             w_layout);
  HK_REQUIRE(num_tokens >= 0 && num_tokens * top_k < (1ll << 31), "moe_forward: bad T");
  HK_REQUIRE(num_experts >= 1 && num_experts <= kMaxExperts, "moe_forward: E=%d outside [1, %d]",
             num_experts, kMaxExperts);
  HK_REQUIRE(top_k >= 1 && top_k <= num_experts && top_k <= kMaxTopK, "moe_forward: bad top_k=%d", top_k);
  HK_REQUIRE(hidden > 0 && hidden % kBN == 0 && hidden <= kGroup * kMaxKBlocks,
             "moe_forward: hidden=%d must be a multiple of 256 and <= %d", hidden, kGroup * kMaxKBlocks);
  HK_REQUIRE(inter > 0 && inter % 128 == 0 && inter <= kGroup * kMaxKBlocks,
             "moe_forward: inter=%d must be a multiple of 128 and <= %d", inter, kGroup * kMaxKBlocks);
  // every operand of the grouped GEMMs is addressed by 32-bit buffer offsets:
  // checked here, before any kernel of the layer is launched
  HK_REQUIRE(2ll * inter * hidden < (1ll << 32), "moe_forward: expert weight too large (2*I*H must be < 2^32)");
  HK_REQUIRE(num_tokens * hidden < (1ll << 32) && num_tokens * top_k * inter < (1ll << 32),
             "moe_forward: T*H and T*k*I must be < 2^32 (32-bit buffer offsets)");
  if (num_tokens == 0) return HKMOE_OK;
  const bool block = scale_mode == HKMOE_SCALE_BLOCK;
  const MoeWorkspace need = carve(nullptr, num_tokens, num_experts, top_k, hidden, inter, scale_mode);
  if (workspace == nullptr || workspace_bytes < need.bytes)
    return fail(HKMOE_ERR_WORKSPACE, "moe_forward: workspace of %zu bytes needed, %zu given", need.bytes,
                workspace_bytes);
  HK_REQUIRE((reinterpret_cast<uintptr_t>(workspace) & 255) == 0, "moe_forward: workspace must be 256-byte aligned");
  const MoeWorkspace w = carve(static_cast<uint8_t*>(workspace), num_tokens, num_experts, top_k,
                               hidden, inter, scale_mode);
  const int64_t rows = num_tokens * top_k;
  auto s = static_cast<hipStream_t>(stream);
  NarrowPlan plan;
  const bool tuned = block && narrow_part_steps(hidden / kBK) && narrow_part_steps(inter / kBK);
  HK_TRY(plan_narrow({num_tokens, rows, num_experts, 3ll * inter * hidden, tuned, !block,
                      w_layout == HKMOE_W_PACKED, aux_ok && block}, s, &plan));
  return moe_enqueue(
      logits, w, num_tokens, num_experts, top_k, hidden, out, s, plan, [] { return HKMOE_OK; },
      // GEMM 1 reads token rows through perm; with block scales it writes the
      // requantised e4m3 intermediate and its 1x128 group scales directly
      [&](const NarrowPart& part, int32_t* ctr, hipStream_t st) {
        return grouped_gemm1_impl(x_q, x_scale, w.perm, top_k, num_tokens, w13, w13_scale, w.offsets, w.mtile_offsets,
                                  w.mtile_list, rows, num_experts, hidden, inter, scale_mode, w_layout,
                                  block ? HKMOE_E4M3 : HKMOE_BF16, block ? static_cast<void*>(w.hq) : w.h,
                                  block ? w.hs : w.amax, ctr, st, part);
      },
      [&] {
        if (block) return static_cast<int>(HKMOE_OK);
        t_role = HKMOE_TIMING_REQUANT;
        return hkmoe_requant(w.h, rows, inter, scale_mode, w.amax, w.hq, w.hs, s);
      },
      [&](const NarrowPart& part, int32_t* ctr, hipStream_t st) {
        return grouped_gemm2_impl(w.hq, w.hs, w2, w2_scale, w.offsets, w.mtile_offsets, w.mtile_list, rows,
                                  num_experts, hidden, inter, scale_mode, w_layout, w.y, ctr, st, part);
      });
}

int hkmoe_moe_forward(const void* x_q, const float* x_scale, const float* logits, const void* w13,
                      const float* w13_scale, const void* w2, const float* w2_scale,
                      int64_t num_tokens, int32_t num_experts, int32_t top_k, int32_t hidden,
                      int32_t inter, int scale_mode, int w_layout, void* out, void* workspace,
                      size_t workspace_bytes, hkmoe_stream_t stream) {
  return moe_forward_impl(x_q, x_scale, logits, w13, w13_scale, w2, w2_scale, num_tokens, num_experts, top_k,
                          hidden, inter, scale_mode, w_layout, out, workspace, workspace_bytes, stream, true);
}

// ---------------------------------------------------------------------------
// quantisers
// ---------------------------------------------------------------------------
int hkmoe_quant_group(const float* x, int64_t rows, int64_t cols, void* q, float* s,
                      hkmoe_stream_t stream) {
  HK_REQUIRE(rows == 0 || (x && q && s), "quant_group: null pointer");
  HK_REQUIRE(rows >= 0 && cols > 0 && cols % kGroup == 0, "quant_group: cols must be a multiple of 128");
  const int64_t groups = rows * (cols / kGroup);
  if (groups == 0) return HKMOE_OK;
  const int64_t grid = (groups + kQuantGroups - 1) / kQuantGroups;
  HK_REQUIRE(grid < (1ll << 31), "quant_group: too large");
  hipLaunchKernelGGL(quant_group_kernel, dim3(static_cast<unsigned>(grid)), dim3(256), 0,
                     static_cast<hipStream_t>(stream), x, groups, static_cast<uint8_t*>(q), s);
  return check_launch("quant_group_kernel");
}

int hkmoe_quant_block(const float* x, int64_t batch, int64_t rows, int64_t cols, void* q, float* s,
                      hkmoe_stream_t stream) {
  HK_REQUIRE(batch == 0 || (x && q && s), "quant_block: null pointer");
  HK_REQUIRE(batch >= 0 && rows > 0 && cols > 0 && rows % kGroup == 0 && cols % kGroup == 0,
             "quant_block: rows and cols must be multiples of 128");
  const int64_t blocks = batch * (rows / kGroup) * (cols / kGroup);
  if (blocks == 0) return HKMOE_OK;
  HK_REQUIRE(blocks < (1ll << 31), "quant_block: too large");
  hipLaunchKernelGGL(quant_block_kernel, dim3(static_cast<unsigned>(blocks)), dim3(256), 0,
                     static_cast<hipStream_t>(stream), x, rows, cols, static_cast<uint8_t*>(q), s);
  return check_launch("quant_block_kernel");
}

int hkmoe_quant_tensor(const float* x, int64_t rows, int64_t cols, void* q, float* s, float* amax_ws,
                       hkmoe_stream_t stream) {
  HK_REQUIRE(s && amax_ws && (rows == 0 || cols == 0 || (x && q)), "quant_tensor: null pointer");
  HK_REQUIRE(rows >= 0 && cols >= 0, "quant_tensor: bad shape");
  const int64_t n = rows * cols;
  auto st = static_cast<hipStream_t>(stream);
  // One launch instead of three while rereading the whole tensor per workgroup
  // costs less than two launches: 32x4096 takes 10.7 us a call (29 before).
  if (n <= kQuantSmall) {
    const int grid = static_cast<int>(std::max<int64_t>(1, (n + 4095) / 4096));
    hipLaunchKernelGGL(quant_tensor_small_kernel, dim3(grid), dim3(1024), 0, st, x, n, static_cast<uint8_t*>(q), s);
    return check_launch("quant_tensor_small_kernel");
  }
  hipLaunchKernelGGL(fill_f32_kernel, dim3(1), dim3(1), 0, st, amax_ws, 0.0f);
  HK_TRY(check_launch("fill_f32_kernel"));
  const int grid = static_cast<int>(std::min<int64_t>((n + 1023) / 1024, 4096));
  // at most two workgroups per CU: each ends in one atomic on the same word,
  // and they all end together (512 / 1024 / 2048 workgroups: 31 / 39 / 53 us for
  // the three launches at 4096x4096)
  const int agrid = static_cast<int>(std::min<int64_t>((n + 16383) / 16384, 512));
  hipLaunchKernelGGL(amax_kernel, dim3(agrid), dim3(256), 0, st, x, n, amax_ws);
  HK_TRY(check_launch("amax_kernel"));
  hipLaunchKernelGGL(quant_tensor_kernel, dim3(grid), dim3(256), 0, st, x, n, amax_ws,
                     static_cast<uint8_t*>(q), s);
  return check_launch("quant_tensor_kernel");
}

// ---------------------------------------------------------------------------
// MX (e8m0 1x32) operands and GEMM
// ---------------------------------------------------------------------------
int hkmoe_quant_mx(const float* x, int64_t rows, int64_t cols, void* q, void* s, hkmoe_stream_t stream) {
  HK_REQUIRE(rows == 0 || (x && q && s), "quant_mx: null pointer");
  HK_REQUIRE(rows >= 0 && cols > 0 && cols % 32 == 0, "quant_mx: cols=%lld must be a positive multiple of 32",
             (long long)cols);
  const int64_t blocks = rows * (cols / 32);
  if (blocks == 0) return HKMOE_OK;
  const bool small = blocks * 32 <= kMxSmall;
  const int64_t per = small ? 512 : 1024, grid = (blocks * 8 + per - 1) / per;  // quads per workgroup
  HK_REQUIRE(grid < (1ll << 31), "quant_mx: too large");
  hipLaunchKernelGGL((small ? quant_mx_kernel<2, false> : quant_mx_kernel<4, true>), dim3(static_cast<unsigned>(grid)),
                     dim3(256), 0, static_cast<hipStream_t>(stream), x, blocks, static_cast<uint8_t*>(q),
                     static_cast<uint8_t*>(s));
  return check_launch("quant_mx_kernel");
}

int hkmoe_mx_pack_scales(const void* s, int64_t rows, int64_t cols, void* packed, hkmoe_stream_t stream) {
  HK_REQUIRE(rows == 0 || (s && packed), "mx_pack_scales: null pointer");
  HK_REQUIRE(rows >= 0 && cols > 0 && cols % kBK == 0,
             "mx_pack_scales: cols=%lld must be a positive multiple of 128", (long long)cols);
  const int64_t rows64 = (rows + 63) / 64 * 64;
  const int64_t words = (cols / kBK) * rows64;
  if (words == 0) return HKMOE_OK;
  const int grid = static_cast<int>(std::min<int64_t>((words + 255) / 256, 8192));
  hipLaunchKernelGGL(mx_pack_scales_kernel, dim3(grid), dim3(256), 0, static_cast<hipStream_t>(stream),
                     static_cast<const uint8_t*>(s), rows, cols / 32, rows64, static_cast<uint32_t*>(packed),
                     words);
  return check_launch("mx_pack_scales_kernel");
}

int hkmoe_gemm_mx(const void* a, const void* a_scale, const void* b, const void* b_scale, void* c, int64_t m,
                  int64_t n, int64_t k, int out_dtype, hkmoe_stream_t stream) {
  HK_REQUIRE(b && b_scale && (m == 0 || (a && a_scale && c)), "gemm_mx: null pointer");
  HK_REQUIRE(m >= 0 && n > 0 && k > 0, "gemm_mx: bad shape M=%lld N=%lld K=%lld", (long long)m, (long long)n,
             (long long)k);
  HK_REQUIRE(k % kBK == 0, "gemm_mx: K=%lld must be a multiple of 128", (long long)k);
  HK_REQUIRE(n % kBN == 0, "gemm_mx: N=%lld must be a multiple of 256", (long long)n);
  const int64_t m64 = (m + 63) / 64 * 64;
  HK_REQUIRE(k <= (1 << 20) && n * k < (1ll << 32) && m * k < (1ll << 32) && m < (1ll << 31) &&
                 m64 * (k / 32) < (1ll << 32) && n * (k / 32) < (1ll << 32),
             "gemm_mx: operand too large for 32-bit buffer offsets (M*K and N*K must be < 2^32)");
  HK_REQUIRE(out_dtype == HKMOE_BF16 || out_dtype == HKMOE_F32, "gemm_mx: bad out_dtype %d", out_dtype);
  if (m == 0) return HKMOE_OK;
  return launch_dense<true>(a, b, c, m, n, k, static_cast<const float*>(a_scale),
                            static_cast<const float*>(b_scale), out_dtype, static_cast<hipStream_t>(stream));
}

int64_t hkmoe_mx_words_per_step(int64_t rows, int32_t num_experts) {
  return rows < 0 || num_experts < 1 ? 0 : mx_words_per_step(rows, num_experts);
}

int hkmoe_mx_pack_weight_scales(const void* s, int64_t num_experts, int64_t n, int64_t k, int32_t gate_up,
                                void* words, hkmoe_stream_t stream) {
  HK_REQUIRE(s && words, "mx_pack_weight_scales: null pointer");
  HK_REQUIRE(num_experts >= 0 && n > 0 && k > 0 && n % kBN == 0 && k % kBK == 0,
             "mx_pack_weight_scales: N=%lld must be a multiple of 256 and K=%lld of 128", (long long)n,
             (long long)k);
  HK_REQUIRE(gate_up == 0 || (gate_up > 0 && 2ll * gate_up == n && gate_up % 128 == 0),
             "mx_pack_weight_scales: gate_up=%d must be 0 or N/2 (a multiple of 128)", gate_up);
  HK_REQUIRE(k <= (1 << 20), "mx_pack_weight_scales: K too large");
  const int64_t n_words = num_experts * n * (k / 128);
  if (n_words == 0) return HKMOE_OK;
  const int grid = static_cast<int>(std::min<int64_t>((n_words + 255) / 256, 8192));
  hipLaunchKernelGGL(mx_pack_weight_words_kernel, dim3(grid), dim3(256), 0, static_cast<hipStream_t>(stream),
                     static_cast<const uint8_t*>(s), n, static_cast<int>(k), gate_up,
                     static_cast<uint32_t*>(words), n_words);
  return check_launch("mx_pack_weight_words_kernel");
}

int hkmoe_mx_gather_scales(const void* s, int64_t x_rows, int32_t k, const int32_t* gather, int32_t gather_div,
                           const int32_t* offsets, const int32_t* mtile_offsets, int32_t num_experts,
                           int64_t rows, void* words, hkmoe_stream_t stream) {
  HK_REQUIRE(offsets && mtile_offsets, "mx_gather_scales: null pointer");
  HK_REQUIRE(rows == 0 || (s && words), "mx_gather_scales: null pointer");
  HK_REQUIRE(k > 0 && k % kBK == 0 && k / 32 <= kMxGatherMaxKb,
             "mx_gather_scales: K=%d must be a multiple of 128 and <= %d", k, 32 * kMxGatherMaxKb);
  HK_REQUIRE(num_experts >= 1 && num_experts <= kMaxExperts, "mx_gather_scales: bad E=%d", num_experts);
  HK_REQUIRE(rows >= 0 && rows < (1ll << 31) && x_rows >= 0, "mx_gather_scales: bad rows");
  HK_REQUIRE(gather != nullptr ? gather_div >= 1 : x_rows >= rows, "mx_gather_scales: bad gather");
  HK_REQUIRE((reinterpret_cast<uintptr_t>(s) & 3) == 0, "mx_gather_scales: exponents must be 4-byte aligned");
  if (rows == 0) return HKMOE_OK;
  const int64_t ws = mx_words_per_step(rows, num_experts);
  // one workgroup per M tile (ws / 256 bounds their number), the tile's exponent
  // rows in LDS
  static bool attr_set[kMaxDevices] = {false};
  int dev = 0;
  (void)hipGetDevice(&dev);
  if (dev >= 0 && dev < kMaxDevices && !attr_set[dev]) {
    const hipError_t err = hipFuncSetAttribute(reinterpret_cast<const void*>(mx_gather_words_kernel),
                                               hipFuncAttributeMaxDynamicSharedMemorySize, 256 * kMxGatherMaxKb);
    if (err != hipSuccess) return fail(HKMOE_ERR_HIP, "hipFuncSetAttribute: %s", hipGetErrorString(err));
    attr_set[dev] = true;
  }
  const int grid = static_cast<int>(std::min<int64_t>(ws / 256, 4096));
  hk_launch(mx_gather_words_kernel, dim3(grid), dim3(256), static_cast<uint32_t>(256 * (k / 32)),
            static_cast<hipStream_t>(stream),
                     static_cast<const uint8_t*>(s), k, gather, gather ? gather_div : 1, offsets, mtile_offsets,
                     num_experts, ws, static_cast<uint32_t*>(words));
  return check_launch("mx_gather_words_kernel");
}

// x_words: the tile-aligned words, or for the narrow kernel (part.active > 0)
// the rows' own exponent bytes [x_rows, H/32].
static int grouped_gemm1_mx_impl(const void* x, const void* x_words, const int32_t* gather, int32_t gather_div,
                                 int64_t x_rows, const void* w13, const void* w13_words, const int32_t* offsets,
                                 const int32_t* mtile_offsets, const int32_t* mtile_list, int64_t rows,
                                 int32_t num_experts, int32_t hidden, int32_t inter, int w_layout, int out_format,
                                 void* h, void* h_words, int32_t* tile_counters, hkmoe_stream_t stream,
                                 const NarrowPart& part) {
  HK_REQUIRE(w13 && w13_words && offsets && mtile_offsets, "grouped_gemm1_mx: null pointer");
  HK_REQUIRE(rows == 0 || (x && x_words && h), "grouped_gemm1_mx: null pointer");
  HK_REQUIRE(num_experts >= 1 && num_experts <= kMaxExperts, "grouped_gemm1_mx: bad E=%d", num_experts);
  HK_REQUIRE(hidden > 0 && hidden % kGroup == 0 && hidden <= kGroup * kMaxKBlocks,
             "grouped_gemm1_mx: hidden=%d must be a multiple of 128 and <= %d", hidden, kGroup * kMaxKBlocks);
  HK_REQUIRE(inter > 0 && inter % 128 == 0, "grouped_gemm1_mx: inter=%d must be a multiple of 128", inter);
  HK_REQUIRE(rows >= 0 && rows < (1ll << 31), "grouped_gemm1_mx: bad rows");
  HK_REQUIRE(x_rows >= (rows > 0 ? 1 : 0) && x_rows * hidden < (1ll << 32), "grouped_gemm1_mx: x_rows=%lld out of range",
             (long long)x_rows);
  HK_REQUIRE(gather == nullptr || gather_div >= 1, "grouped_gemm1_mx: gather_div must be >= 1");
  HK_REQUIRE(gather != nullptr || x_rows >= rows, "grouped_gemm1_mx: x has fewer rows than rows");
  HK_REQUIRE(2ll * inter * hidden < (1ll << 32), "grouped_gemm1_mx: expert weight too large");
  HK_REQUIRE(w_layout == HKMOE_W_ROWS || w_layout == HKMOE_W_PACKED, "grouped_gemm1_mx: bad w_layout %d",
             w_layout);
  HK_REQUIRE(out_format == HKMOE_BF16 || out_format == HKMOE_E4M3, "grouped_gemm1_mx: bad out_format %d",
             out_format);
  HK_REQUIRE(out_format != HKMOE_E4M3 || h_words != nullptr, "grouped_gemm1_mx: e4m3 output needs h_words");
  if (rows == 0) return HKMOE_OK;
  const int64_t ws = mx_words_per_step(rows, num_experts);
  HK_REQUIRE(ws * (std::max(hidden, inter) / kBK) * 4 < (1ll << 32), "grouped_gemm1_mx: too many rows");
  GemmParams p{};
  p.a = static_cast<const uint8_t*>(x);
  p.a_gather = gather;
  p.gather_div = gather ? gather_div : 1;
  p.b = static_cast<const uint8_t*>(w13);
  p.c = h;
  p.a_scale = static_cast<const float*>(x_words);
  p.b_scale = static_cast<const float*>(w13_words);
  p.c_scale = static_cast<float*>(h_words);
  p.offsets = offsets;
  p.mtile_offsets = mtile_offsets;
  p.rows = rows;
  p.a_rows = x_rows;
  p.as_rs = ws;
  p.cs_rs = ws;
  p.num_experts = num_experts;
  p.K = hidden;
  p.nb = 2 * inter;
  p.n_out = inter;
  p.n_tiles = inter / 128;
  p.b_packed = w_layout == HKMOE_W_PACKED;
  p.mtile_list = mtile_list;
  p.blk_m_log2 = block_m_log2(1);  // 2 x 16 tile blocks by default
  p.tile_ctr = tile_counters;
  p.narrow_cnt = part.count;
  p.yield_from = part.yield_from;
  p.narrow_active = part.active;
  auto st = static_cast<hipStream_t>(stream);
  if (part.active > 0) {
    p.as_rs = hidden / kGroup;  // one dword of exponents per row and K step, row-major
    p.as_ks = 1;
    return launch_narrow<Epi::kSiluMx, Scale::kMX>(p, st, part);
  }
  const int grid = part.yield_from < 0 ? part.grid : 0;
  return out_format == HKMOE_E4M3 ? launch_gemm<Epi::kSiluMx, Scale::kMX>(p, st, grid)
                                  : launch_gemm<Epi::kSiluBf16, Scale::kMX>(p, st, grid);
}

int hkmoe_grouped_gemm1_mx(const void* x, const void* x_words, const int32_t* gather, int32_t gather_div,
                           int64_t x_rows, const void* w13, const void* w13_words, const int32_t* offsets,
                           const int32_t* mtile_offsets, const int32_t* mtile_list, int64_t rows,
                           int32_t num_experts, int32_t hidden, int32_t inter, int w_layout, int out_format,
                           void* h, void* h_words, int32_t* tile_counters, hkmoe_stream_t stream) {
  return grouped_gemm1_mx_impl(x, x_words, gather, gather_div, x_rows, w13, w13_words, offsets, mtile_offsets,
                               mtile_list, rows, num_experts, hidden, inter, w_layout, out_format, h, h_words,
                               tile_counters, stream, NarrowPart{});
}

static int grouped_gemm2_mx_impl(const void* hq, const void* hq_words, const void* w2, const void* w2_words,
                                 const int32_t* offsets, const int32_t* mtile_offsets, const int32_t* mtile_list,
                                 int64_t rows, int32_t num_experts, int32_t hidden, int32_t inter, int w_layout,
                                 void* y, int32_t* tile_counters, hkmoe_stream_t stream, const NarrowPart& part) {
  HK_REQUIRE(w2 && w2_words && offsets && mtile_offsets, "grouped_gemm2_mx: null pointer");
  HK_REQUIRE(rows == 0 || (hq && hq_words && y), "grouped_gemm2_mx: null pointer");
  HK_REQUIRE(num_experts >= 1 && num_experts <= kMaxExperts, "grouped_gemm2_mx: bad E=%d", num_experts);
  HK_REQUIRE(hidden > 0 && hidden % kBN == 0, "grouped_gemm2_mx: hidden=%d must be a multiple of 256", hidden);
  HK_REQUIRE(inter > 0 && inter % kGroup == 0 && inter <= kGroup * kMaxKBlocks,
             "grouped_gemm2_mx: inter=%d must be a multiple of 128 and <= %d", inter, kGroup * kMaxKBlocks);
  HK_REQUIRE(rows >= 0 && rows < (1ll << 31), "grouped_gemm2_mx: bad rows");
  HK_REQUIRE(rows * inter < (1ll << 32), "grouped_gemm2_mx: rows*inter must be < 2^32 (32-bit buffer offsets into hq)");
  HK_REQUIRE(static_cast<int64_t>(hidden) * inter < (1ll << 32), "grouped_gemm2_mx: expert weight too large");
  HK_REQUIRE(w_layout == HKMOE_W_ROWS || w_layout == HKMOE_W_PACKED, "grouped_gemm2_mx: bad w_layout %d",
             w_layout);
  if (rows == 0) return HKMOE_OK;
  const int64_t ws = mx_words_per_step(rows, num_experts);
  HK_REQUIRE(ws * (inter / kBK) * 4 < (1ll << 32), "grouped_gemm2_mx: too many rows");
  GemmParams p{};
  p.a = static_cast<const uint8_t*>(hq);
  p.b = static_cast<const uint8_t*>(w2);
  p.c = y;
  p.a_scale = static_cast<const float*>(hq_words);
  p.b_scale = static_cast<const float*>(w2_words);
  p.offsets = offsets;
  p.mtile_offsets = mtile_offsets;
  p.rows = rows;
  p.a_rows = rows;
  p.as_rs = ws;
  p.num_experts = num_experts;
  p.K = inter;
  p.nb = hidden;
  p.n_out = hidden;
  p.n_tiles = hidden / kBN;
  p.b_packed = w_layout == HKMOE_W_PACKED;
  p.mtile_list = mtile_list;
  p.blk_m_log2 = block_m_log2(2);
  p.tile_ctr = tile_counters;
  p.narrow_cnt = part.count;
  p.yield_from = part.yield_from;
  p.narrow_active = part.active;
  auto st = static_cast<hipStream_t>(stream);
  if (part.active > 0) {
    p.as_rs = 1;  // one dword of exponents per row and K step, in the M tile's words
    p.as_ks = ws;
    return launch_narrow<Epi::kStoreBf16, Scale::kMX>(p, st, part);
  }
  return launch_gemm<Epi::kStoreBf16, Scale::kMX>(p, st);
}

int hkmoe_grouped_gemm2_mx(const void* hq, const void* hq_words, const void* w2, const void* w2_words,
                           const int32_t* offsets, const int32_t* mtile_offsets, const int32_t* mtile_list,
                           int64_t rows, int32_t num_experts, int32_t hidden, int32_t inter, int w_layout,
                           void* y, int32_t* tile_counters, hkmoe_stream_t stream) {
  return grouped_gemm2_mx_impl(hq, hq_words, w2, w2_words, offsets, mtile_offsets, mtile_list, rows, num_experts,
                               hidden, inter, w_layout, y, tile_counters, stream, NarrowPart{});
}

int hkmoe_moe_forward_mx(const void* x_q, const void* x_e8m0, const float* logits, const void* w13,
                         const void* w13_words, const void* w2, const void* w2_words, int64_t num_tokens,
                         int32_t num_experts, int32_t top_k, int32_t hidden, int32_t inter, int w_layout,
                         void* out, void* workspace, size_t workspace_bytes, hkmoe_stream_t stream) {
  // with no tokens the activations, the output and the workspace may be empty (null)
  HK_REQUIRE(w13 && w13_words && w2 && w2_words, "moe_forward_mx: null pointer");
  HK_REQUIRE(num_tokens == 0 || (x_q && x_e8m0 && logits && out), "moe_forward_mx: null pointer");
  HK_REQUIRE(w_layout == HKMOE_W_ROWS || w_layout == HKMOE_W_PACKED, "moe_forward_mx: bad w_layout %d",
             w_layout);
  HK_REQUIRE(num_tokens >= 0 && num_tokens * top_k < (1ll << 31), "moe_forward_mx: bad T");
  HK_REQUIRE(num_experts >= 1 && num_experts <= kMaxExperts, "moe_forward_mx: E=%d outside [1, %d]",
             num_experts, kMaxExperts);
  HK_REQUIRE(top_k >= 1 && top_k <= num_experts && top_k <= kMaxTopK, "moe_forward_mx: bad top_k=%d", top_k);
  HK_REQUIRE(hidden > 0 && hidden % kBN == 0 && hidden <= kGroup * kMaxKBlocks,
             "moe_forward_mx: hidden=%d must be a multiple of 256 and <= %d", hidden, kGroup * kMaxKBlocks);
  HK_REQUIRE(inter > 0 && inter % 128 == 0 && inter <= kGroup * kMaxKBlocks,
             "moe_forward_mx: inter=%d must be a multiple of 128 and <= %d", inter, kGroup * kMaxKBlocks);
  HK_REQUIRE(2ll * inter * hidden < (1ll << 32), "moe_forward_mx: expert weight too large (2*I*H must be < 2^32)");
  HK_REQUIRE(num_tokens * hidden < (1ll << 32) && num_tokens * top_k * inter < (1ll << 32),
             "moe_forward_mx: T*H and T*k*I must be < 2^32 (32-bit buffer offsets)");
  if (num_tokens == 0) return HKMOE_OK;
  // both the word gather and the narrow kernel read a row's exponents as dwords
  HK_REQUIRE((reinterpret_cast<uintptr_t>(x_e8m0) & 3) == 0, "mx_gather_scales: exponents must be 4-byte aligned");
  const MoeWorkspace need = carve(nullptr, num_tokens, num_experts, top_k, hidden, inter, HKMOE_SCALE_MX);
  if (workspace == nullptr || workspace_bytes < need.bytes)
    return fail(HKMOE_ERR_WORKSPACE, "moe_forward_mx: workspace of %zu bytes needed, %zu given", need.bytes,
                workspace_bytes);
  HK_REQUIRE((reinterpret_cast<uintptr_t>(workspace) & 255) == 0, "moe_forward_mx: workspace must be 256-byte aligned");
  const MoeWorkspace w = carve(static_cast<uint8_t*>(workspace), num_tokens, num_experts, top_k, hidden,
                               inter, HKMOE_SCALE_MX);
  const int64_t rows = num_tokens * top_k;
  auto s = static_cast<hipStream_t>(stream);
  NarrowPlan plan;
  HK_TRY(plan_narrow({num_tokens, rows, num_experts, 3ll * inter * hidden, false, false,
                      w_layout == HKMOE_W_PACKED, true}, s, &plan));
  return moe_enqueue(
      logits, w, num_tokens, num_experts, top_k, hidden, out, s, plan,
      // token exponents -> tile-aligned words in expert order (x rows stay in place)
      [&] {
        t_role = HKMOE_TIMING_MX_WORDS;
        return hkmoe_mx_gather_scales(x_e8m0, num_tokens, hidden, w.perm, top_k, w.offsets, w.mtile_offsets,
                                      num_experts, rows, w.xw, s);
      },
      [&](const NarrowPart& part, int32_t* ctr, hipStream_t st) {
        return grouped_gemm1_mx_impl(x_q, part.active > 0 ? x_e8m0 : w.xw, w.perm, top_k, num_tokens, w13, w13_words,
                                     w.offsets, w.mtile_offsets, w.mtile_list, rows, num_experts, hidden, inter,
                                     w_layout, HKMOE_E4M3, w.hq, w.hs, ctr, st, part);
      },
      [] { return HKMOE_OK; },
      [&](const NarrowPart& part, int32_t* ctr, hipStream_t st) {
        return grouped_gemm2_mx_impl(w.hq, w.hs, w2, w2_words, w.offsets, w.mtile_offsets, w.mtile_list, rows,
                                     num_experts, hidden, inter, w_layout, w.y, ctr, st, part);
      });
}

// ---------------------------------------------------------------------------
// kernel timing of the layer entry points
// ---------------------------------------------------------------------------
int hkmoe_kernel_timing(int32_t calls) {
  HK_REQUIRE(calls >= 0 && calls <= 4096, "kernel_timing: calls=%d outside [0, 4096]", calls);
  std::lock_guard<std::mutex> g(g_timing_mu);
  for (hipEvent_t e : g_timing.ev) (void)hipEventDestroy(e);
  g_timing = KernelTiming{};
  if (calls == 0) return HKMOE_OK;
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess) return fail(HKMOE_ERR_HIP, "kernel_timing: no device");
  const size_t n = static_cast<size_t>(calls) * HKMOE_TIMING_ROLES * 2;
  g_timing.ev.reserve(n);
  for (size_t i = 0; i < n; ++i) {
    hipEvent_t e = nullptr;
    if (hipEventCreate(&e) != hipSuccess) {
      for (hipEvent_t x : g_timing.ev) (void)hipEventDestroy(x);
      g_timing = KernelTiming{};
      return fail(HKMOE_ERR_HIP, "kernel_timing: hipEventCreate failed");
    }
    g_timing.ev.push_back(e);
  }
  g_timing.used.assign(static_cast<size_t>(calls) * HKMOE_TIMING_ROLES, 0);
  g_timing.first.assign(calls, -1);
  g_timing.last.assign(calls, -1);
  g_timing.device = dev;
  g_timing.calls = calls;
  return HKMOE_OK;
}

int hkmoe_kernel_timing_read(int32_t set, float* begin_ms, float* end_ms, int32_t n) {
  HK_REQUIRE(begin_ms && end_ms && n >= HKMOE_TIMING_ROLES, "kernel_timing_read: need %d floats per array",
             HKMOE_TIMING_ROLES);
  std::lock_guard<std::mutex> g(g_timing_mu);
  HK_REQUIRE(set >= 0 && set < g_timing.calls, "kernel_timing_read: set=%d outside [0, %d)", set,
             g_timing.calls);
  const size_t base = static_cast<size_t>(set) * HKMOE_TIMING_ROLES;
  const int f = g_timing.first[set];
  for (int r = 0; r < HKMOE_TIMING_ROLES; ++r) {
    begin_ms[r] = end_ms[r] = -1.0f;
    if (f < 0 || !g_timing.used[base + r]) continue;
    const hipEvent_t t0 = g_timing.ev[2 * (base + f)];
    if (hipEventElapsedTime(&begin_ms[r], t0, g_timing.ev[2 * (base + r)]) != hipSuccess ||
        hipEventElapsedTime(&end_ms[r], t0, g_timing.ev[2 * (base + r) + 1]) != hipSuccess)
      return fail(HKMOE_ERR_HIP, "kernel_timing_read: events of set %d not complete", set);
  }
  return HKMOE_OK;
}

// ---------------------------------------------------------------------------
// allocation-free layer (hkmoe_moe_forward_noalloc)
// ---------------------------------------------------------------------------
int hkmoe_moe_forward_noalloc(const void* x_q, const float* x_scale, const float* logits, const void* w13,
                              const float* w13_scale, const void* w2, const float* w2_scale,
                              int64_t num_tokens, int32_t num_experts, int32_t top_k, int32_t hidden,
                              int32_t inter, int scale_mode, int w_layout, void* out, hkmoe_stream_t stream) {
  HK_REQUIRE(num_tokens >= 0 && num_experts >= 1 && top_k >= 1 && hidden > 0 && inter > 0,
             "moe_forward_noalloc: bad shape");
  HK_REQUIRE(scale_mode == HKMOE_SCALE_TENSOR || scale_mode == HKMOE_SCALE_BLOCK,
             "moe_forward_noalloc: bad scale_mode %d", scale_mode);
  const size_t need = carve(nullptr, num_tokens, num_experts, top_k, hidden, inter, scale_mode).bytes;
  if (need > kScratchBytes)
    return fail(HKMOE_ERR_WORKSPACE,
                "moe_forward_noalloc: the layer needs %zu bytes of workspace, the library's per-device scratch "
                "holds %zu (HKMOE_NOALLOC_SCRATCH_BYTES); pass a workspace to hkmoe_moe_forward instead",
                need, kScratchBytes);
  if (num_tokens == 0) return moe_forward_impl(x_q, x_scale, logits, w13, w13_scale, w2, w2_scale, num_tokens,
                                               num_experts, top_k, hidden, inter, scale_mode, w_layout, out,
                                               nullptr, 0, stream, false);
  void* ws = nullptr;
  HK_TRY(scratch_ptr(&ws));
  return moe_forward_impl(x_q, x_scale, logits, w13, w13_scale, w2, w2_scale, num_tokens, num_experts, top_k,
                          hidden, inter, scale_mode, w_layout, out, ws, kScratchBytes, stream, false);
}
}  // extern "C"
