// The attention kernel with one workgroup per 16-row window, and its launchers, as templates:
// f3s_attention.hip builds them with 32-bit row offsets in the K / V gathers (arrays below
// 4 GiB), f3s_attention_wide.hip with 64-bit offsets (the reference indexes rows with int64_t,
// src/F3S_kernel.cu:1422-1423); two translation units, because keeping both address forms in one
// kernel costs the common one 17 vector registers.
//
// Replaces the reference kernels f3sKernel1tb1rw / ...Scheduled / ...ScheduledPermutedQKV
// [ScaleQK], f2sKernel1tb1rw and f3sKernel1tb1tcb (src/F3S_kernel.cu:997-1175, 1371-1800,
// 1999-2182, 2186-2327, 677-877) and their launchers (src/F3S_kernel.cu:325-458, 581-671).
//
// A workgroup of four waves owns one window. The window's TC blocks are cut into four contiguous
// runs, one per wave; a wave walks its run with the shared pair pipeline (f3s_pair_pipeline.h:
// K/V rows gathered straight into the wave's LDS ring, scores and outputs in MFMA accumulators,
// running (m, l, O) in registers), and one LDS merge per window combines the four partial
// results (log-sum-exp) instead of the reference's three block barriers per iteration.
#pragma once
#include <stdlib.h>
#include <string.h>

#include "f3s_common.h"
#include "f3s_pair_pipeline.h"

namespace f3s {
namespace window {

using pipe::float4v;
using pipe::kLog2e;

// Waves and ring stages of a workgroup. Bound by the latency of the gathers and of the chain of loads
// in front of the first one, so what counts is the pairs in flight on a CU, and how long the longest
// window takes alone.
//   TEAM_SHORT  one workgroup for every window: four waves of one stage. Four workgroups per CU at
//               D = 32, three at D = 64 (two stages allow two), two up to D = 128, one above.
//   TEAM_PAIRS  the same with two stages at D = 32, where they cost no workgroup (see two_stages).
// Graphs of short windows take f3s_fwd_mixed_kernel instead (f3s_attention_mixed.hip).
enum Team { TEAM_SHORT, TEAM_PAIRS };
constexpr int kTeamWaves = 4;  // MergedRows takes four
constexpr int team_stages(Team t) { return t == TEAM_SHORT ? 1 : 2; }
constexpr int waves_per_simd(int d) { return d > 128 ? 1 : d > 64 ? 2 : d > 32 ? 3 : 4; }

// Whether TEAM_PAIRS takes the windows rather than TEAM_SHORT (nTcb16: blocks of 16 columns). At D = 32
// four workgroups fit a CU either way, so the second stage only has to pay for its longer loop.
// One -> two stages in us, heavy-first order, one head unless stated. It pays
// - where blocks are few and the longest window of a skewed graph decides. 17 to 30 blocks a window:
//   R-MAT 65 521 nodes 38.8 -> 32.9, 3 heads 65.1 -> 64.5, 169 343 nodes 71.9 -> 61.1, 3 heads 167 -> 172,
//   600 000 nodes 268 -> 273; 38 to 57: R-MAT 100 000 nodes 79.1 -> 66.9, 200 000 nodes 146 -> 125; 81 to 90:
//   30 000 nodes 32.1 -> 28.9; uniform and community graphs of 5 to 21: within 2 %, with 3 and 5 heads 0 to
//   5 % faster.
// - where windows are long, many, and the rows come from beyond the L2s (K + V of 20 MB): 100 000 nodes,
//   406 blocks, 3 heads 2463 -> 2136, 5 heads 4628 -> 4441; 35 000, 294, 5 heads 820 -> 749; 140 000, 274, 3
//   heads 2211 -> 2133, 5 heads 4110 -> 4259; 180 000, 408 1348 -> 1328, 3 heads 4920 -> 4723, 5 heads 10 070 ->
//   10 170; 233 000, 448 2155 -> 2068, but 188 with 3 heads 2638 -> 2685, 5 heads 4957 -> 5282.
// In between all CUs are busy to the end, mostly with rows from the L2s: 50 000 nodes, 114 61.3 -> 62.9, 3
// heads 215 -> 231, 5 heads 420 -> 449; 148 77.2 -> 80.4, 3 heads 292 -> 315; 30 000, 329 90.1 -> 92.7, 3 heads
// 308 -> 326 (5 heads 736 -> 688); 100 000, 121 164 -> 174, 3 heads 569 -> 607; 233 000, 188 881 -> 902; R-MAT
// 100 000, 39, 3 heads 147 -> 150, 200 000, 40, 3 heads 345 -> 369.
// (Even numbers of heads come here only where there is little to do: pairs_pay.)
// At D = 64 a second stage costs the third workgroup: windows of 160 to 390 blocks 0 to 14 % slower, up
// to 2 % faster on 100 000 nodes and more; R-MAT of 10 blocks a window up to 25 % slower (169 343 nodes
// 69 -> 85), uniform graphs 10 to 24 %. Against that, R-MAT of 20 to 29 blocks and up to 100 000 nodes
// would gain (65 521 nodes 53.6 -> 47.7 and 65.2 -> 54.0), but a less skewed graph of the same size and
// block count loses (40 000 nodes 29.8 -> 32.4), and sizes do not tell the two apart.
inline bool two_stages(int d, int64_t nTcb16, int heads, int N) {
  if (d > 32) return false;
  const int64_t nRW = ((int64_t)N + kWinRows - 1) / kWinRows;
  if (nTcb16 * heads < 96 * nRW) return true;
  return nRW >= 2048 && nTcb16 >= 160 * nRW && nTcb16 * heads >= 400 * nRW &&
         (int64_t)N * d * heads * 4 >= (int64_t)20 << 20;
}

// LDS of a workgroup: its waves' rings
constexpr size_t team_lds(Team t, int d) {
  return (size_t)kTeamWaves * (team_stages(t) * 128 * d + 2 * 768);
}

// Constant-rate (100 MHz) timestamp shared by all CUs, and an id of the CU this wave runs on:
// XCC id in bits 8.., {SE, SH, CU} of HW_ID in bits 0..7. Used only by the timed variant, which
// replaces the reference's %globaltimer / %smid reads (src/F3S_kernel.cu:30-40).
__device__ __forceinline__ unsigned long long realtime_ticks() {
  return __builtin_amdgcn_s_memrealtime();
}
__device__ __forceinline__ unsigned cu_key() {
  unsigned hw, xcc;
  asm volatile("s_getreg_b32 %0, hwreg(HW_REG_HW_ID)" : "=s"(hw));
  asm volatile("s_getreg_b32 %0, hwreg(HW_REG_XCC_ID)" : "=s"(xcc));
  return ((xcc & 0xFu) << 8) | ((hw >> 8) & 0xFFu);
}

// HEADS = false: Q/K/V are [N, D] contiguous, one workgroup per window (blockIdx.x = position in
// the window order). HEADS = true: Q/K/V are [N, nHeads, D] with a row pitch of ldIn elements,
// out is [N, nHeads * D] with a row pitch of ldOut floats. Workgroup b runs on XCD b % 8; the XCDs are
// dealt groups of heads (split_heads: of at least a line of a row) and, 8 / headGroups of them to a
// group, the positions of the order, the heads of a position one after the other: an XCD gathers one
// group's part of the rows, and whole lines of it. With blockIdx.x = position * nHeads + head the two
// heads of a line came from two XCDs, each of which fetched all of it (bf16, 200 000 nodes, 48 blocks a
// window, 4 x 32: 823 -> 472 us; R-MAT of 1 000 000 nodes and 25 blocks, 2 x 32: 1203 -> 836 us; 40 000
// nodes, 19 blocks, 8 x 32: 111 -> 100 us). 1, 2, 4 and 8 heads of 64 and more come out the same either
// way; other numbers gain where an XCD's share of the rows shrinks and lose nowhere (graphs of 20 000 to
// 160 000 nodes and 22 to 92 blocks a window: 3, 5 and 7 heads of 64 0 to 4 %, 12 of 64 2 to 7 %, 16 of 64
// and 3 of 128 0 to 2 %, 12 of 128 4 to 7 %, 6 of 96 12 to 22 %).
// W8 = true: the structure comes from preprocessing with 8-column blocks (the reference's
// 1tb1tcb path, src/F3S_kernel.cu:677-877). Column ids and bitmap words of two consecutive 16x8
// blocks are laid out exactly like one 16x16 block, so the same pipeline runs over four 16x8
// blocks per step; rowWindowOffset then counts 16x8 blocks, a window may end in the middle of a
// step, and sddmm (if not null) receives the masked, unscaled scores, row-major 16x8 per block
// (saveSddmmResult, src/F3S_kernel.cu:99-115).
// PERSIST = true (single head, 16x16 blocks, not timed): the grid is as many workgroups as fit the
// GPU at once; a workgroup starts at position blockIdx.x of the window order and draws every
// further position from a device-wide cursor (the draw for the next window is in flight while the
// current one is computed), so the order is served first come, first served without relying on
// the order in which the hardware starts workgroups. The cursor is put back to zero by a
// one-thread kernel in front of every launch of this form (a launch that was cut short must not
// leave it behind); launches of this form must not overlap on one device.
static __device__ int g_windowCursor = 0;

template <int UNUSED = 0>
__global__ void reset_window_cursor_kernel() {
  g_windowCursor = 0;
}

// WIDE: 64-bit row offsets in the K / V gathers.
// NH = 2: D = 64 stands for two heads of 32; nHeads and headGroups count such pairs.
template <typename ET, int D, Team TEAM, bool SOFTMAX, bool CLOCKED, bool HEADS, bool W8,
          bool WIDE, bool PERSIST = false, int NH = 1>
__global__ __launch_bounds__(kTeamWaves * 64)
__attribute__((amdgpu_waves_per_eu(waves_per_simd(D), waves_per_simd(D)))) void
f3s_fwd_kernel(
    const int32_t* __restrict__ rowWindowOffset, const int32_t* __restrict__ windowOrder,
    const int32_t* __restrict__ sparseAToXidx, const uint8_t* __restrict__ bitmapBytes, int N,
    int nRW, int64_t nTcb, const ET* __restrict__ Q, const ET* __restrict__ K,
    const ET* __restrict__ V, float scaleLog2, float* __restrict__ out,
    unsigned long long* __restrict__ cuTimer, int nHeads, int headGroups, int ldIn, int ldOut,
    float* __restrict__ sddmm) {
  constexpr int NWAVES = kTeamWaves;
  constexpr int WAVE_BYTES = pipe::Geo<D, team_stages(TEAM)>::WAVE_BYTES;
  static_assert(team_lds(TEAM, D) == (size_t)NWAVES * WAVE_BYTES, "what the launch asks for");
  typedef pipe::PairPipeline<ET, D, SOFTMAX, HEADS, W8, team_stages(TEAM), WIDE, NH> Pipe;
  constexpr int BPS = W8 ? 4 : 2;  // blocks of the structure per pipeline step
  extern __shared__ __align__(1024) unsigned char smem[];
  unsigned long long tBegin = 0;
  if constexpr (CLOCKED) tBegin = realtime_ticks();

  static_assert(!PERSIST || (!CLOCKED && !HEADS && !W8), "the persistent form is single-head");
  __shared__ int sNextPos[2];
  int pos = (int)blockIdx.x, head = 0;
  if constexpr (HEADS) {
    const unsigned perGroup = (unsigned)nHeads / (unsigned)headGroups;
    const unsigned xcd = blockIdx.x % kXcds, u = blockIdx.x / kXcds, p = u / perGroup;
    const unsigned shares = kXcds / (unsigned)headGroups;  // of the positions
    pos = (int)(p * shares + xcd / (unsigned)headGroups);
    head = (int)(xcd % (unsigned)headGroups * perGroup + (u - p * perGroup));
    if (pos >= nRW) return;
  }
  const int pitchOut = HEADS ? ldOut : D;
  const int wave = pipe::uniform(threadIdx.x >> 6);
  for (int iter = 0;; iter++) {
  if constexpr (PERSIST) {
    if (pos >= nRW) break;
    // position of the window after this one; read at the end of this iteration
    if (threadIdx.x == 0) sNextPos[iter & 1] = atomicAdd(&g_windowCursor, 1) + (int)gridDim.x;
  }
  do {
  const int w = windowOrder ? windowOrder[pos] : pos;
  if ((unsigned)w >= (unsigned)nRW) break;  // a corrupt order entry must not index out of range

  int t0 = rowWindowOffset[w];
  int t1 = rowWindowOffset[w + 1];
  // block ranges that do not fit the structure (a mismatched rowWindowOffset) are not followed:
  // the window is treated as empty
  if (t0 < 0 || (int64_t)t1 > nTcb || t1 < t0) t1 = t0;
  const int nSteps = (t1 - t0 + BPS - 1) / BPS;

  pipe::Problem<ET> pb;
  pb.sparseAToXidx = sparseAToXidx;
  pb.bitmapBytes = bitmapBytes;
  pb.Q = Q;
  pb.K = K;
  pb.V = V;
  pb.N = N;
  pb.scaleLog2 = scaleLog2;
  pb.pitchIn = HEADS ? ldIn : D;
  pb.pitchQ = pb.pitchIn;
  pb.nTcb = nTcb;
  pb.sddmm = sddmm;
  const unsigned ringAddr =
      (unsigned)(uintptr_t)(F3S_LDS unsigned char*)smem + (unsigned)wave * WAVE_BYTES;
  Pipe pp;
  pp.init(pb, w, ringAddr, head);
  {
    // wave v takes steps [v * nSteps / NWAVES, (v + 1) * nSteps / NWAVES)
    const int sb = (int)((int64_t)wave * nSteps / NWAVES);
    const int se = (int)((int64_t)(wave + 1) * nSteps / NWAVES);
    const int rb = t0 + sb * BPS;
    const int re = (t0 + se * BPS) < t1 ? (t0 + se * BPS) : t1;
    if (re > rb) pp.run(pb, rb, re);
  }

  // one LDS merge per window; the buffers reuse the rings' memory once every wave has left its loop
  pipe::put_partials<D, NWAVES, SOFTMAX, NH>(pp, smem, wave);
  pipe::MergedRows<D, NWAVES, SOFTMAX, NH> rows;
  rows.merge(smem, 0);
  rows.store(w, N, out + head * D, pitchOut);
  } while (false);
  if constexpr (!PERSIST) break;
  __syncthreads();  // the merge buffers are free again, the next position has arrived
  if constexpr (PERSIST) pos = sNextPos[iter & 1];
  }
  if constexpr (CLOCKED) {
    // {first tick, last tick, CU} of this workgroup, as the reference's timed kernels record
    // {begin, end, smid} per block (src/F3S_kernel.cu:1363-1367)
    __syncthreads();
    if (threadIdx.x == 0) {
      cuTimer[3 * (size_t)blockIdx.x + 0] = tBegin;
      cuTimer[3 * (size_t)blockIdx.x + 1] = realtime_ticks();
      cuTimer[3 * (size_t)blockIdx.x + 2] = cu_key();
    }
  }
}

// above 64 KiB of LDS the kernel has to be told
template <typename KernelT>
int allow_lds(KernelT kernel, size_t bytes) {
  if (bytes > 64 * 1024)
    F3S_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                      hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes));
  return 0;
}

// F3S_WINDOW_PERSISTENT=1 in the environment (read per call): the workgroup-per-window kernel in
// its cursor form
inline bool window_cursor_requested() {
  const char* e = getenv("F3S_WINDOW_PERSISTENT");
  return e && strcmp(e, "1") == 0;
}

struct HeadLayout {
  int nHeads;       // 0: contiguous [N, d] single head
  int ldIn;         // row pitch of Q/K/V in elements
  int ldOut;        // row pitch of out in floats
  int64_t nTcb;     // TC blocks of the structure (bounds every window's block range)
};

// 32-wide heads are computed one by one where there is little to do: the longest window decides there, and
// one workgroup takes longer for two of its heads (us; blocks times pairs of heads). One pair: R-MAT 57 000
// 35 -> 43, 88 000 59 -> 63, uniform 39 000 24 -> 26, power-law 75 000 56 -> 64, 72 000 35 -> 28; from
// 118 000 on no measured graph lost (52 -> 44, 69 -> 60, 79 -> 75, 223 -> 177, 836 -> 682). Two pairs: R-MAT
// 30 000 29 -> 34, 55 000 33 -> 32, 60 000 44 -> 44, power-law 68 000 33 -> 28, uniform 78 000 58 -> 40. Four:
// R-MAT 60 000 38 -> 39, uniform 55 000 33 -> 28, R-MAT 110 000 59 -> 48.
inline bool pairs_pay(int64_t nTcb, int pairs) {
  return nTcb * pairs >= (pairs == 1 ? 100000 : 50000);
}

// NH = 2: D = 64 stands for two heads of 32, hl.nHeads for the number of pairs.
template <typename ET, int D, bool SOFTMAX, bool WIDE, int NH = 1>
int launch_d(const int32_t* rwo, const int32_t* order, const int32_t* atox, const uint64_t* bitmap,
             int N, const void* Q, const void* K, const void* V, float scaleLog2, float* out,
             unsigned long long* cuTimer, HeadLayout hl, hipStream_t stream) {
  const int nRW = (N + kWinRows - 1) / kWinRows;
  if (nRW == 0) return 0;
  if constexpr (D == 32) {
    if (heads_in_pairs(D, hl.nHeads) && pairs_pay(hl.nTcb, hl.nHeads / 2)) {
      hl.nHeads /= 2;
      return launch_d<ET, 64, SOFTMAX, WIDE, 2>(rwo, order, atox, bitmap, N, Q, K, V, scaleLog2, out,
                                                cuTimer, hl, stream);
    }
  }
  const auto* bm = reinterpret_cast<const uint8_t*>(bitmap);
  const auto* q = static_cast<const ET*>(Q);
  const auto* k = static_cast<const ET*>(K);
  const auto* v = static_cast<const ET*>(V);
  const unsigned gw = (unsigned)nRW;
  const int heads = hl.nHeads > 0 ? hl.nHeads : 1;
  const int headGroups = head_groups(D, heads);
  const unsigned shares = kXcds / (unsigned)headGroups;
  const unsigned headGrid = (gw + shares - 1) / shares * (heads / headGroups) * kXcds;
#define F3S_LAUNCH(TEAM_, CLOCKED_, HEADS_, GRID)                                              \
  {                                                                                            \
    auto kernel = f3s_fwd_kernel<ET, D, TEAM_, SOFTMAX, CLOCKED_, HEADS_, false, WIDE, false,  \
                                 HEADS_ ? NH : 1>;                                             \
    constexpr size_t lds = team_lds(TEAM_, D);                                                 \
    if (int rc = allow_lds(kernel, lds)) return rc;                                            \
    hipLaunchKernelGGL(kernel, dim3(GRID), dim3(kTeamWaves * 64), lds, stream, rwo,            \
                       order, atox, bm, N, nRW, hl.nTcb, q, k, v, scaleLog2, out, cuTimer,     \
                       heads, headGroups, hl.nHeads > 0 ? hl.ldIn : D,                         \
                       hl.nHeads > 0 ? hl.ldOut : D,                                           \
                       (float*)nullptr);                                                       \
  }
  if (NH > 1) {
    F3S_LAUNCH(TEAM_SHORT, false, true, headGrid)
  } else if (!WIDE && hl.nHeads == 0 && !cuTimer && window_cursor_requested()) {
    // F3S_WINDOW_PERSISTENT=1: as many workgroups as the GPU holds at once, windows drawn from
    // a cursor (measured slower than launch order, which therefore stays the default)
    if constexpr (!WIDE && NH == 1) {
      auto kernel = f3s_fwd_kernel<ET, D, TEAM_SHORT, SOFTMAX, false, false, false, false, true>;
      constexpr size_t lds = team_lds(TEAM_SHORT, D);
      constexpr int threads = kTeamWaves * 64;
      if (int rc = allow_lds(kernel, lds)) return rc;
      int dev = 0, nCu = 0, perCu = 0;
      F3S_HIP_CHECK(hipGetDevice(&dev));
      F3S_HIP_CHECK(hipDeviceGetAttribute(&nCu, hipDeviceAttributeMultiprocessorCount, dev));
      F3S_HIP_CHECK(hipOccupancyMaxActiveBlocksPerMultiprocessor(
          &perCu, reinterpret_cast<const void*>(kernel), threads, lds));
      unsigned grid = (unsigned)(nCu * (perCu > 0 ? perCu : 1));
      if (grid > gw) grid = gw;
      hipLaunchKernelGGL(reset_window_cursor_kernel<0>, dim3(1), dim3(1), 0, stream);
      hipLaunchKernelGGL(kernel, dim3(grid), dim3(threads), lds, stream, rwo, order, atox, bm, N,
                         nRW, hl.nTcb, q, k, v, scaleLog2, out, cuTimer, 1, 1, D, D,
                         (float*)nullptr);
    }
  } else if constexpr (NH == 1) {
    constexpr Team kPairs = D <= 32 ? TEAM_PAIRS : TEAM_SHORT;  // no second kernel above D = 32
    const bool pairs = two_stages(D, hl.nTcb, heads, N);
    if (hl.nHeads > 0) {
      if (pairs) F3S_LAUNCH(kPairs, false, true, headGrid)
      else F3S_LAUNCH(TEAM_SHORT, false, true, headGrid)
    } else if (cuTimer) {
      if (pairs) F3S_LAUNCH(kPairs, true, false, gw)
      else F3S_LAUNCH(TEAM_SHORT, true, false, gw)
    } else {
      if (pairs) F3S_LAUNCH(kPairs, false, false, gw)
      else F3S_LAUNCH(TEAM_SHORT, false, false, gw)
    }
  }
#undef F3S_LAUNCH
  F3S_HIP_CHECK(hipGetLastError());
  return 0;
}

template <int D, bool SOFTMAX, bool WIDE>
int launch_tcb8(const int32_t* rwo, const int32_t* order, const int32_t* atox,
                const uint64_t* bitmap, int N, const void* Q, const void* K, const void* V,
                float scaleLog2, float* out, float* sddmm, int64_t nTcb8, hipStream_t stream) {
  const int nRW = (N + kWinRows - 1) / kWinRows;
  if (nRW == 0) return 0;
  constexpr Team kPairs = D <= 32 ? TEAM_PAIRS : TEAM_SHORT;
  const bool pairs = two_stages(D, nTcb8 / 2, 1, N);
  const size_t lds = pairs ? team_lds(kPairs, D) : team_lds(TEAM_SHORT, D);
  auto kernel = pairs ? f3s_fwd_kernel<_Float16, D, kPairs, SOFTMAX, false, false, true, WIDE>
                      : f3s_fwd_kernel<_Float16, D, TEAM_SHORT, SOFTMAX, false, false, true, WIDE>;
  if (int rc = allow_lds(kernel, lds)) return rc;
  hipLaunchKernelGGL(kernel, dim3(nRW), dim3(kTeamWaves * 64), lds, stream, rwo, order, atox,
                     reinterpret_cast<const uint8_t*>(bitmap), N, nRW, nTcb8,
                     static_cast<const _Float16*>(Q), static_cast<const _Float16*>(K),
                     static_cast<const _Float16*>(V), scaleLog2, out, nullptr, 1, 1, D, D, sddmm);
  F3S_HIP_CHECK(hipGetLastError());
  return 0;
}

template <typename ET, bool WIDE>
int dispatch_d(const int32_t* rwo, const int32_t* order, const int32_t* atox,
               const uint64_t* bitmap, int N, int d, const void* Q, const void* K, const void* V,
               float scaleLog2, int applySoftmax, float* out, unsigned long long* cuTimer,
               HeadLayout hl, hipStream_t stream) {
#define F3S_DISPATCH(DD)                                                                        \
  if (d == DD)                                                                                  \
    return applySoftmax ? launch_d<ET, DD, true, WIDE>(rwo, order, atox, bitmap, N, Q, K, V,    \
                                                       scaleLog2, out, cuTimer, hl, stream)     \
                        : launch_d<ET, DD, false, WIDE>(rwo, order, atox, bitmap, N, Q, K, V,   \
                                                        scaleLog2, out, cuTimer, hl, stream);
  F3S_FOR_EACH_HEAD_DIM(F3S_DISPATCH)
#undef F3S_DISPATCH
  return fail(-2, "f3s_attention_fwd: head dim %d unsupported (a multiple of 32 up to 256)", d);
}


}  // namespace window
}  // namespace f3s
