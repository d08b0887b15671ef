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
//   TEAM_LONG   the few long windows of a graph of short ones, one workgroup after the other per CU:
//               as many bytes in flight as one CU's LDS holds, eight waves of two stages up to
//               D = 64, eight of one stage up to D = 128, four above.
enum Team { TEAM_SHORT, TEAM_PAIRS, TEAM_LONG };
constexpr int team_waves(Team t, int d) { return t == TEAM_LONG && d <= 128 ? 8 : 4; }
constexpr int team_stages(Team t, int d) { return t != TEAM_SHORT && d <= 64 ? 2 : 1; }
constexpr int waves_per_simd(Team t, int d) {
  if (d > 128) return 1;
  return t == TEAM_LONG || d > 64 ? 2 : d > 32 ? 3 : 4;
}

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
  const int dp = d <= 32 ? 32 : d <= 64 ? 64 : d <= 128 ? 128 : 256;
  return (size_t)team_waves(t, d) * (team_stages(t, d) * 128 * dp + 2 * 768);
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
__global__ __launch_bounds__(team_waves(TEAM, D) * 64)
__attribute__((amdgpu_waves_per_eu(waves_per_simd(TEAM, D), waves_per_simd(TEAM, D)))) void
f3s_fwd_kernel(
    const int32_t* __restrict__ rowWindowOffset, const int32_t* __restrict__ windowOrder,
    const int32_t* __restrict__ sparseAToXidx, const uint8_t* __restrict__ bitmapBytes, int N,
    int nRW, int64_t nTcb, const ET* __restrict__ Q, const ET* __restrict__ K,
    const ET* __restrict__ V, float scaleLog2, float* __restrict__ out,
    unsigned long long* __restrict__ cuTimer, int nHeads, int headGroups, int ldIn, int ldOut,
    float* __restrict__ sddmm, int minBlocks, int nPositions) {
  constexpr int NWAVES = team_waves(TEAM, D);
  constexpr int WAVE_BYTES = pipe::Geo<D, team_stages(TEAM, D)>::WAVE_BYTES;
  static_assert(team_lds(TEAM, D) == (size_t)NWAVES * WAVE_BYTES, "what the launch asks for");
  typedef pipe::PairPipeline<ET, D, SOFTMAX, HEADS, W8, team_stages(TEAM, D), WIDE, NH> Pipe;
  constexpr int T = D / 16;
  constexpr int OSTRIDE = D + 4;
  constexpr int BPS = W8 ? 4 : 2;  // blocks of the structure per pipeline step
  extern __shared__ __align__(1024) unsigned char smem[];
  unsigned long long tBegin = 0;
  if constexpr (CLOCKED) tBegin = realtime_ticks();

  static_assert(!PERSIST || (!CLOCKED && !HEADS && !W8), "the persistent form is single-head");
  __shared__ int sNextPos[2];
  constexpr bool scan = TEAM == TEAM_LONG;
  __shared__ int sUnitCount;
  __shared__ int sUnitList[scan ? NWAVES * 64 : 1];
  int pos = (int)blockIdx.x, head = 0;
  if constexpr (HEADS && !scan) {
    const unsigned perGroup = (unsigned)nHeads / (unsigned)headGroups;
    const unsigned xcd = blockIdx.x % kXcds, u = blockIdx.x / kXcds, p = u / perGroup;
    const unsigned shares = kXcds / (unsigned)headGroups;  // of the positions
    pos = (int)(p * shares + xcd / (unsigned)headGroups);
    head = (int)(xcd % (unsigned)headGroups * perGroup + (u - p * perGroup));
    if (pos >= nPositions) return;
  }
  // A launch that shares the windows with the wave-per-window kernel (TEAM_LONG, minBlocks >= 0)
  // covers the (position, head) units of the order's first nPositions positions with a grid of its
  // own size: thread t of workgroup b looks at unit b + t * gridDim.x, and the workgroup computes
  // the units it finds long, one after the other. When no window is long, which is the usual
  // case on a graph of short windows, the launch is a few hundred workgroups that read a count each
  // and leave, instead of one workgroup per unit; in a heavy-first order the long units are the
  // first ones and are dealt out round-robin.
  int nMine = 1;
  if constexpr (scan) {
    if (threadIdx.x == 0) sUnitCount = 0;
    __syncthreads();
    const int heads = HEADS ? nHeads : 1;
    const int64_t nUnits = (int64_t)nPositions * heads;
    const int64_t u = (int64_t)blockIdx.x + (int64_t)threadIdx.x * (int64_t)gridDim.x;
    if (u < nUnits) {
      const int p = (int)(u / heads);
      const int w = windowOrder ? windowOrder[p] : p;
      if ((unsigned)w < (unsigned)nRW) {
        const int t0 = rowWindowOffset[w];
        const int t1 = rowWindowOffset[w + 1];
        if (t0 >= 0 && (int64_t)t1 <= nTcb && t1 - t0 > minBlocks)
          sUnitList[atomicAdd(&sUnitCount, 1)] = (int)u;
      }
    }
    __syncthreads();
    nMine = sUnitCount;
  }
  const int pitchOut = HEADS ? ldOut : D;
  const int lane = threadIdx.x & 63;
  const int wave = pipe::uniform(threadIdx.x >> 6);
  const int g = lane >> 4;
  const int c = lane & 15;
  for (int iter = 0;; iter++) {
  if constexpr (scan) {
    if (iter >= nMine) break;
    const int u = sUnitList[iter];
    pos = HEADS ? u / nHeads : u;
    head = HEADS ? u - pos * nHeads : 0;
  }
  if constexpr (PERSIST) {
    if (pos >= nPositions) break;
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
  // windows of at most minBlocks blocks belong to the wave-per-window kernel of the same call
  // (f3s_fwd_unit_kernel); -1 when this kernel computes every window
  if (t1 - t0 <= minBlocks) break;
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

  // ---- merge the waves' partial (m, l, O) and write the window's rows. The merge buffers reuse
  // the rings' memory once every wave has left its loop.
  __syncthreads();
  float* sM = reinterpret_cast<float*>(smem);                    // [NH][NWAVES][16]
  float* sL = sM + NH * NWAVES * 16;                             // [NH][NWAVES][16]
  float* sO = sL + NH * NWAVES * 16;                             // [NWAVES][16][OSTRIDE]
#pragma unroll
  for (int h = 0; h < NH; h++) {
    float l = pp.l[h];
    if constexpr (SOFTMAX) l = pipe::row_sum4(l);
    if (g == 0) {
      sM[(h * NWAVES + wave) * 16 + c] = pp.m[h];
      sL[(h * NWAVES + wave) * 16 + c] = l;
    }
  }
#pragma unroll
  for (int j = 0; j < T; j++)
    *reinterpret_cast<float4v*>(&sO[(wave * 16 + c) * OSTRIDE + 16 * j + 4 * g]) = pp.o[j];
  __syncthreads();

  constexpr int VEC_PER_ROW = D / 4;
  for (int idx = threadIdx.x; idx < 16 * VEC_PER_ROW; idx += NWAVES * 64) {
    const int q = idx / VEC_PER_ROW;
    const int cv = idx % VEC_PER_ROW;
    const int64_t row = (int64_t)w * 16 + q;
    if (row >= N) continue;
    float4 acc = {0.f, 0.f, 0.f, 0.f};
    if constexpr (SOFTMAX) {
      const int ml = (NH > 1 ? cv / (VEC_PER_ROW / NH) * NWAVES * 16 : 0) + q;  // of this head and row
      float mAll = sM[ml];
#pragma unroll
      for (int v = 1; v < NWAVES; v++) mAll = fmaxf(mAll, sM[v * 16 + ml]);
      float lAll = 0.0f;
#pragma unroll
      for (int v = 0; v < NWAVES; v++) {
        const float f = pipe::fast_exp2(sM[v * 16 + ml] - mAll);
        lAll = fmaf(f, sL[v * 16 + ml], lAll);
        const float4 ov = *reinterpret_cast<const float4*>(&sO[(v * 16 + q) * OSTRIDE + cv * 4]);
        acc.x = fmaf(f, ov.x, acc.x);
        acc.y = fmaf(f, ov.y, acc.y);
        acc.z = fmaf(f, ov.z, acc.z);
        acc.w = fmaf(f, ov.w, acc.w);
      }
      const float inv = (lAll == 0.0f) ? 0.0f : 1.0f / lAll;
      acc.x *= inv;
      acc.y *= inv;
      acc.z *= inv;
      acc.w *= inv;
    } else {
#pragma unroll
      for (int v = 0; v < NWAVES; v++) {
        const float4 ov = *reinterpret_cast<const float4*>(&sO[(v * 16 + q) * OSTRIDE + cv * 4]);
        acc.x += ov.x;
        acc.y += ov.y;
        acc.z += ov.z;
        acc.w += ov.w;
      }
    }
    store_out(out + row * pitchOut + head * D + cv * 4, out_vec{acc.x, acc.y, acc.z, acc.w});
  }
  } while (false);
  if constexpr (!PERSIST) {
    if constexpr (!scan) break;
  }
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
  int minBlocks;    // this kernel skips windows of at most minBlocks blocks (-1: none)
  int gridWindows;  // positions of the window order this launch covers (<= nRW)
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
  const unsigned gw = (unsigned)(hl.gridWindows < nRW ? hl.gridWindows : nRW);
  if (gw == 0) return 0;
  const int heads = hl.nHeads > 0 ? hl.nHeads : 1;
  const unsigned units = gw * (unsigned)heads;
  const int headGroups = head_groups(D, heads);
  const unsigned shares = kXcds / (unsigned)headGroups;
  const unsigned headGrid = (gw + shares - 1) / shares * (heads / headGroups) * kXcds;
#define F3S_LAUNCH(TEAM_, CLOCKED_, HEADS_, GRID)                                              \
  {                                                                                            \
    auto kernel = f3s_fwd_kernel<ET, D, TEAM_, SOFTMAX, CLOCKED_, HEADS_, false, WIDE, false,  \
                                 HEADS_ ? NH : 1>;                                             \
    constexpr size_t lds = team_lds(TEAM_, D);                                                 \
    if (int rc = allow_lds(kernel, lds)) return rc;                                            \
    hipLaunchKernelGGL(kernel, dim3(GRID), dim3(team_waves(TEAM_, D) * 64), lds, stream, rwo,  \
                       order, atox, bm, N, nRW, hl.nTcb, q, k, v, scaleLog2, out, cuTimer,     \
                       heads, headGroups, hl.nHeads > 0 ? hl.ldIn : D,                         \
                       hl.nHeads > 0 ? hl.ldOut : D,                                           \
                       (float*)nullptr, hl.minBlocks, (int)gw);                                \
  }
  if (hl.minBlocks >= 0) {
    // a launch next to the wave-per-window kernel looks for its units itself (see the kernel): one
    // unit per thread at most, two workgroups per CU (one at a time) when that is enough
    if constexpr (WIDE) {
      return fail(-2, "f3s_attention: windows are not shared in the 64-bit form");
    } else {
      const unsigned threads = (unsigned)team_waves(TEAM_LONG, D) * 64;
      unsigned grid = (units + threads - 1) / threads;
      if (grid < 512u) grid = units < 512u ? units : 512u;
      if (NH > 1 || hl.nHeads > 0) F3S_LAUNCH(TEAM_LONG, false, true, grid)
      else if constexpr (NH == 1) F3S_LAUNCH(TEAM_LONG, false, false, grid)
    }
  } else if (NH > 1) {
    F3S_LAUNCH(TEAM_SHORT, false, true, headGrid)
  } else if (!WIDE && hl.nHeads == 0 && !cuTimer && window_cursor_requested()) {
    // F3S_WINDOW_PERSISTENT=1: as many workgroups as the GPU holds at once, windows drawn from
    // a cursor (measured slower than launch order, which therefore stays the default)
    if constexpr (!WIDE && NH == 1) {
      auto kernel = f3s_fwd_kernel<ET, D, TEAM_SHORT, SOFTMAX, false, false, false, false, true>;
      constexpr size_t lds = team_lds(TEAM_SHORT, D);
      constexpr int threads = team_waves(TEAM_SHORT, D) * 64;
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
                         nRW, hl.nTcb, q, k, v, scaleLog2, out, cuTimer, 1, 1, D, D, (float*)nullptr,
                         hl.minBlocks, (int)gw);
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
  static_assert(team_waves(kPairs, D) == team_waves(TEAM_SHORT, D), "one launch for both");
  if (int rc = allow_lds(kernel, lds)) return rc;
  hipLaunchKernelGGL(kernel, dim3(nRW), dim3(team_waves(TEAM_SHORT, D) * 64), lds, stream, rwo, order, atox,
                     reinterpret_cast<const uint8_t*>(bitmap), N, nRW, nTcb8,
                     static_cast<const _Float16*>(Q), static_cast<const _Float16*>(K),
                     static_cast<const _Float16*>(V), scaleLog2, out, nullptr, 1, 1, D, D, sddmm, -1,
                     nRW);
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
