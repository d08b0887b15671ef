// Fused 3S attention with one wave per unit of work (gfx950). The step over a TC-block pair is
// the one every attention kernel here runs (f3s_pair_pipeline.h documents its data flow and its
// numerics); what differs from the workgroup-per-window kernel of f3s_attention.hip is the
// decomposition.
//
// Column-sliced schedule, for graphs with long windows:
//   * the column range is cut into slices and an XCD only ever works on one slice (of some of the
//     heads, for some of the windows: XcdSplit) at a time. The K/V rows of a slice mostly stay in
//     the XCD's 4 MiB L2, so a row is fetched from the memory side about once per XCD instead of
//     once per window that names it;
//   * a wave computes one (window, slice[, head]) unit: the window's TC blocks whose first column
//     falls into the slice, with (m, l, O) in registers, and writes the unit's partial result to
//     scratch. A second kernel merges a window's partials (log-sum-exp) and writes its rows;
//   * two forms of the unit kernel. f3s_fwd_unit_kernel: the launch order is the schedule
//     (workgroup b of a launch runs on XCD b % 8: that is how the hardware deals workgroups when
//     all eight XCDs sit behind one device; elsewhere the results are the same and only the
//     locality is lost). f3s_fwd_resident_kernel: a grid that fits the GPU at once, every
//     workgroup asks the hardware which XCD it runs on and works through that XCD's units.
//
// The reference has no counterpart: its kernels (src/F3S_kernel.cu:1371-1583) walk one window
// per thread block from its first TC block to its last. Its window order (src/utils.cu:400-436)
// is kept: units are issued heavy windows first.
#include <stdlib.h>

#include "f3s_common.h"
#include "f3s_pair_pipeline.h"
#include "f3s_wave_units.h"

namespace f3s {
namespace {

constexpr int kMaxPhases = 16;  // slices that an XCD works through one after the other at most
constexpr int kUnitWaves = 4;  // waves (= units) per workgroup; they do not cooperate

// Stages of a wave's LDS ring and waves per SIMD the register allocator is held to. Units are runs of dozens
// of blocks: two stages, as many waves as the rings allow (four workgroups of four waves per CU at D = 32,
// two up to D = 128, one above).
constexpr int unit_stages(int d) { return d <= 64 ? 2 : 1; }
constexpr int unit_waves_per_simd(int d) { return d <= 32 ? 4 : d <= 128 ? 2 : 1; }

// Partial result of a unit: the O^T tiles as the lanes hold them, one coalesced 1 KiB row of 16
// bytes per lane and tile (lane (g, c) holds O[q = c][16j + 4g + i] in o[j][i]), then m[16] and
// l[16].
template <int D>
constexpr int partial_floats() {
  return 16 * D + 32;
}

// probe builds: the partials through the caches instead of past them
#ifdef F3S_PROBE_PARTIAL_CACHED_STORE
#define F3S_PARTIAL_STORE(v, p) (*(p) = (v))
#else
#define F3S_PARTIAL_STORE(v, p) __builtin_nontemporal_store((v), (p))
#endif
#ifdef F3S_PROBE_PARTIAL_CACHED_LOAD
#define F3S_PARTIAL_LOAD(p) (*(p))
#else
#define F3S_PARTIAL_LOAD(p) __builtin_nontemporal_load(p)
#endif

// of NH heads of D / NH features each, whose partials lie `stride` floats apart
template <int D, int NH, typename PipeT>
__device__ __forceinline__ void store_partial(const PipeT& pp, float* __restrict__ dst,
                                              int64_t stride) {
  constexpr int TH = D / NH / 16;
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int h = 0; h < NH; h++) {
#pragma unroll
    for (int jj = 0; jj < TH; jj++)
      F3S_PARTIAL_STORE(pp.o[h * TH + jj], reinterpret_cast<float4v*>(dst) + jj * 64 + lane);
    const float l = pipe::row_sum4(pp.l[h]);  // m is the same in the four lanes of a row already
    if (lane < 32) F3S_PARTIAL_STORE(lane < 16 ? pp.m[h] : l, dst + 16 * (D / NH) + lane);
    dst += stride;
  }
}

// One wave per unit, kUnitWaves independent units per workgroup. A unit is the TC blocks of one (window,
// column slice[, head]); the result is a partial (m, l, O). Workgroup b: XCD b % 8, then (phase, group of
// kUnitWaves consecutive units of that XCD and phase); which position, head and slice a unit is: XcdSplit.
// NH = 2: D = 64 stands for two heads of 32; split counts such pairs, nHeads heads.
template <typename ET, int D, bool SOFTMAX, bool HEADS, int NH = 1>
__global__ __launch_bounds__(kUnitWaves * 64)
__attribute__((amdgpu_waves_per_eu(unit_waves_per_simd(D), unit_waves_per_simd(D)))) void
f3s_fwd_unit_kernel(const int32_t* __restrict__ windowOrder,
                    const int32_t* __restrict__ sparseAToXidx,
                    const uint8_t* __restrict__ bitmapBytes,
                    const int32_t* __restrict__ sliceStart, XcdSplit split, int nGroups, int N,
                    int nRW, int64_t nTcb, const ET* __restrict__ Q, const ET* __restrict__ K,
                    const ET* __restrict__ V, float scaleLog2, float* __restrict__ partial,
                    int nHeads, int ldIn, int ldQ) {
  constexpr int STAGES = unit_stages(D);
  typedef pipe::PairPipeline<ET, D, SOFTMAX, HEADS, false, STAGES, false, NH> Pipe;
  extern __shared__ __align__(1024) unsigned char smem[];

  const int wave = uniform(threadIdx.x >> 6);

  // Workgroup b runs on XCD b % 8; its waves take consecutive units of that XCD's list.
  const int j = blockIdx.x / kXcds;
  const int phase = j / nGroups;
#ifdef F3S_PROBE_SAME_UNIT
  // probe: the four waves of a workgroup all compute its first unit, at the same time
  const unsigned u = (unsigned)(j - phase * nGroups) * kUnitWaves;
#else
  const unsigned u = (unsigned)(j - phase * nGroups) * kUnitWaves + wave;
#endif
  const Unit un = split.unit(blockIdx.x % kXcds, phase, u);
  const int pos = un.pos;
  const int head = HEADS ? un.head : 0;
  if (pos >= nRW) return;
  const int w = uniform(windowOrder ? windowOrder[pos] : pos);
  if ((unsigned)w >= (unsigned)nRW) return;  // a corrupt order entry must not index out of range
  const int64_t at = (int64_t)w * (split.slices() + 1) + un.slice;
  const int t0 = uniform(sliceStart[at]);
  const int t1 = uniform(sliceStart[at + 1]);
  if (t1 <= t0) return;  // empty unit: nothing is written, the merge skips it
  // block ranges that do not fit the structure (a mismatched rowWindowOffset) are not followed;
  // the slice index never holds one (sliced_setup_kernel makes such a window empty)
  if (t0 < 0 || (int64_t)t1 > nTcb) return;

  const pipe::Problem<ET> pb = make_problem<ET, D, HEADS>(sparseAToXidx, bitmapBytes, Q, K, V, N,
                                                          scaleLog2, ldIn, nTcb, ldQ);
  const unsigned ringAddr =
      (unsigned)(uintptr_t)(F3S_LDS unsigned char*)smem + (unsigned)wave * pipe::Geo<D, STAGES>::WAVE_BYTES;
  Pipe pp;
  pp.init(pb, w, ringAddr, head);
  pp.run(pb, t0, t1);

  const int64_t wh = (int64_t)w * (HEADS ? nHeads : 1) + head * NH;
  const int64_t stride = (int64_t)split.slices() * partial_floats<D / NH>();
  store_partial<D, NH>(pp, partial + wh * stride + un.slice * partial_floats<D / NH>(), stride);
}

// ---- workspace of the column-sliced schedule (f3s_attention_workspace_bytes) ------------------
//   header (256 B) | tickets of the resident grid (256 B) | sliceStart [nRW * (S + 1)] |
//   partial results [nRW * nHeads * S]
// The slice boundaries depend on the TC-block structure only. sliced_setup_kernel builds them at
// the start of every call unless the header says that f3s_attention_prepare built them for
// exactly these arrays.
struct SlicedHeader {
  uint32_t magic;
  int32_t N, S, prepared;
  int64_t nTcb;
  const void* rwo;
  const void* atox;
};
constexpr uint32_t kSlicedMagic = 0xF35C0DE5u;

// Rows of 128 bytes gathered from addresses that are multiples of 256 are served faster than rows
// from the odd 128-byte lines in between (233k-node graph, d = 64: 1.42 ms with every row on an
// even line, 1.55 ms with every row on an odd line, 1.48 ms for contiguous rows, which alternate;
// the L2 hit and miss counts are the same in all three). The single-head call at d = 64 therefore
// gathers from copies of K and V with a row pitch of 256 bytes, made at the start of the call.
constexpr int kPaddedRowBytes = 256;
typedef int pad_chunk __attribute__((ext_vector_type(4)));

// sliceStart[w * (S + 1) + s] = first TC block of window w whose first (smallest) column id is
// >= s * sliceWidth; entry S is the window's end. 16 lanes per window look at 16 evenly spaced
// blocks together, then each finishes one boundary by binary search between two of them (their first
// columns ascend). Bound by memory: what is left after the first look costs a line or two per step
// and boundary, 100 MB at 233k nodes. Boundaries interpolated instead of searched read a third of
// that, but the twentieth of the blocks they leave in the wrong slice slows the unit kernel down by
// 5 to 14 %. A block range that does not fit the structure (a mismatched rowWindowOffset) makes the
// window empty: every entry 0.
// mode 0: part of an attention call, index rebuilt; mode 1: f3s_attention_prepare (index built,
// header written); mode 2: part of an attention call whose caller says the workspace is prepared:
// the index is kept if the header confirms it and rebuilt otherwise.
// Workgroups from setupBlocks on copy K and V instead (if the call wants the copies): the searches
// are short chains of loads, the copy is bound by memory, and one launch saves the gap of two
// (233k nodes: 16 + 21 us and the gap apart, 34 us together).
__global__ __launch_bounds__(256) void sliced_setup_kernel(
    const int32_t* __restrict__ rowWindowOffset, const int32_t* __restrict__ sparseAToXidx, int N,
    int nRW, int S, int sliceWidth, int64_t nTcb, SlicedHeader* __restrict__ hdr, int mode,
    int32_t* __restrict__ tickets, int32_t* __restrict__ sliceStart, int setupBlocks,
    const pad_chunk* __restrict__ K, const pad_chunk* __restrict__ V, int64_t chunks,
    pad_chunk* __restrict__ Kp, pad_chunk* __restrict__ Vp) {
  if ((int)blockIdx.x >= setupBlocks) {
    // K and V rows of 128 bytes to a pitch of 256 bytes (one thread per 16 bytes of each)
    const int64_t i = (int64_t)((int)blockIdx.x - setupBlocks) * blockDim.x + threadIdx.x;
    if (i >= chunks) return;
    const int64_t at = (i >> 3) * (kPaddedRowBytes / 16) + (i & 7);
    const pad_chunk k = __builtin_nontemporal_load(K + i);  // read once, by nobody else
    const pad_chunk v = __builtin_nontemporal_load(V + i);
    Kp[at] = k;
    Vp[at] = v;
    return;
  }
  const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx < kXcds) tickets[idx] = 0;
  if (mode == 2) {
    const bool cached = hdr->magic == kSlicedMagic && hdr->prepared == 1 && hdr->N == N &&
                        hdr->S == S && hdr->nTcb == nTcb && hdr->rwo == rowWindowOffset &&
                        hdr->atox == sparseAToXidx;
    if (cached) return;
  }
  if (idx == 0) {
    if (mode == 1) {
      hdr->magic = kSlicedMagic;
      hdr->N = N;
      hdr->S = S;
      hdr->nTcb = nTcb;
      hdr->rwo = rowWindowOffset;
      hdr->atox = sparseAToXidx;
      hdr->prepared = 1;
    } else {
      hdr->prepared = 0;  // the index no longer belongs to an earlier f3s_attention_prepare
    }
  }
  const int sub = threadIdx.x & 15;
  const int w = (int)(idx >> 4);
  int first = 0, end = 0;
  if (w < nRW) {
    first = rowWindowOffset[w];
    end = rowWindowOffset[w + 1];
    if (first < 0 || (int64_t)end > nTcb || end < first) first = end = 0;
  }
  const int n = end - first;
  const int probe = first + (int)((int64_t)sub * n / 16);
  const int seen = n > 0 ? sparseAToXidx[(int64_t)probe * 16] : 0;
  int32_t* dst = sliceStart + (int64_t)w * (S + 1);
  for (int b0 = 0; b0 < S; b0 += 16) {
    const int64_t limit = (int64_t)(b0 + sub) * sliceWidth;
    int below = 0;  // of the window's probes in front of this lane's boundary
#pragma unroll
    for (int k = 0; k < 16; k++) below += (__shfl(seen, k, 16) < limit) ? 1 : 0;
    const int left = below > 0 ? below - 1 : 0;
    // the boundary is the first block of (lo, hi) at or beyond `limit`, or hi
    int lo = first + (int)((int64_t)left * n / 16) + 1;
    int hi = first + (int)((int64_t)below * n / 16);
    while (lo < hi) {
      const int mid = (lo + hi) >> 1;
      if (sparseAToXidx[(int64_t)mid * 16] < limit)
        lo = mid + 1;
      else
        hi = mid;
    }
    if (w < nRW && b0 + sub < S) dst[b0 + sub] = hi;
  }
  if (w < nRW && sub == 0) dst[S] = end;
}

// The resident form: as many workgroups as the GPU holds at once, NW independent waves each.
//   * A workgroup takes a ticket of the XCD it runs on (XCC_ID from the hardware) and with it a
//     slot (xcd, rank); if that XCD's slots are gone (the hardware did not deal the workgroups
//     evenly) it takes a slot of the next XCD. Every slot is taken exactly once, so the result
//     does not depend on where workgroups run; only the L2 locality does.
//   * Slot (x, r) owns groups of NW consecutive units of XCD x's list (phase by phase, heavy
//     windows first), dealt to the ranks in boustrophedon order (r, 2R-1-r, 2R+r, ...: every rank
//     gets an equal share of heavy and light units); the workgroup's waves draw their next unit
//     from a counter in LDS. No device-wide atomic is on the path of a unit.
//   * The window of the unit after next and the block range of the next unit are requested before
//     the current unit runs, so they have arrived when it ends.
// Measured on the 233k-node benchmark graph at d = 64: 1.58 ms against 1.46 ms for the launch-order
// kernel (static shares leave a tail that the hardware's dispatch of fresh workgroups does not; and
// this form gathers from the rows in place, which costs the other 0.02 ms), so it is the one to ask for
// (F3S_SLICED_PERSISTENT=1) where workgroups are not dealt round-robin to the XCDs. A variant in which
// the wave that finishes a window's last unit merges its partials (an arrival counter per window,
// partials written through) took 1.92 ms: the wait for the stores and the returning atomic sit on
// every unit's path.
template <typename ET, int D, bool SOFTMAX, bool HEADS, int NW, int NH = 1>
__global__ __launch_bounds__(NW * 64)
__attribute__((amdgpu_waves_per_eu(unit_waves_per_simd(D), unit_waves_per_simd(D)))) void
f3s_fwd_resident_kernel(const int32_t* __restrict__ windowOrder,
                        const int32_t* __restrict__ sliceStart, XcdSplit split, int nRW, int N,
                        int64_t nTcb, int32_t* __restrict__ tickets,
                        const int32_t* __restrict__ sparseAToXidx,
                        const uint8_t* __restrict__ bitmapBytes, const ET* __restrict__ Q,
                        const ET* __restrict__ K, const ET* __restrict__ V, float scaleLog2,
                        float* __restrict__ partial, int nHeads, int ldIn) {
  typedef pipe::PairPipeline<ET, D, SOFTMAX, HEADS, false, unit_stages(D), false, NH> Pipe;
  extern __shared__ __align__(1024) unsigned char smem[];
  __shared__ int sCtl[2];  // slot of this workgroup; next unit of its sequence

  const int lane = threadIdx.x & 63;
  const int wave = uniform(threadIdx.x >> 6);
  const int per = (int)(gridDim.x / kXcds);  // slots per XCD
  if (threadIdx.x == 0) {
    unsigned xcc;
    asm volatile("s_getreg_b32 %0, hwreg(HW_REG_XCC_ID)" : "=s"(xcc));
    int slot = -1;
    for (int k = 0; k < kXcds && slot < 0; k++) {
      const int x = (int)((xcc + k) & (kXcds - 1));
      const int r = __hip_atomic_fetch_add(&tickets[x], 1, __ATOMIC_RELAXED,
                                           __HIP_MEMORY_SCOPE_AGENT);
      if (r < per) slot = x * per + r;
    }
    sCtl[0] = slot;
    sCtl[1] = 0;
  }
  __syncthreads();
  const int slot = sCtl[0];
  if (slot < 0) return;  // cannot happen: the grid is a multiple of 8, every workgroup finds a slot
  const int x = slot / per;
  const int r = slot - x * per;
  const int heads = HEADS ? nHeads : 1;
  const int S = split.slices();
  const int64_t perPhase = split.units(nRW);
  const int64_t units = perPhase * split.phases;  // units of one XCD

  const pipe::Problem<ET> pb = make_problem<ET, D, HEADS>(sparseAToXidx, bitmapBytes, Q, K, V, N,
                                                          scaleLog2, ldIn, nTcb);
  const unsigned ringAddr =
      (unsigned)(uintptr_t)(F3S_LDS unsigned char*)smem + (unsigned)wave * pipe::Geo<D, unit_stages(D)>::WAVE_BYTES;

  // k-th unit of this workgroup's sequence -> index in the XCD's unit space, -1 past its end,
  // -2 when the sequence is over
  auto unit_index = [&](int k) -> int64_t {
    const int j = k / NW;
    if ((int64_t)j * per * NW >= units) return -2;
    const int grp = (j & 1) ? j * per + (per - 1 - r) : j * per + r;
    const int64_t u = (int64_t)grp * NW + (k - j * NW);
    return u < units ? u : -1;
  };
  auto claim = [&]() -> int64_t {
    int k = 0;
    if (lane == 0)
      k = __hip_atomic_fetch_add(&sCtl[1], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    return unit_index(uniform(k));
  };
  auto unit_of = [&](int64_t u) -> Unit {
    const int phase = (int)(u / perPhase);
    return split.unit(x, phase, (unsigned)(u - phase * perPhase));
  };
  auto window_of = [&](int64_t u) -> int {
    if (u < 0) return -1;
    const int pos = unit_of(u).pos;
    if (pos >= nRW) return -1;
    const int w = windowOrder ? windowOrder[pos] : pos;
    return (unsigned)w < (unsigned)nRW ? w : -1;
  };
  auto slice_of = [&](int64_t u) -> int { return unit_of(u).slice; };

  // three units in flight: `u` runs, u1 has its window and is fetching its block range, u2 is
  // fetching its window
  int64_t u = claim();
  int w = window_of(u);
  int t0 = 0, t1 = 0;
  if (w >= 0) {
    t0 = sliceStart[(int64_t)w * (S + 1) + slice_of(u)];
    t1 = sliceStart[(int64_t)w * (S + 1) + slice_of(u) + 1];
  }
  int64_t u1 = u == -2 ? -2 : claim();
  int w1 = window_of(u1);
  while (u != -2) {
    int t0n = 0, t1n = 0;
    if (w1 >= 0) {
      t0n = sliceStart[(int64_t)w1 * (S + 1) + slice_of(u1)];
      t1n = sliceStart[(int64_t)w1 * (S + 1) + slice_of(u1) + 1];
    }
    const int64_t u2 = u1 == -2 ? -2 : claim();
    const int w2 = window_of(u2);
    const int wu = uniform(w), t0u = uniform(t0), t1u = uniform(t1);
    if (wu >= 0 && t1u > t0u && t0u >= 0 && (int64_t)t1u <= nTcb) {
      const int head = HEADS ? unit_of(u).head : 0;
      Pipe pp;
      pp.init(pb, wu, ringAddr, head);
      pp.run(pb, t0u, t1u);
      const int64_t wh = (int64_t)wu * heads + head * NH;
      const int64_t stride = (int64_t)S * partial_floats<D / NH>();
      store_partial<D, NH>(pp, partial + wh * stride + slice_of(u) * partial_floats<D / NH>(), stride);
    }
    u = u1;
    w = w1;
    t0 = t0n;
    t1 = t1n;
    u1 = u2;
    w1 = w2;
  }
}

// One wave per (window, head): log-sum-exp merge of the unit partials in slice order, then the
// window's rows. Lane (g, c) holds O[q = c][16j + 4g + i] in O[j][i], as in the unit kernels; the
// partials of up to B live slices are requested together. The rows leave through LDS, as in the
// unit kernel.
// Bound by memory: 0.54 GB of partials at 233k nodes and 8 slices. (Lanes that hold O row by row
// from the start need no LDS, but read the tiles in pieces of 64 bytes: 101 -> 120 us there.)
template <int D, bool SOFTMAX>
__global__ __launch_bounds__(256) void f3s_merge_slices_kernel(
    const int32_t* __restrict__ sliceStart, int S, int N, int nRW, int nHeads,
    const float* __restrict__ partial, float* __restrict__ out, int ldOut) {
  constexpr int T = D / 16;
  constexpr int B = D <= 64 ? 4 : D <= 128 ? 2 : 1;
  extern __shared__ __align__(1024) unsigned char smem[];
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int64_t wh = (int64_t)blockIdx.x * 4 + wave;
  if (wh >= (int64_t)nRW * nHeads) return;
  const int w = (int)(wh / nHeads);
  const int head = (int)(wh - (int64_t)w * nHeads);
  const int c = lane & 15;
  float M = 0.0f, L = 0.0f;
  float4v O[T];
#pragma unroll
  for (int j = 0; j < T; j++) O[j] = float4v{0.f, 0.f, 0.f, 0.f};
  const int32_t* ss = sliceStart + (int64_t)w * (S + 1);
  const float* base = partial + wh * S * partial_floats<D>();
  for (int s0 = 0; s0 < S; s0 += 64) {
    const int s = s0 + lane;
    unsigned long long live = __builtin_amdgcn_ballot_w64(s < S && ss[s + 1] > ss[s]);
    while (live) {
      int sel[B];
      float ms[B], ls[B];
      float4v v[B][T];
#pragma unroll
      for (int k = 0; k < B; k++) {
        sel[k] = -1;
        if (live) {
          sel[k] = s0 + __builtin_ctzll(live);
          live &= live - 1;
          const float* src = base + (int64_t)sel[k] * partial_floats<D>();
#pragma unroll
          for (int j = 0; j < T; j++)
            v[k][j] = F3S_PARTIAL_LOAD(reinterpret_cast<const float4v*>(src) + j * 64 + lane);
          if constexpr (SOFTMAX) {
            ms[k] = F3S_PARTIAL_LOAD(src + 16 * D + c);
            ls[k] = F3S_PARTIAL_LOAD(src + 16 * D + 16 + c);
          }
        }
      }
#pragma unroll
      for (int k = 0; k < B; k++) {
        if (sel[k] < 0) continue;
        if constexpr (SOFTMAX) {
          const float mx = fmaxf(M, ms[k]);
          const float a = pipe::fast_exp2(M - mx), b = pipe::fast_exp2(ms[k] - mx);
          M = mx;
          L = fmaf(a, L, b * ls[k]);
#pragma unroll
          for (int j = 0; j < T; j++)
#pragma unroll
            for (int i = 0; i < 4; i++) O[j][i] = fmaf(a, O[j][i], b * v[k][j][i]);
        } else {
#pragma unroll
          for (int j = 0; j < T; j++) O[j] += v[k][j];
        }
      }
    }
  }
  const float inv = SOFTMAX ? (L == 0.0f ? 0.0f : 1.0f / L) : 1.0f;
#pragma unroll
  for (int j = 0; j < T; j++) O[j] *= inv;
  store_rows<D>(O, reinterpret_cast<float*>(smem) + wave * rows_lds_floats<D>(), w, N,
                out + head * D, ldOut);
}

// LDS of a workgroup of rings; above 64 KiB the kernel has to be told once
template <typename KernelT>
int allow_lds(KernelT kernel, size_t bytes) {
  if (bytes > 64 * 1024)
    F3S_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                      hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes));
  return 0;
}

// Slices of a column-sliced call: how many bytes of K + V (of a group's heads) a slice should have at
// most, and what a window's blocks have to be worth for another slice, in parts of a hundred. A slice more
// brings a slice's rows closer to the size of an XCD's L2, and costs every window a partial result more
// (64 d + 128 bytes, written and merged) and a unit's start. From sweeps of 2 to 16 slices over power-law
// graphs of 40 000 to 200 000 nodes and 60 to 430 blocks a window, fp16, 1 to 8 heads:
// - the best number grows with the square root of the blocks per window (d = 128, K + V of 102 MB: 4, 6
//   and 8 slices at 67, 123 and 276 blocks);
// - short rows want smaller slices (d = 32: 8 x 32, 270 blocks: 2.37 ms with 8 MiB, 1.96 ms with 2 MiB), long
//   ones, whose kernels run one wave per SIMD and spend more on arithmetic, larger ones (d = 192, 154 MB,
//   67 blocks: 2.02 ms with 16 slices, 1.01 ms with 2).
// With the blocks per window left out (8 MiB slices, at most sixteen) against now, in us: 100 000 nodes,
// 66 blocks, d = 192 733 -> 493; 200 000, 67: d = 128 857 -> 644, d = 256 2365 -> 1376; 200 000, 123, d = 256
// 2842 -> 2161; 200 000, 276, d = 192 3986 -> 3137; 100 000, 270, 8 x 32 2369 -> 1937; 200 000, 141, 4 x 128
// 5267 -> 4353; 1 000 000, 99, d = 128 6993 -> 5658; 233 000, 450, d = 64 1481 -> 1478.
constexpr int64_t slice_bytes(int d) {
  return (d <= 32 ? 3 : d <= 128 ? 8 : d < 256 ? 25 : 20) * (int64_t)1024 * 1024;
}
constexpr int64_t slice_weight(int d) { return d <= 32 ? 55 : d <= 128 ? 45 : d < 256 ? 30 : 40; }

// How the units are dealt to the XCDs: head groups (split_heads), then column slices; XCDs left over share
// the windows. nTcb < 0: the most slices that any number of blocks asks for (the size of the workspace),
// 8 MiB each above d = 32.
// F3S_SLICE_PHASES = P in the environment forces 8 P slices of all heads.
XcdSplit choose_split(int N, int d, int heads, int64_t nTcb) {
  const char* e = getenv("F3S_SLICE_PHASES");  // read per call: tests walk through the phases
  const int forced = e ? atoi(e) : 0;
  const int units = heads_in_pairs(d, heads) ? heads / 2 : heads;  // that a window and slice are
  if (forced > 0) return {forced > kMaxPhases ? kMaxPhases : forced, kXcds, 1, 1, units, 1};
  const int dUnit = heads / units * d;  // columns of a row that a unit gathers
  XcdSplit s = split_heads(dUnit, units);
  const int64_t nRW = (N + kWinRows - 1) / kWinRows;
  // K + V of a group's heads
  const int64_t bytes = (int64_t)N * dUnit * s.headsPerGroup * 4;
  const int64_t most = nTcb < 0 && dUnit > 32 ? slice_bytes(64) : slice_bytes(dUnit);
  int64_t need = (bytes + most - 1) / most;
  if (nTcb >= 0 && nRW > 0) {  // (weight / 100) sqrt(blocks per window), rounded
    int64_t worth = 2;
    while ((2 * worth + 1) * (2 * worth + 1) * 2500 * nRW <= slice_weight(dUnit) * slice_weight(dUnit) * nTcb)
      worth++;
    if (need > worth) need = worth;
  }
  if (need < 2) need = 2;  // one unit per window would be the windows themselves
  // Slices one after the other keep all XCDs on the same columns at a time, which the memory side
  // serves faster (100k nodes, 4 x 128: 1.77 -> 1.67 ms; 60k nodes, 4 x 64: 0.87 -> 0.82 ms), as
  // long as a phase has units for two rounds of waves; with fewer the second phase's heavy windows
  // start when the first phase's light ones should fill the end (60k nodes, d = 32: 188 -> 206 us).
  // The slices at a time are a power of two, the nearest one rather than the next (50k nodes, d = 96:
  // 123 us with 4 slices, 146 with 8).
  const int64_t waves = 32 * 4 * unit_waves_per_simd(dUnit);  // of one XCD
  if (s.units(nRW) < 2 * waves) {
    while (s.windowGroups > 1 && (nTcb < 0 ? s.sliceGroups < need : 3 * s.sliceGroups <= 2 * need)) {
      s.sliceGroups *= 2;
      s.windowGroups /= 2;
    }
  }
  int64_t phases = (need + (nTcb < 0 ? s.sliceGroups - 1 : s.sliceGroups / 2)) / s.sliceGroups;
  if (phases < 1) phases = 1;
  s.phases = phases > kMaxPhases ? kMaxPhases : (int)phases;
  return s;
}

// The same slices for the resident form. Its waves move on to the next phase one by one, so an XCD's
// L2 has to hold two slices while they do: as few phases as the slices divide into evenly, the XCDs on
// different slices instead. (Unevenly some XCDs would have nothing to do in the last phase: 3 slices in
// groups of 4 0.48 instead of 0.43 ms.) 233k-node graph, d = 64, 8 slices: 1.82 -> 1.58 ms; 34k nodes,
// 8 x 32, 2 slices: 1.27 -> 1.16 ms.
XcdSplit resident_split(XcdSplit s) {
  while (s.windowGroups > 1 && s.phases % 2 == 0) {
    s.sliceGroups *= 2;
    s.windowGroups /= 2;
    s.phases /= 2;
  }
  return s;
}

size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

// byte offsets of the parts of the workspace
struct SlicedLayout {
  XcdSplit split;
  int S;
  size_t tickets, sliceStart, partial, total;
  size_t padded;  // 0, or where the copies of K and V with 256-byte rows start (single head, d = 64)
};
// nHeads = 0: the single-head layout. nTcb < 0: the largest that any structure of N nodes asks for.
SlicedLayout sliced_layout(int N, int d, int nHeads, int64_t nTcb) {
  const int heads = nHeads > 0 ? nHeads : 1;
  SlicedLayout L;
  L.split = choose_split(N, d, heads, nTcb);
  L.S = L.split.slices();
  const size_t nRW = (size_t)(N + kWinRows - 1) / kWinRows;
  L.tickets = 256;
  L.sliceStart = L.tickets + 256;
  L.partial = L.sliceStart + align256(nRW * (L.S + 1) * sizeof(int32_t));
  L.total = align256(L.partial + nRW * heads * L.S * (size_t)(16 * d + 32) * sizeof(float));
  L.padded = 0;
  if (nHeads == 0 && d == 64) {
    L.padded = L.total;
    L.total += 2 * (size_t)N * kPaddedRowBytes;
  }
  return L;
}

bool padded_rows_requested() {
  const char* e = getenv("F3S_PAD_ROWS");  // read per call; 0 switches the copies off
  return !(e && e[0] == '0');
}

// workgroups of NW waves the GPU holds at once (LDS rings, waves per SIMD), a multiple of 8
template <int D, int NW>
int resident_grid(int* grid) {
  constexpr int kMaxDev = 64;
  static int cusOf[kMaxDev] = {};
  int dev = 0;
  F3S_HIP_CHECK(hipGetDevice(&dev));
  int cus = (dev >= 0 && dev < kMaxDev) ? cusOf[dev] : 0;
  if (cus == 0) {
    F3S_HIP_CHECK(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    if (dev >= 0 && dev < kMaxDev) cusOf[dev] = cus;
  }
  // the rings plus the 1 KiB the two control words cost in front of the 1 KiB-aligned rings
  constexpr size_t lds = (size_t)NW * pipe::Geo<D, unit_stages(D)>::WAVE_BYTES + 1024;
  int perCu = (int)((160 * 1024) / lds);
  const int byWaves = unit_waves_per_simd(D) * 4 / NW;
  if (perCu > byWaves) perCu = byWaves;
  if (perCu < 1) perCu = 1;
  int gsz = cus * perCu / kXcds * kXcds;
  if (gsz < kXcds) gsz = kXcds;
  *grid = gsz;
  return 0;
}

bool resident_requested() {
  const char* e = getenv("F3S_SLICED_PERSISTENT");  // read per call
  return e && e[0] == '1';
}

template <typename ET, int D, bool SOFTMAX, bool HEADS, int NH = 1>
int launch_sliced_units(const int32_t* rwo, const int32_t* order, const int32_t* atox,
                        const uint8_t* bm, int N, int nRW, const ET* Q, const ET* K, const ET* V,
                        float scaleLog2, float* out, int32_t* tickets, int32_t* sliceStart,
                        float* partial, const SlicedLayout& L, int heads, int ldIn, int ldOut,
                        int64_t nTcb, hipStream_t stream, int ldQ = 0) {
  constexpr size_t lds = (size_t)kUnitWaves * pipe::Geo<D, unit_stages(D)>::WAVE_BYTES;
  if (resident_requested()) {
    auto kernel = f3s_fwd_resident_kernel<ET, D, SOFTMAX, HEADS, kUnitWaves, NH>;
    if (int rc = allow_lds(kernel, lds)) return rc;
    int grid = 0;
    if (int rc = resident_grid<D, kUnitWaves>(&grid)) return rc;
    hipLaunchKernelGGL(kernel, dim3((unsigned)grid), dim3(kUnitWaves * 64), lds, stream, order,
                       sliceStart, resident_split(L.split), nRW, N, nTcb, tickets, atox, bm, Q, K, V, scaleLog2,
                       partial, heads, ldIn);
  } else {
    auto kernel = f3s_fwd_unit_kernel<ET, D, SOFTMAX, HEADS, NH>;
    if (int rc = allow_lds(kernel, lds)) return rc;
    const int64_t nGroups = (L.split.units(nRW) + kUnitWaves - 1) / kUnitWaves;
    const int64_t grid = L.split.phases * nGroups * kXcds;
    if (grid >= ((int64_t)1 << 31))
      return fail(-2, "f3s_attention: too many (window, slice, head) units for one launch");
    hipLaunchKernelGGL(kernel, dim3((unsigned)grid), dim3(kUnitWaves * 64), lds, stream, order,
                       atox, bm, sliceStart, L.split, (int)nGroups, N, nRW, nTcb, Q, K, V, scaleLog2,
                       partial, heads, ldIn, ldQ);
  }
  F3S_HIP_CHECK(hipGetLastError());
  return 0;
}

template <typename ET, int D, bool SOFTMAX>
int launch_sliced_d(const int32_t* rwo, const int32_t* order, const int32_t* atox,
                    const uint64_t* bitmap, int N, const void* Q, const void* K, const void* V,
                    float scaleLog2, float* out, char* ws, const SlicedLayout& L, int nHeads,
                    int ldIn, int ldOut, int mode, int64_t nTcb, hipStream_t stream) {
  const int nRW = (N + kWinRows - 1) / kWinRows;
  const int S = L.S;
  const int sliceWidth = (N + S - 1) / S;
  const int heads = nHeads > 0 ? nHeads : 1;
  auto* hdr = reinterpret_cast<SlicedHeader*>(ws);
  auto* tickets = reinterpret_cast<int32_t*>(ws + L.tickets);
  auto* sliceStart = reinterpret_cast<int32_t*>(ws + L.sliceStart);
  auto* partial = reinterpret_cast<float*>(ws + L.partial);
  const unsigned setupBlocks = (unsigned)(((int64_t)nRW * 16 + 255) / 256);
  // copies of K and V with 256-byte rows, gathered through the pitched (multi-head) form of the
  // unit kernel with one head; Q stays where it is
  const bool padded = mode != 1 && nHeads == 0 && L.padded != 0 && padded_rows_requested() &&
                      !resident_requested() &&
                      !gather_needs_wide_offsets(N, kPaddedRowBytes, true);
  auto* kp = padded ? reinterpret_cast<ET*>(ws + L.padded) : nullptr;
  auto* vp = padded ? kp + (size_t)N * (kPaddedRowBytes / sizeof(ET)) : nullptr;
  const int64_t chunks = padded ? (int64_t)N * (D * (int)sizeof(ET) / 16) : 0;
  hipLaunchKernelGGL(sliced_setup_kernel, dim3(setupBlocks + (unsigned)((chunks + 255) / 256)),
                     dim3(256), 0, stream, rwo, atox, N, nRW, S, sliceWidth, nTcb, hdr, mode,
                     tickets, sliceStart, (int)setupBlocks, static_cast<const pad_chunk*>(K),
                     static_cast<const pad_chunk*>(V), chunks, reinterpret_cast<pad_chunk*>(kp),
                     reinterpret_cast<pad_chunk*>(vp));
  F3S_HIP_CHECK(hipGetLastError());
  if (mode == 1) return 0;
  const auto* bm = reinterpret_cast<const uint8_t*>(bitmap);
  const auto* q = static_cast<const ET*>(Q);
  const auto* k = static_cast<const ET*>(K);
  const auto* v = static_cast<const ET*>(V);
  int rc;
  if (D == 32 && heads_in_pairs(D, nHeads)) {
    rc = launch_sliced_units<ET, D == 32 ? 64 : D, SOFTMAX, true, D == 32 ? 2 : 1>(
        rwo, order, atox, bm, N, nRW, q, k, v, scaleLog2, out, tickets, sliceStart, partial, L, heads,
        ldIn, ldOut, nTcb, stream);
  } else if (nHeads > 0) {
    rc = launch_sliced_units<ET, D, SOFTMAX, true>(rwo, order, atox, bm, N, nRW, q, k, v,
                                                   scaleLog2, out, tickets, sliceStart, partial, L,
                                                   heads, ldIn, ldOut, nTcb, stream);
  } else if (padded) {
    rc = launch_sliced_units<ET, D, SOFTMAX, true>(
        rwo, order, atox, bm, N, nRW, q, kp, vp, scaleLog2, out, tickets, sliceStart, partial, L, 1,
        kPaddedRowBytes / (int)sizeof(ET), D, nTcb, stream, D);
  } else {
    rc = launch_sliced_units<ET, D, SOFTMAX, false>(rwo, order, atox, bm, N, nRW, q, k, v,
                                                    scaleLog2, out, tickets, sliceStart, partial,
                                                    L, 1, D, D, nTcb, stream);
  }
  if (rc != 0) return rc;
  const int64_t merges = (int64_t)nRW * heads;
  auto merge = f3s_merge_slices_kernel<D, SOFTMAX>;
  constexpr size_t mergeLds = (size_t)4 * rows_lds_floats<D>() * sizeof(float);
  if ((rc = allow_lds(merge, mergeLds)) != 0) return rc;
  hipLaunchKernelGGL(merge, dim3((unsigned)((merges + 3) / 4)), dim3(256), mergeLds, stream, sliceStart, S, N, nRW, heads, partial, out,
                     nHeads > 0 ? ldOut : D);
  F3S_HIP_CHECK(hipGetLastError());
  return 0;
}

}  // namespace

size_t attention_sliced_workspace_bytes(int N, int d, int nHeads) {
  return sliced_layout(N, d, nHeads, -1).total;
}

// mode 0 / 2: an attention call (2: on a prepared workspace); mode 1: f3s_attention_prepare
// (index only, Q/K/V/out unused)
int launch_attention_sliced(const int32_t* rowWindowOffset, const int32_t* windowOrder,
                            const int32_t* sparseAToXidx, const uint64_t* bitmap, int N, int d,
                            int dtype, const void* Q, const void* K, const void* V,
                            float scaleLog2, int applySoftmax, float* out, void* workspace,
                            size_t wsBytes, int64_t nTcb, int nHeads, int ldIn, int ldOut,
                            int mode, hipStream_t stream) {
  if (!head_dim_supported(d))
    return fail(-2, "f3s_attention: head dim %d unsupported (a multiple of 32 up to 256)", d);
  const SlicedLayout L = sliced_layout(N, d, nHeads, nTcb);
  if (wsBytes < L.total)
    return fail(-2, "f3s_attention: workspace %zu B < required %zu B", wsBytes, L.total);
  char* ws = static_cast<char*>(workspace);
#define F3S_SLICED(DD)                                                                         \
  if (d == DD) {                                                                               \
    if (dtype == 0)                                                                            \
      return applySoftmax ? launch_sliced_d<_Float16, DD, true>(                               \
                                rowWindowOffset, windowOrder, sparseAToXidx, bitmap, N, Q, K,  \
                                V, scaleLog2, out, ws, L, nHeads, ldIn, ldOut, mode,     \
                                nTcb, stream)                                                  \
                          : launch_sliced_d<_Float16, DD, false>(                              \
                                rowWindowOffset, windowOrder, sparseAToXidx, bitmap, N, Q, K,  \
                                V, scaleLog2, out, ws, L, nHeads, ldIn, ldOut, mode,     \
                                nTcb, stream);                                                 \
    return applySoftmax ? launch_sliced_d<__bf16, DD, true>(                                   \
                              rowWindowOffset, windowOrder, sparseAToXidx, bitmap, N, Q, K, V, \
                              scaleLog2, out, ws, L, nHeads, ldIn, ldOut, mode, nTcb,    \
                              stream)                                                          \
                        : launch_sliced_d<__bf16, DD, false>(                                  \
                              rowWindowOffset, windowOrder, sparseAToXidx, bitmap, N, Q, K, V, \
                              scaleLog2, out, ws, L, nHeads, ldIn, ldOut, mode, nTcb,    \
                              stream);                                                         \
  }
  F3S_FOR_EACH_HEAD_DIM(F3S_SLICED)
#undef F3S_SLICED
  return fail(-2, "f3s_attention: head dim %d unsupported (a multiple of 32 up to 256)", d);
}

}  // namespace f3s
