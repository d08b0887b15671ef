// Attention on graphs of short windows (gfx950): a wave per window and, in the same launch, a workgroup per
// long one. The step over a TC-block pair is the one every attention kernel here runs (f3s_pair_pipeline.h).
//
// The reference has no counterpart: its kernels (src/F3S_kernel.cu:1371-1583) give every window a thread
// block. Its window order (src/utils.cu:400-436) is kept: it says which windows start first.
#include "f3s_common.h"
#include "f3s_pair_pipeline.h"
#include "f3s_wave_units.h"

namespace f3s {
namespace {

// Stages of a wave's LDS ring, and waves per SIMD the register allocator is held to: as many as the rings leave room
// for in a CU's LDS, 16 up to D = 64, eight up to D = 128, four above. Two stages fit 16 waves at D = 32, where 20
// of one stage leave a long window's four waves waiting for every step's rows. One head, d = 32, 20 waves of one
// stage -> 16 of two (a launch for each kind of window), us; nodes, blocks a window: power-law 110 000, 15 49 -> 41
// (47), 200 000, 7 69 -> 55 (64), 11 81 -> 67 (74); R-MAT 46 000, 12 20 -> 17 (24), 200 000, 13 66 -> 54 (64), 600 000, 15 220
// -> 187 (221); communities 200 000, 9 28 -> 27 (35); uniform 110 000, 11 34 -> 36 (36), 15 42 -> 46 (43); three heads of
// 200 000 nodes, power-law, 11 142 -> 130 (151), R-MAT, 9 93 -> 97 (108), uniform, 11 171 -> 172 (171).
constexpr int mixed_stages(int d) { return d == 32 ? 2 : 1; }
constexpr int mixed_waves_per_simd(int d) { return d <= 64 ? 4 : d <= 128 ? 2 : 1; }

// Waves of a workgroup, four or eight. Eight compute a long window in half the time, and the longest one decides a
// call of one or two heads on a skewed graph. A wave that has finished its own window keeps its ring until the
// workgroup ends, which costs less with four, so those take calls of more heads and, above D = 64, of two, large
// ones and those whose last round of waves would be less than half full. Eight -> four, us (heads x d, blocks a
// window): R-MAT 40 000 nodes, 12: 1 x 64 34 -> 38, 2 x 64 40 -> 43, 4 x 64 57 -> 52, 8 x 64 100 -> 93, 4 x 128 106 -> 92;
// 169 343 nodes, 17: 1 x 64 76 -> 95; 200 000, 27: 1 x 64 111 -> 143, 1 x 128 241 -> 253, 8 x 64 1063 -> 1050; 600 000, 20: 1 x 64
// 294 -> 326, 1 x 128 648 -> 628; uniform 25 000, 9: 1 x 64 25.7 -> 25.5, 8 x 64 70 -> 66; 30 000, 21: 1 x 128 45.7 -> 46.1, 8 x 64
// 128 -> 133; 33 000, 15: 2 x 128 66 -> 59; R-MAT 65 000, 14: 2 x 128 78 -> 71.
// Rounds: at D = 96 and 128 a workgroup of eight waves fills a CU and 2 048 windows the chip. One window more, and a
// uniform graph takes another round of which a CU or two do anything. Below 16 blocks a window, 1 x 128: uniform 33 000
// nodes (2 063 windows), 15: 40 -> 33 (with a launch for either kind of window 33); 66 000 (4 125), 11: 0.89 of those two
// launches -> 1.01; 46 000 (2 875), 15: 0.92 -> 1.01; 50 000 (3 125): 1.01 -> 1.01; R-MAT 33 000, 14 1.50 -> 1.32, 54 000, 11 1.47 -> 1.19;
// power-law 66 000, 11 1.39 -> 1.19.
// A long window is cut into as many runs of blocks whether four or eight waves compute them, so that a head's
// rows do not depend on how many heads the call has. With two heads of 32 to a wave there are always four of
// each, as what four waves keep of the first four runs would not fit the registers there, and so at D = 32, whose
// rows are those of the pairs.
constexpr int mixed_runs(int d, int nh) { return d == 32 || nh == 2 || d > 128 ? 4 : 8; }
inline int mixed_waves(int d, bool w8, int nRW, int64_t nTcb16, int heads) {
  if (heads >= 3) return 4;
  if (d <= 64) return 8;
  if (heads == 2 || nTcb16 >= 500000) return 4;
  constexpr int kRound = 256 * 8;
  const bool below16 = !w8 && nTcb16 < 16 * (int64_t)nRW;
  return below16 && nRW > kRound && nRW < 3 * kRound && (nRW - 1) % kRound < kRound / 2 ? 4 : 8;
}

// How the (position, head) units of a call are dealt to the XCDs: XcdSplit with one slice and with shifts in the
// place of most divisions, which stand in front of a wave's first load.
struct WaveSplit {
  int headGroups, windowGroups;  // powers of two, 8 together
  int headsPerGroup, headShift;  // headShift: its logarithm, or -1
  int chunkShift;                // positions an XCD takes in a row
  __host__ __device__ int64_t units(int nRW) const {
    const int64_t run = (int64_t)windowGroups << chunkShift;
    return (((int64_t)nRW + run - 1) / run << chunkShift) * headsPerGroup;
  }
  __device__ __forceinline__ Unit unit(int group, int groupUnits, int k) const {
    const int xcd = group % kXcds;
    const unsigned u = (unsigned)(group / kXcds) * groupUnits + k;
    const unsigned p = headShift >= 0 ? u >> headShift : u / (unsigned)headsPerGroup;
    const unsigned run = p >> chunkShift;
    Unit r;
    r.pos = (int)(((run * windowGroups + xcd / headGroups) << chunkShift) + (p - (run << chunkShift)));
    r.head = (xcd & (headGroups - 1)) * headsPerGroup + (int)(u - p * headsPerGroup);
    r.slice = 0;
    return r;
  }
};

// Workgroups of two kinds.
//   teams   the first teamGroups of the grid look through all positions of the order, a thread per (position,
//           head) unit, and compute the windows of more than maxBlocks TC blocks that they find, one after the
//           other with all of their waves. In a heavy-first order those are its first positions, and they
//           are dealt round-robin; in any other they start first all the same. (Looked for among as many positions
//           as there can be long windows, those of other orders were left to single waves: d = 64, R-MAT 169 343
//           nodes, 17 blocks a window, longest 759, natural order given as the order: 218 us, now 86.)
//   others  a wave takes a whole window (of one head, or of NH) that is not a long one and writes its rows from
//           its registers.
// Where the order's first window has at most evenBlocks, all have if the order is heavy-first: evenTeams are then
// enough to look, the other teams leave, and the waves take the windows in natural order instead of the given
// one, 1 << evenShift in a row to an XCD. Windows that follow each other in a graph of communities name the same
// rows, of which a heavy-first order makes as many visits as there are block counts (100 000 nodes, 6 blocks a
// window, 8 x 32: 74 us in the given order, 58); and when the longest window is little more than twice the mean, it
// does not matter which one starts last. It does where one of four times the mean is short all the same (R-MAT
// 33 000 nodes, 7 blocks, longest 32, d = 256: 48 us, heavy-first 40). An order that ends in an entry out of range, or
// twice in the same one, names some of the windows and is filled up: it is followed as it stands.
// W8: 16x8 blocks, with the scores to sddmm if it is not null; maxBlocks and nTcb then count such blocks.
template <typename ET, int D, int NWAVES, bool SOFTMAX, bool HEADS, bool W8, int NH = 1>
__global__ __launch_bounds__(NWAVES * 64)
__attribute__((amdgpu_waves_per_eu(mixed_waves_per_simd(D), mixed_waves_per_simd(D)))) void
f3s_fwd_mixed_kernel(const int32_t* __restrict__ windowOrder,
                     const int32_t* __restrict__ rowWindowOffset,
                     const int32_t* __restrict__ sparseAToXidx,
                     const uint8_t* __restrict__ bitmapBytes, WaveSplit split, int evenShift,
                     int teamGroups, int evenTeams, int evenBlocks, int maxBlocks, int N, int nRW, int64_t nTcb,
                     const ET* __restrict__ Q, const ET* __restrict__ K, const ET* __restrict__ V,
                     float scaleLog2, float* __restrict__ out, int nHeads, int ldIn, int ldOut,
                     float* __restrict__ sddmm) {
  constexpr int WAVE_BYTES = pipe::Geo<D, mixed_stages(D)>::WAVE_BYTES;
  typedef pipe::PairPipeline<ET, D, SOFTMAX, HEADS, W8, mixed_stages(D), false, NH> Pipe;
  constexpr int TH = D / NH / 16;
  constexpr int BPS = W8 ? 4 : 2;  // blocks of the structure per step
  // four waves take eight runs in two turns
  constexpr int RUNS = mixed_runs(D, NH), TURNS = RUNS / NWAVES;
  extern __shared__ __align__(1024) unsigned char smem[];
  __shared__ int sList[NWAVES * 64];
  __shared__ int sFound;
  const int wave = uniform(threadIdx.x >> 6);
  const int pitchOut = HEADS ? ldOut : D;
  // block ranges that do not fit the structure (a mismatched rowWindowOffset) are not followed: such a window
  // is treated as empty, and so is one that does not exist (a corrupt order entry must not index out of range).
  // An end in front of the begin is looked at before the two are subtracted: the difference may not fit.
  const auto fits = [&](int t0, int t1) { return t0 >= 0 && t1 >= t0 && (int64_t)t1 <= nTcb; };
  const auto is_long = [&](int t0, int t1) { return fits(t0, t1) && t1 - t0 > maxBlocks; };

  // Where this wave stands in the given and in natural order, and what it will ask for, in two rounds of loads.
  const int waveGroups = (int)gridDim.x - teamGroups;
  const Unit given = split.unit(max((int)blockIdx.x - teamGroups, 0), NWAVES, wave);
  WaveSplit evenSplit = split;
  evenSplit.chunkShift = evenShift;
  const Unit natural = evenSplit.unit(max((int)blockIdx.x - evenTeams, 0), NWAVES, wave);
  int firstWindow = -1, nextToLast = -1, lastWindow = -1, givenWindow = given.pos;
  if (windowOrder) {
    firstWindow = windowOrder[0];
    nextToLast = windowOrder[nRW - 2];
    lastWindow = windowOrder[nRW - 1];
    givenWindow = windowOrder[min(given.pos, nRW - 1)];
  }
  const int natural0 = rowWindowOffset[min(natural.pos, nRW - 1)];
  const int natural1 = rowWindowOffset[min(natural.pos, nRW - 1) + 1];
  asm volatile("" : : "s"(firstWindow), "s"(nextToLast), "s"(lastWindow), "s"(givenWindow), "s"(natural0), "s"(natural1));
  const int first = (unsigned)firstWindow < (unsigned)nRW ? firstWindow : 0;
  const int most = rowWindowOffset[first + 1] - rowWindowOffset[first];
  const int ask = (unsigned)givenWindow < (unsigned)nRW ? givenWindow : 0;
  const int given0 = rowWindowOffset[ask], given1 = rowWindowOffset[ask + 1];
  asm volatile("" : : "s"(most), "s"(given0), "s"(given1));
  const bool filledUp =
      (unsigned)nextToLast >= (unsigned)nRW || (unsigned)lastWindow >= (unsigned)nRW || nextToLast == lastWindow;
  const bool even = firstWindow == first && most <= evenBlocks && !filledUp;
  const int teams = even ? evenTeams : teamGroups;
  const bool team = (int)blockIdx.x < teams;
  if (even && (int)blockIdx.x >= evenTeams + waveGroups) return;

  int found = 0;  // units of a team in sList
  if (team) {
    if (threadIdx.x == 0) sFound = 0;
    __syncthreads();
    const int64_t u = (int64_t)blockIdx.x + (int64_t)threadIdx.x * teams;
    if (u < (int64_t)nRW * nHeads) {
      const int pos = (int)(u / nHeads), w = windowOrder && !even ? windowOrder[pos] : pos;
      if ((unsigned)w < (unsigned)nRW && is_long(rowWindowOffset[w], rowWindowOffset[w + 1]))
        sList[atomicAdd(&sFound, 1)] = (int)u;
    }
    __syncthreads();
    found = uniform(sFound);
  }
  pipe::Problem<ET> pb =
      make_problem<ET, D, HEADS>(sparseAToXidx, bitmapBytes, Q, K, V, N, scaleLog2, ldIn, nTcb);
  pb.sddmm = sddmm;
  unsigned char* const ring = smem + wave * WAVE_BYTES;
  pipe::MergedRows<D, NWAVES, SOFTMAX, NH> firstRuns;
  const int turns = team ? found * TURNS : 1;
  for (int k = 0; k < turns; k++) {
    int w, head = 0, t0, t1;
    if (team) {
      const int u = uniform(sList[k / TURNS]);
      const int pos = HEADS ? u / nHeads : u;
      if constexpr (HEADS) head = u - pos * nHeads;
      w = uniform(windowOrder && !even ? windowOrder[pos] : pos);
      const int from = rowWindowOffset[w], to = rowWindowOffset[w + 1];
      // run r: steps [r * nSteps / RUNS, (r + 1) * nSteps / RUNS)
      const int nSteps = (to - from + BPS - 1) / BPS, r = k % TURNS * NWAVES + wave;
      t0 = from + BPS * (int)((int64_t)r * nSteps / RUNS);
      t1 = min(from + BPS * (int)((int64_t)(r + 1) * nSteps / RUNS), to);
    } else {
      w = even ? natural.pos : givenWindow;
      t0 = even ? natural0 : given0;
      t1 = even ? natural1 : given1;
      if constexpr (HEADS) head = even ? natural.head : given.head;
      if ((even ? natural.pos : given.pos) >= nRW || (unsigned)w >= (unsigned)nRW) return;
      if (is_long(t0, t1)) return;  // a team's
      if (!fits(t0, t1)) t1 = t0;
    }
    Pipe pp;
    pp.init(pb, w, (unsigned)(uintptr_t)(F3S_LDS unsigned char*)ring, head);
    pp.run(pb, t0, t1);
    float* const dst = out + head * D;
    if (team) {
      pipe::put_partials<D, NWAVES, SOFTMAX, NH>(pp, smem, wave);
      pipe::MergedRows<D, NWAVES, SOFTMAX, NH> rows;
      rows.merge(smem, 0);
      if constexpr (NWAVES == 8) {
        firstRuns = rows;
        rows.merge(smem, 4);
      }
      if (k % TURNS < TURNS - 1) {
        firstRuns = rows;
      } else {
        if constexpr (RUNS == 8) {
          firstRuns.add(rows);
          firstRuns.store(w, N, dst, pitchOut);
        } else {
          rows.store(w, N, dst, pitchOut);
        }
      }
      __syncthreads();  // the merge buffers are free again
    } else {
#pragma unroll
      for (int h = 0; h < NH; h++) {
        float inv = 1.0f;
        if constexpr (SOFTMAX) {
          const float lAll = pipe::row_sum4(pp.l[h]);
          inv = (lAll == 0.0f) ? 0.0f : 1.0f / lAll;
        }
#pragma unroll
        for (int j = 0; j < TH; j++) pp.o[h * TH + j] *= inv;
      }
      // the wave's ring is free now
      static_assert(rows_lds_floats<D>() * 4 <= WAVE_BYTES, "rows fit the ring");
      store_rows<D>(pp.o, reinterpret_cast<float*>(ring), w, N, dst, pitchOut);
    }
  }
}

template <typename KernelT>
int allow_lds(KernelT kernel, size_t bytes) {  // above 64 KiB a kernel has to be told
  if (bytes > 64 * 1024)
    F3S_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                      hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes));
  return 0;
}

// Positions of the given order an XCD takes in a row (as a power of two): windows of equal block counts are in
// window order and often name the same rows, which then come from one L2. Of more in a row the first XCD
// would get too many of the heaviest.
constexpr int kOrderShift = 4;
// The same in natural order, of large enough graphs for every XCD to take sixteen such turns (100k-node
// community layer, 8 x 32: 8, 16, 32, 64 windows 86, 82, 79, 77 us; 60k nodes, 4 x 64: 60, 59, 56, 55).
constexpr int kEvenShift = 6;

// 32-wide heads are computed one by one where one or two pairs of them make too few waves to fill the CUs: a
// wave then takes longer for two heads than two waves for one each. Head by head against pairs, us; blocks of
// the graph. One pair: uniform 10 000 10.7 against 12.0, 19 000 14.1 15.7, 26 000 17.8 16.9, 29 000 18.3 17.2;
// communities 9 000 9.7 11.1, 31 000 17.1 17.7 or 19.3 18.6, 38 000 23.3 23.1; power-law 24 000 24.1 25.5, 40 000
// 32.1 33.0; R-MAT 13 000 18.6 22.5, 31 000 28.0 29.2, 37 000 29.6 30.9, 51 000 35.9 35.9, 69 000 44.4 42.7. Two
// pairs: uniform 10 000 14.7 15.3, 23 000 23.8 20.8; communities 9 000 12.9 14.0, 31 000 26.2 25.9; R-MAT 13 000
// 23.6 25.5, 23 000 31.9 32.6, 26 000 34.0 34.8, 31 000 41.0 39.0; power-law 24 000 30.0 31.0, 40 000 47.8 45.9.
// Three and more lose at most 3 % (four: R-MAT 13 000 30.9 31.7) and gain 1 to 25 % (three: communities 9 000
// 18.5 16.7; eight: uniform 6 000 28.7 26.5).
bool pairs_fill(int64_t nTcb, int pairs) { return pairs >= 3 || nTcb * pairs >= 50000; }

struct MixedCall {
  const int32_t *rwo, *order, *atox;
  const uint8_t* bitmap;
  int N, nHeads, ldIn, ldOut;  // nHeads = 0: contiguous [N, d] single head
  const void *Q, *K, *V;
  float scaleLog2;
  float *out, *sddmm;
  int64_t nTcb;  // blocks of the structure
  hipStream_t stream;
};

// NH = 2: D = 64 stands for two heads of 32
template <typename ET, int D, int NWAVES, bool SOFTMAX, bool HEADS, bool W8, int NH = 1>
int launch_mixed_waves(const MixedCall& c) {
  const int nRW = (c.N + kWinRows - 1) / kWinRows;
  const int heads = HEADS ? c.nHeads / NH : 1;
  // 9/4 of the mean, and 32 blocks of 16 columns at least, make a window a long one (24, 32, 48, 64, 96 blocks, us,
  // d = 64; R-MAT 40 000 nodes, 12 a window: 32, 33, 39, 41, 49; 19: 44, 42, 40, 48, 52; 60 000, 28: 73, 66, 62, 53, 55;
  // 200 000, 27: 121, 116, 109, 109, 111; d = 192 alike)
  const int64_t longer = (9 * c.nTcb + 4 * (int64_t)nRW - 1) / (4 * (int64_t)nRW);
  const int maxBlocks = (int)(longer > (W8 ? 64 : 32) ? longer : (W8 ? 64 : 32));
  const int evenBlocks = (int)(longer > (W8 ? 32 : 16) ? longer : (W8 ? 32 : 16));
  const int64_t longMax = c.order ? c.nTcb / (maxBlocks + 1) + 1 : nRW;
  WaveSplit split;
  split.headGroups = head_groups(D, heads);
  split.windowGroups = kXcds / split.headGroups;
  split.headsPerGroup = heads / split.headGroups;
  split.headShift = 0;
  while (1 << split.headShift < split.headsPerGroup) split.headShift++;
  if (1 << split.headShift != split.headsPerGroup) split.headShift = -1;
  split.chunkShift = kOrderShift;
  WaveSplit evenSplit = split;
  evenSplit.chunkShift = kEvenShift;
  while (evenSplit.chunkShift > kOrderShift && nRW < 16 * evenSplit.windowGroups << evenSplit.chunkShift)
    evenSplit.chunkShift--;
  const int64_t given = split.units(nRW), natural = evenSplit.units(nRW);
  const int64_t waveGroups = ((given > natural ? given : natural) + NWAVES - 1) / NWAVES * kXcds;
  // a quarter of the long windows that there can be, 256 to 2048, and at least a thread for each unit (256, 512, 1024,
  // 2048 teams, us, d = 64: R-MAT 40 000 nodes, 12 blocks a window: 32, 36, 35, 36; 19: 41, 37, 38, 44; 169 343, 17: 93, 84, 78,
  // 76; d = 32, 600 000, 15: 238, 222, 208, 195). 256 of them, or a thread for each unit, where the order names no
  // long window first (64, 128, 256, as many as ever, us: communities, 8 x 32 58.3, 58.1, 58.3, 60.1; R-MAT 169 343
  // in a shuffled order 183, 119, 86, 68), and half as many above D = 128, where they would keep every CU from its
  // first waves (R-MAT 100 000, 25 blocks, d = 160, shuffled: 191, 192, 192, 189).
  const int64_t units = (int64_t)nRW * heads;
  const int64_t longUnits = (longMax < nRW ? longMax : nRW) * heads;
  const auto at_least = [&](int64_t n) {
    const int64_t look = (units + NWAVES * 64 - 1) / (NWAVES * 64);
    return ((n > look ? n : look) + kXcds - 1) / kXcds * kXcds;
  };
  const int64_t teams = at_least(longUnits / 4 < 256 ? 256 : longUnits / 4 > 2048 ? 2048 : longUnits / 4);
  const int64_t evenTeams = at_least(D > 128 ? 128 : 256);
  if (waveGroups + teams >= ((int64_t)1 << 31))
    return fail(-2, "f3s_attention: too many (window, head) units for one launch");
  auto kernel = f3s_fwd_mixed_kernel<ET, D, NWAVES, SOFTMAX, HEADS, W8, NH>;
  constexpr size_t lds = (size_t)NWAVES * pipe::Geo<D, mixed_stages(D)>::WAVE_BYTES;
  if (int rc = allow_lds(kernel, lds)) return rc;
  hipLaunchKernelGGL(kernel, dim3((unsigned)(waveGroups + teams)), dim3(NWAVES * 64), lds, c.stream, c.order,
                     c.rwo, c.atox, c.bitmap, split, evenSplit.chunkShift, (int)teams, (int)evenTeams, evenBlocks,
                     maxBlocks, c.N, nRW, c.nTcb, static_cast<const ET*>(c.Q), static_cast<const ET*>(c.K),
                     static_cast<const ET*>(c.V), c.scaleLog2, c.out, heads, HEADS ? c.ldIn : D,
                     HEADS ? c.ldOut : D, c.sddmm);
  F3S_HIP_CHECK(hipGetLastError());
  return 0;
}

template <typename ET, int D, bool SOFTMAX, bool HEADS, bool W8, int NH = 1>
int launch_mixed_kernel(const MixedCall& c) {
  if constexpr (mixed_runs(D, NH) == 8) {
    const int nRW = (c.N + kWinRows - 1) / kWinRows;
    if (mixed_waves(D, W8, nRW, W8 ? c.nTcb / 2 : c.nTcb, HEADS ? c.nHeads / NH : 1) == 8)
      return launch_mixed_waves<ET, D, 8, SOFTMAX, HEADS, W8, NH>(c);
  }
  return launch_mixed_waves<ET, D, 4, SOFTMAX, HEADS, W8, NH>(c);
}

template <typename ET, int D, bool SOFTMAX>
int launch_mixed_d(const MixedCall& c) {
  if constexpr (D == 32) {
    if (heads_in_pairs(D, c.nHeads) && pairs_fill(c.nTcb, c.nHeads / 2))
      return launch_mixed_kernel<ET, 64, SOFTMAX, true, false, 2>(c);
  }
  return c.nHeads > 0 ? launch_mixed_kernel<ET, D, SOFTMAX, true, false>(c)
                      : launch_mixed_kernel<ET, D, SOFTMAX, false, false>(c);
}

}  // namespace

// Where this kernel takes a call (nTcb16: blocks of 16 columns; w8: of a structure of 16x8 blocks). Against a workgroup
// of four waves for every window, us, with an order, one head unless heads are given; nodes, blocks a window:
// - blocks of 16 columns, less than 16 a window, d <= 128: here. Communities 200 000, 14 d = 64 97 -> 57, d = 32 61 -> 32;
//   uniform 65 000, 7 d = 64 21 -> 19; R-MAT 110 000, 9 d = 128 68 -> 64; power-law 110 000, 15 d = 32 37 -> 41.
// - more of them and 16x8 blocks, d = 64 to 128: up to 32 a window, and where windows times heads (or pairs of 32-wide
//   heads) are 11/8 of the waves that fit the chip at a time. Below that line a window that one wave computes
//   lasts longer than all of the rest. d = 64, 5 632 of them: power-law 24 000, 16 15 -> 21, 27 18 -> 29; 46 000, 28 28 -> 32;
//   72 000, 27 42 -> 47; flat R-MAT 24 000, 28 15 -> 27; 72 000, 28 44 -> 48; but R-MAT 46 000, 17 30 -> 24; 72 000, 17 38 -> 31;
//   uniform 46 000, 17 27 -> 25. Beyond: power-law 90 000, 17 44 -> 41, 27 55 -> 54, 30 57 -> 58; 200 000, 28 132 -> 127; flat
//   R-MAT 90 000, 28 57 -> 57; R-MAT 90 000, 18 47 -> 37; 200 000, 31 132 -> 105; uniform 90 000, 28 81 -> 70. d = 128, 2 816:
//   power-law 24 000, 27 29 -> 45; 33 000, 17 30 -> 34; but R-MAT 33 000, 16 33 -> 31. Beyond: power-law 48 000, 17 43 -> 42,
//   27 57 -> 59; 200 000, 28 296 -> 287; uniform 200 000, 18 247 -> 254; 90 000, 28 177 -> 151; R-MAT 48 000, 26 59 -> 50.
//   16x8 blocks of the same graphs: d = 64, power-law 24 000, 7 13 -> 19; 110 000, 7 42 -> 35, 28 68 -> 72. Three heads and
//   more have workgroups of four waves here, which end sooner: all the waves that fit are enough (4 x 64: power-law
//   17 000, 16 28 -> 22, 27 36 -> 30; flat R-MAT 17 000, 28 35 -> 31). Nothing on the host tells uniform from power-law
//   graphs, which is why these stop at 32 blocks (power-law 20 000, 46 35 -> 41; 50 000, 47 57 -> 68; 100 000, 57 119 ->
//   120; but uniform 60 000, 60 106 -> 76).
// - the same at d = 32: pairs of heads, which are 64 wide, from two on (4 x 32: power-law 45 000, 17 39 -> 32; R-MAT 45 000, 29
//   48 -> 51; 110 000, 18 92 -> 73). One pair takes longer than window by window head for head (2 x 32: power-law 110 000, 17 53
//   -> 62; R-MAT 110 000, 26 70 -> 75; 33 000, 22 1.35 times), and so do single heads.
// - d > 128, where four waves were all that a CU held and a window's last step kept three of them waiting: up to 64
//   blocks a window. d = 192, R-MAT 40 000, 12 86 -> 63; 200 000, 27 521 -> 400; uniform 60 000, 60 (d = 224) 443 -> 273;
//   power-law 20 000, 46 90 -> 91; 60 000, 52 257 -> 213; 180 000, 48 762 -> 644. From 16 blocks on not the few windows above
//   d = 192 (1 025 windows, d = 256: power-law 54 blocks 74 -> 83, R-MAT 25 45 -> 47; 1 250: power-law 55 95 -> 96).
// - K + V of 1 GiB and more, which come from HBM as fast as it gives them, window by window: R-MAT 2 449 029, 25, d = 128
//   4398 against 4428.
// - without an order, on graphs of more windows than f3s_window_order takes: d = 192, flat R-MAT 1 000 000, 26 3300 -> 2820,
//   R-MAT 800 000, 15 2000 -> 1533, uniform 300 000, 17 670 -> 576; but d = 64, R-MAT 800 000, 15 466 -> 344, flat 300 000,
//   18 184 -> 195, 1 000 000, 26 904 -> 926, uniform 197 -> 204, d = 128 900 -> 729, 369 -> 394, 1780 -> 1820, 377 -> 388.
bool mixed_windows_pay(bool ordered, int nRW, int64_t nTcb16, int d, int nHeads, bool w8) {
  if (nRW < 1024) return false;
  const int heads = nHeads > 0 ? nHeads : 1;
  const bool pairs = heads_in_pairs(d, nHeads);
  const int64_t units = (int64_t)nRW * (pairs ? heads / 2 : heads);
  const bool below16 = nTcb16 < 16 * (int64_t)nRW;
  if (d > 128) {
    if (d > 192 && !below16 && units < 1200) return false;
    return nTcb16 < 64 * (int64_t)nRW && (ordered || nRW > 16384);
  }
  if (!ordered || (int64_t)nRW * kWinRows * d * heads * 4 >= (int64_t)1 << 30) return false;
  if (below16 && !w8) return true;
  if (d == 32 && !(pairs && heads >= 4)) return false;
  const int64_t fit = 256 * 4 * mixed_waves_per_simd(d);
  const bool fourWaves = (pairs ? heads / 2 : heads) >= 3;
  return nTcb16 < 32 * (int64_t)nRW && units >= (fourWaves ? fit : fit * 11 / 8);
}

int launch_attention_mixed(const int32_t* rowWindowOffset, const int32_t* windowOrder,
                           const int32_t* sparseAToXidx, const uint64_t* bitmap, int N, int d, int dtype,
                           const void* Q, const void* K, const void* V, float scaleLog2,
                           int applySoftmax, float* out, int nHeads, int ldIn, int ldOut,
                           int64_t nTcb, hipStream_t stream) {
  const MixedCall c = {rowWindowOffset, windowOrder, sparseAToXidx, reinterpret_cast<const uint8_t*>(bitmap), N,
                       nHeads, ldIn, ldOut, Q, K, V, scaleLog2, out, nullptr, nTcb, stream};
#define F3S_MIXED(DD)                                                                  \
  if (d == DD) {                                                                       \
    if (dtype == 0)                                                                    \
      return applySoftmax ? launch_mixed_d<_Float16, DD, true>(c)                      \
                          : launch_mixed_d<_Float16, DD, false>(c);                    \
    return applySoftmax ? launch_mixed_d<__bf16, DD, true>(c)                          \
                        : launch_mixed_d<__bf16, DD, false>(c);                        \
  }
  F3S_FOR_EACH_HEAD_DIM(F3S_MIXED)
#undef F3S_MIXED
  return fail(-2, "f3s_attention: head dim %d unsupported (a multiple of 32 up to 256)", d);
}

int launch_tcb8_mixed(const int32_t* rowWindowOffset, const int32_t* windowOrder,
                      const int32_t* sparseAToXidx, const uint64_t* bitmap, int N, int d,
                      const void* Q, const void* K, const void* V, float scaleLog2,
                      int applySoftmax, float* out, float* sddmm, int64_t nTcb8,
                      hipStream_t stream) {
  const MixedCall c = {rowWindowOffset, windowOrder, sparseAToXidx, reinterpret_cast<const uint8_t*>(bitmap), N,
                       0, d, d, Q, K, V, scaleLog2, out, sddmm, nTcb8, stream};
#define F3S_MIXED(DD)                                                                     \
  if constexpr (DD > 32) {                                                                \
    if (d == DD)                                                                          \
      return applySoftmax ? launch_mixed_kernel<_Float16, DD, true, false, true>(c)       \
                          : launch_mixed_kernel<_Float16, DD, false, false, true>(c);     \
  }
  F3S_FOR_EACH_HEAD_DIM(F3S_MIXED)
#undef F3S_MIXED
  return fail(-2, "f3s_attention_fwd_tcb8: head dim %d unsupported (a multiple of 32 up to 256)", d);
}

}  // namespace f3s
