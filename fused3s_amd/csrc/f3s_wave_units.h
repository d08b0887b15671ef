// What the kernels with a wave per unit of work share (f3s_attention_units.hip, f3s_attention_mixed.hip): how
// units are dealt to the XCDs, the problem description for the pipeline, and a window's rows from the registers
// of one wave to memory.
#pragma once
#include "f3s_common.h"
#include "f3s_pair_pipeline.h"

namespace f3s {
namespace {

using pipe::float4v;
using pipe::uniform;

template <typename ET, int D, bool HEADS>
__device__ __forceinline__ pipe::Problem<ET> make_problem(const int32_t* sparseAToXidx,
                                                          const uint8_t* bitmapBytes, const ET* Q,
                                                          const ET* K, const ET* V, int N,
                                                          float scaleLog2, int ldIn,
                                                          int64_t nTcb, int ldQ = 0) {
  pipe::Problem<ET> pb;
  pb.sparseAToXidx = sparseAToXidx;
  pb.bitmapBytes = bitmapBytes;
  pb.Q = Q;
  pb.K = K;
  pb.V = V;
  pb.N = N;
  pb.scaleLog2 = scaleLog2;
  pb.pitchIn = HEADS ? ldIn : D;
  pb.pitchQ = (HEADS && ldQ > 0) ? ldQ : pb.pitchIn;  // Q may lie apart from K / V
  pb.nTcb = nTcb;
  pb.sddmm = nullptr;
  return pb;
}

// How the units of a call are dealt to the XCDs. XCD x works on one column slice of one group of
// heads at a time, for its share of the order's positions:
//   x = sg + sliceGroups * (hg + headGroups * wg), slice = phase * sliceGroups + sg,
//   heads hg * headsPerGroup .. + headsPerGroup - 1,
//   positions [wg * chunk, (wg + 1) * chunk) of every run of windowGroups * chunk positions.
struct Unit {
  int pos, head, slice;
};
struct XcdSplit {
  int phases;         // slices an XCD works through, one after the other
  int sliceGroups;    // slices in work at a time; sliceGroups * headGroups * windowGroups == 8
  int headGroups;
  int windowGroups;
  int headsPerGroup;
  int chunk;
  __host__ __device__ int slices() const { return phases * sliceGroups; }
  // units of one XCD and phase
  __host__ __device__ int64_t units(int nRW) const {
    const int64_t run = (int64_t)windowGroups * chunk;
    return ((int64_t)nRW + run - 1) / run * chunk * headsPerGroup;
  }
  // u-th unit of the XCD in the phase: heads innermost (they share ids, bitmaps and lines)
  __device__ __forceinline__ Unit unit(int xcd, int phase, unsigned u) const {
    const int sg = xcd & (sliceGroups - 1);  // the group counts are powers of two
    const int rest = xcd / sliceGroups;
    const int hg = rest & (headGroups - 1);
    const int wg = rest / headGroups;
    const unsigned p = u / (unsigned)headsPerGroup;
    const unsigned run = p / (unsigned)chunk;
    Unit r;
    r.pos = (int)((run * windowGroups + wg) * chunk + (p - run * chunk));
    r.head = hg * headsPerGroup + (int)(u - p * headsPerGroup);
    r.slice = phase * sliceGroups + sg;
    return r;
  }
};

// Head groups come first: an XCD that works on some of the heads gathers only their part of the
// rows, so its share of K + V shrinks without cutting windows into more units. The part stays at
// least a line of 128 bytes.
inline XcdSplit split_heads(int d, int heads) {
  const int groups = head_groups(d, heads);
  return {1, 1, groups, kXcds / groups, heads / groups, 1};
}

// A window's 16 rows of D floats from the lanes' O^T tiles (already normalised) to memory, through
// `lds` of the wave (rows_lds_floats<D>() floats): stored as the lanes hold them, a row would leave
// in pieces of 64 bytes; this way a store instruction fills whole lines.
template <int D>
constexpr int rows_lds_floats() {
  return 16 * (D + 4);
}
template <int D>
__device__ __forceinline__ void store_rows(const float4v (&o)[D / 16], float* lds, int w, int N,
                                           float* __restrict__ out, int ldOut) {
  constexpr int LPR = D / 4;  // lanes per row, 16 bytes each
  int lane = threadIdx.x & 63;
  pipe::pin(lane);
  const int g = lane >> 4, c = lane & 15;
#pragma unroll
  for (int j = 0; j < D / 16; j++)
    *reinterpret_cast<float4v*>(lds + c * (D + 4) + 16 * j + 4 * g) = o[j];
  __builtin_amdgcn_wave_barrier();
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
  for (int k = 0; k < 16 * LPR / 64; k++) {
    const int q = (k * 64 + lane) / LPR, cv = (k * 64 + lane) % LPR;
    const int64_t row = (int64_t)w * 16 + q;
    if (row < N)
      store_out(out + row * ldOut + cv * 4,
                *reinterpret_cast<const float4v*>(lds + q * (D + 4) + cv * 4));
  }
}

}  // namespace
}  // namespace f3s
