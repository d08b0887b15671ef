// CSR -> 16-row windows of column-compacted TC blocks with per-block bitmaps, on gfx950.
//
// Replaces the reference's preprocessing pipeline (src/F3S.cpp:40-87, src/utils.cu:23-436):
// a global thrust::sort of (window, column) pairs followed by two kernels that walk each
// window with a single thread. Here a window never leaves its workgroup:
//
//   window_rank_bins_kernel / window_rank_small_kernel
//                        short windows, one WAVE per window, no workgroup barrier. Graphs of
//                        <= 2^22 nodes, windows of <= 960 edges: (column, position) words sorted by
//                        bins of LDS counters, ranks of the distinct columns back to the edges.
//                        Larger graphs, <= 1024 edges: bitonic sort of the column ids, ballot /
//                        popcount compaction of the distinct ones, rank by binary search.
//   window_rank_mid_kernel, window_rank_rest_kernel
//                        longer windows where the columns take several bitset passes, one workgroup
//                        per window: sorted by bins as well, above 16 384 edges by the bitset.
//   window_rank_kernel   larger windows, one workgroup per window. Column ids are OR-ed into an
//                        LDS bitset (a column range per pass when N exceeds the LDS range), a
//                        wave64 popcount prefix scan turns the bitset into ranks, and every edge
//                        reads its compacted column index back: the sorted unique column list
//                        (reference: sort + inplace_deduplication + binarysearch,
//                        src/utils.cu:102-153,281-289) is never materialised.
//   window_scan_kernel, finalize_count_kernel, finalize_*_kernel
//                        scan of the per-window block counts (src/utils.cu:293-300) and the windows
//                        by descending block count (src/utils.cu:400-436): places from a histogram
//                        of the counts, or on graphs of very many windows (and in the count / fill
//                        calls of graphs of many) a stable LSD radix sort.
//   window_rank_all_kernel, window_fill_all_kernel
//                        the two phases on graphs of up to 16384 windows that are not all long: the
//                        wave per short window, the workgroup per long one and the order of the
//                        windows side by side in one launch each.
//   window_count_kernel, window_rank_fill_kernel
//                        graphs of long windows through the one-call entry: block counts, then
//                        ranks, rows, ids, bitmaps and tile ids of a window while its bitset sits
//                        in LDS.
//   window_fill_kernel, window_fill_short_kernel, window_fill_long_kernel
//                        one workgroup (or one wave, for short windows) per window: bitmaps and
//                        per-(row, block) edge counts are accumulated in LDS, a scan yields the
//                        per-block offsets, and the tile ids are written per block from its bitmap
//                        when the window's rows ascend, else placed edge by edge in CSR order
//                        (src/utils.cu:173-224, 23-36, 53-65).
//
// All results are bit-identical to the reference's algorithm with edgeToRow[e] = row(e).

#include <mutex>
#include <type_traits>

#include "f3s_common.h"

// Device scratch of f3s_preprocess_count_static, owned by the library instead of the caller: every
// GPU the library runs on holds its own copy (8 MiB) at its own address until the process ends.
// In host code the name below is only a handle for hipGetSymbolAddress, never an address.
static constexpr size_t kF3sStaticScratchBytes = (size_t)8 << 20;
static __device__ __align__(256) unsigned char scratch[kF3sStaticScratchBytes];

namespace f3s {
namespace {

constexpr int kRangeMax = 393216;  // columns per bitset pass: 48 KiB of bits + 12 KiB of prefixes
constexpr int kSortMax = 1024;     // windows up to this many edges are ranked by a per-wave LDS sort
constexpr int kBinsMax = 960;      // the same on graphs of at most 2^22 nodes (26 waves per CU)
// TC blocks held in LDS at once by window_fill_kernel: windows with strictly ascending rows (96
// bytes of LDS per 16x16 block) and windows with repeated or descending columns (96 bytes as
// well, but a second pass per chunk)
constexpr int kFillChunk = 640;
constexpr int kFillChunkGeneric = 512;
// both, for the long windows of graphs of short ones: of up to kFillMid edges, and longer (or all)
constexpr int kFillChunkMid = 320, kFillChunkLong = 1280;
constexpr int kFillMid = 4096;
constexpr int kFillFewLong = 4096;

// The windows that the kernels with a wave per window leave to larger workgroups, as those kernels meet
// them: `mid` of up to midMax edges from the front of an array of nRW entries, `large` of more from its
// back. The counts lie in the workspace header and are cleared before phase 1.
struct LongLists {
  int mid, large;
};
struct LongQueue {
  LongLists* counts;  // null: no lists, nobody asks for them (or they are looked for, find_windows)
  int32_t* list;
  int nRW;
  int midMax;
  __device__ __forceinline__ void add(int w, int edges) const {
    if (edges <= midMax)
      list[atomicAdd(&counts->mid, 1)] = w;
    else
      list[nRW - 1 - atomicAdd(&counts->large, 1)] = w;
  }
  __device__ __forceinline__ int size(bool large) const { return large ? counts->large : counts->mid; }
  __device__ __forceinline__ int at(bool large, int k) const { return list[large ? nRW - 1 - k : k]; }
};

// workspace header (bytes 0..255)
struct WsHeader {
  int error;    // graphs of long windows: a column index outside [0, N) was met
  int maxCount; // largest per-window block count (multi-workgroup finalize)
  LongLists rank, fill;
};
// Where phase 1 leaves its result: a device array of the caller's, or pinned host memory that the
// host reads when the stream is done, without a copy (a copy to pageable memory costs 7 us more).
struct ResultPtr {
  long long* nTcb;
  int* error;  // 0 before the first kernel; a kernel that meets a column outside [0, N) stores 1
};

// The windows of more than minEdges and at most maxEdges edges are few and lie anywhere: thread t of
// workgroup b of `stride` looks at window b + t * stride (of those from `first` on), so that they are dealt out
// evenly without a queue. list: one entry per thread, in LDS. Returns their number; every thread of
// the workgroup calls this.
__device__ __forceinline__ int find_windows(const int32_t* __restrict__ rowPtr, int N, int nRW,
                                            int64_t first, int stride, int minEdges,
                                            int maxEdges, int* list, int* listLen) {
  __syncthreads();  // the list before this one has been worked through
  if (threadIdx.x == 0) *listLen = 0;
  __syncthreads();
  const int64_t w = first + blockIdx.x + (int64_t)threadIdx.x * stride;
  if (w < nRW) {
    const int n = rowPtr[min((int)w * 16 + 16, N)] - rowPtr[(int)w * 16];
    if (n > minEdges && n <= maxEdges) list[atomicAdd(listLen, 1)] = (int)w;
  }
  __syncthreads();
  return *listLen;
}
constexpr size_t kWsHeaderBytes = 256;

// Inclusive prefix sum over the wave's 64 lanes with data-parallel-primitive moves: shifts within
// rows of 16 lanes (lanes shifted in from outside a row read 0), then lane 15 of a row added to the
// whole next row and lane 31 to the upper half of the wave. Every lane of the wave must be active.
__device__ __forceinline__ unsigned wave_inclusive_scan(unsigned v, int /*lane*/) {
  v += (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xf, 0xf, true);   // row_shr:1
  v += (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xf, 0xf, true);   // row_shr:2
  v += (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xf, 0xf, true);   // row_shr:4
  v += (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xf, 0xf, true);   // row_shr:8
  v += (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xa, 0xf, false);  // row_bcast:15
  v += (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xc, 0xf, false);  // row_bcast:31
  return v;
}

__device__ __forceinline__ int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }

// 16 bytes of an output that this call does not read again, past the caches
__device__ __forceinline__ void store_streaming(uint4* p, const uint4& v) {
  typedef unsigned uint4v __attribute__((ext_vector_type(4)));
  __builtin_nontemporal_store(uint4v{v.x, v.y, v.z, v.w}, reinterpret_cast<uint4v*>(p));
}

// largest r in [0,15] with sRow[r] <= e (sRow[0] <= e < sRow[16])
__device__ __forceinline__ int row_of_edge(const int* sRow, int e) {
  int r = 0;
  if (sRow[r + 8] <= e) r += 8;
  if (sRow[r + 4] <= e) r += 4;
  if (sRow[r + 2] <= e) r += 2;
  if (sRow[r + 1] <= e) r += 1;
  return r;
}

// Writes a TC block's tile ids (row * W + column of every set bit, rows top to bottom, columns
// left to right) to dst[pos...]. words: the block's bitmap, 8x8 sub-blocks in column-major order,
// rows of a sub-block MSB first. The bitmap is first brought into row-major order as dwords whose
// bit 31 - p stands for tile id 32 q + p (two rows of 16 columns, or four of 8, per dword): for
// 16 columns that interleaves the bytes of the left and the right sub-block (two byte permutes
// per four rows), for 8 columns the words are in that order already.
template <int W>
__device__ __forceinline__ void walk_tile_ids(const unsigned long long (&words)[16 * W / 64],
                                              uint8_t* __restrict__ dst, unsigned pos) {
  constexpr int NQ = 16 * W / 32;
  unsigned rm[NQ];
  if constexpr (W == 16) {
#pragma unroll
    for (int half = 0; half < 2; half++) {  // rows 0-7 (sub-blocks 0 and 2), rows 8-15 (1 and 3)
      const unsigned long long left = words[half], right = words[2 + half];
#pragma unroll
      for (int k = 0; k < 2; k++) {  // rows 4k .. 4k+3 of the half: the dword from the top
        const unsigned a = k == 0 ? (unsigned)(left >> 32) : (unsigned)left;
        const unsigned c = k == 0 ? (unsigned)(right >> 32) : (unsigned)right;
        rm[4 * half + 2 * k] = __builtin_amdgcn_perm(a, c, 0x07030602u);      // rows +0, +1
        rm[4 * half + 2 * k + 1] = __builtin_amdgcn_perm(a, c, 0x05010400u);  // rows +2, +3
      }
    }
  } else {
#pragma unroll
    for (int k = 0; k < 2; k++) {
      rm[2 * k] = (unsigned)(words[k] >> 32);
      rm[2 * k + 1] = (unsigned)words[k];
    }
  }
#pragma unroll
  for (int q = 0; q < NQ; q++) {
    unsigned x = rm[q];
    while (x) {
      const int p = __builtin_clz(x);
      dst[pos++] = (uint8_t)(32 * q + p);
      x &= ~(0x80000000u >> p);
    }
  }
}

// Tile ids (row * W + column of every set bit, rows top to bottom, columns left to right) of rows
// 8 half .. 8 half + 7 of a TC block to dst[pos...]. left, right: those rows of the columns 0-7 and
// 8-15 (W = 8: left only), MSB first. Brought into row-major order as dwords whose bit 31 - p stands
// for tile id 8 W half + 32 q + p, two rows of 16 columns or four of 8 in each.
template <int W>
__device__ __forceinline__ void walk_half_block(unsigned long long left, unsigned long long right,
                                                int half, uint8_t* dst, unsigned pos) {
  constexpr int NQ = W / 4;
  unsigned rm[NQ];
  if constexpr (W == 16) {
#pragma unroll
    for (int k = 0; k < 2; k++) {  // four rows: the dword from the top
      const unsigned a = k == 0 ? (unsigned)(left >> 32) : (unsigned)left;
      const unsigned c = k == 0 ? (unsigned)(right >> 32) : (unsigned)right;
      rm[2 * k] = __builtin_amdgcn_perm(a, c, 0x07030602u);      // rows +0, +1
      rm[2 * k + 1] = __builtin_amdgcn_perm(a, c, 0x05010400u);  // rows +2, +3
    }
  } else {
    rm[0] = (unsigned)(left >> 32);
    rm[1] = (unsigned)left;
  }
#pragma unroll
  for (int q = 0; q < NQ; q++) {
    unsigned x = rm[q];
    const int id0 = 8 * W * half + 32 * q;
    while (x) {
      const int p = __builtin_clz(x);
      dst[pos++] = (uint8_t)(id0 + p);
      x &= ~(0x80000000u >> p);
    }
  }
}

// ------------------------------------------------------------------ phase 1
// compiler-level ordering point between LDS phases of ONE wave (its LDS operations execute in
// program order, so no hardware barrier is needed)
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_wave_barrier();
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
}

// Windows of at most kSortMax edges: one WAVE per window, no workgroup barrier. The wave sorts
// the window's column ids in its LDS slice (bitonic network, 32 compare-exchanges per step and
// lane row), compacts the distinct ones with ballot + popcount prefixes, and ranks every edge by
// binary search in the distinct list.
template <int W>
__global__ __launch_bounds__(64) void window_rank_small_kernel(
    const int32_t* __restrict__ rowPtr, const int32_t* __restrict__ colIdx, int N, int nRW,
    LongQueue queue, int32_t* __restrict__ blockPartition, int32_t* __restrict__ edgeToColumn,
    int32_t* __restrict__ edgeToRow, int* __restrict__ error) {
  __shared__ uint32_t sKeys[kSortMax];
  __shared__ uint32_t sUniq[kSortMax];
  __shared__ int sRowW[17];
  const int lane = threadIdx.x;
  const int w = blockIdx.x;
  const int r0 = w * 16;
  int* sRow = sRowW;
  if (lane < 17) sRow[lane] = rowPtr[min(r0 + lane, N)];
  wave_lds_sync();
  const int eS = sRow[0], eE = sRow[16];
  const int n = eE - eS;
  if (n == 0) {
    if (lane == 0) blockPartition[w] = 0;
    return;
  }
  if (n > kSortMax) {  // left to another kernel
    if (lane == 0 && queue.counts) queue.add(w, n);
    return;
  }
  uint32_t* keys = sKeys;
  uint32_t* uniq = sUniq;
  int P = 64;
  while (P < n) P <<= 1;
  bool bad = false;
  for (int i = lane; i < P; i += 64) {
    uint32_t k = 0xFFFFFFFFu;  // padding sorts last
    if (i < n) {
      k = (uint32_t)colIdx[eS + i];
      if (k >= (uint32_t)N) {
        bad = true;
        k = 0xFFFFFFFEu;
      }
    }
    keys[i] = k;
  }
  if (bad) *error = 1;
  wave_lds_sync();
  for (int k = 2; k <= P; k <<= 1) {
    for (int j = k >> 1; j > 0; j >>= 1) {
      // all of the lane's compare-exchanges of this step: reads first, then writes, so the
      // LDS latencies overlap (at most kSortMax / 128 pairs per lane)
      constexpr int MAXP = kSortMax / 128;
      uint32_t va[MAXP], vb[MAXP];
      const int nPairsLane = P >> 7;  // P/2 pairs over 64 lanes (P >= 128), 0 when P == 64
      if (nPairsLane == 0) {
        if (lane < 32) {
          const int lo = ((lane & ~(j - 1)) << 1) | (lane & (j - 1));
          const int hi = lo | j;
          const uint32_t x = keys[lo], y = keys[hi];
          const bool up = (lo & k) == 0;
          if ((x > y) == up) {
            keys[lo] = y;
            keys[hi] = x;
          }
        }
      } else {
#pragma unroll
        for (int q = 0; q < MAXP; q++) {
          if (q < nPairsLane) {
            const int i = lane + 64 * q;
            const int lo = ((i & ~(j - 1)) << 1) | (i & (j - 1));
            va[q] = keys[lo];
            vb[q] = keys[lo | j];
          }
        }
#pragma unroll
        for (int q = 0; q < MAXP; q++) {
          if (q < nPairsLane) {
            const int i = lane + 64 * q;
            const int lo = ((i & ~(j - 1)) << 1) | (i & (j - 1));
            const bool up = (lo & k) == 0;
            const bool swap = (va[q] > vb[q]) == up;
            keys[lo] = swap ? vb[q] : va[q];
            keys[lo | j] = swap ? va[q] : vb[q];
          }
        }
      }
      wave_lds_sync();
    }
  }
  int nUniq = 0;
  const unsigned long long ltMask = (1ull << lane) - 1ull;
  for (int base = 0; base < P; base += 64) {
    const int i = base + lane;
    const uint32_t k = keys[i];
    const bool first = k < 0xFFFFFFFEu && (i == 0 || keys[i - 1] != k);
    const unsigned long long bal = __ballot(first);
    if (first) uniq[nUniq + __popcll(bal & ltMask)] = k;
    nUniq += __popcll(bal);
  }
  wave_lds_sync();
  for (int e = eS + lane; e < eE; e += 64) {
    const uint32_t col = (uint32_t)colIdx[e];
    int lo = 0, hi = nUniq - 1, found = 0;
    while (lo <= hi) {
      const int mid = (lo + hi) >> 1;
      const uint32_t v = uniq[mid];
      if (v == col) {
        found = mid;
        break;
      }
      if (v < col)
        lo = mid + 1;
      else
        hi = mid - 1;
    }
    edgeToColumn[e] = found;
    edgeToRow[e] = r0 + row_of_edge(sRow, e);
  }
  if (lane == 0) blockPartition[w] = (nUniq + W - 1) / W;
}

// A wave's n words, groups of 64 in key[], into buf at the places that hist holds for the values of their
// `bits` bits above `shift`, in order: a lane's place is that plus the number of lanes before it in its
// group with the same value (one ballot per bit).
template <int G>
__device__ __forceinline__ void wave_scatter_in_order(const uint32_t (&key)[G], uint32_t* buf, uint32_t* hist,
                                                      int n, int shift, int bits, int lane) {
  const unsigned long long ltMask = (1ull << lane) - 1ull;
#pragma unroll
  for (int u = 0; u < G; u++) {
    if (64 * u >= n) break;
    const bool valid = lane < n - 64 * u;
    const unsigned dgt = (key[u] >> shift) & ((1u << bits) - 1u);
    unsigned long long peers = __ballot(valid);
    for (int b = 0; b < bits; b++) {
      const bool bit = (dgt >> b) & 1u;
      const unsigned long long bal = __ballot(bit);
      peers &= bit ? bal : ~bal;
    }
    if (valid) buf[hist[dgt] + __popcll(peers & ltMask)] = key[u];
    // the last peer advances the value's position; the wave's LDS operations stay in order
    if (valid && (peers >> lane) == 1ull) hist[dgt] += __popcll(peers);
  }
}

// The same where the order does not matter: words with the same value are put in order by the later
// passes of a sort or name the same column, and equal columns only have to end up next to each other. A
// returning LDS atomic hands out the places, a tenth of the instructions.
template <int G>
__device__ __forceinline__ void wave_scatter(const uint32_t (&key)[G], uint32_t* buf, uint32_t* hist, int n,
                                             int shift, int bits, int lane) {
#pragma unroll
  for (int u = 0; u < G; u++) {
    if (64 * u >= n) break;
    if (lane < n - 64 * u) buf[atomicAdd(&hist[(key[u] >> shift) & ((1u << bits) - 1u)], 1u)] = key[u];
  }
}

// LSD radix sort of a wave's n words in `buf` (LDS) by the colBits bits above IDX_BITS: every pass holds
// the words in registers, G groups of 64 at most, while it scatters them back. hist: 256 counters. buf: 64 G
// words.
template <int IDX_BITS, int G>
__device__ __forceinline__ void wave_radix_sort(uint32_t* buf, uint32_t* hist, int n, int colBits,
                                                int lane) {
  // Digits: the first pass takes eight bits, the stable passes share the rest evenly (22 column
  // bits: 8 + 7 + 7; 18: 8 + 5 + 5), so that a stable pass spends one ballot per bit it needs.
  const int firstBits = colBits < 8 ? colBits : 8;
  const int restBits = colBits - firstBits;
  const int nStable = (restBits + 7) / 8;
  int shift = IDX_BITS;
  for (int pass = 0; pass <= nStable; pass++) {
    const int db = pass == 0 ? firstBits
                             : restBits / nStable + (pass <= restBits % nStable ? 1 : 0);
    const unsigned mask = (1u << db) - 1u;
#pragma unroll
    for (int k = 0; k < 4; k++) hist[lane + 64 * k] = 0;
    uint32_t key[G];
#pragma unroll
    for (int u = 0; u < G; u++) {
      if (64 * u >= n) break;
      key[u] = buf[64 * u + lane];
    }
    wave_lds_sync();
#pragma unroll
    for (int u = 0; u < G; u++) {
      if (64 * u >= n) break;
      if (lane < n - 64 * u) atomicAdd(&hist[(key[u] >> shift) & mask], 1u);
    }
    wave_lds_sync();
    {
      // exclusive scan of the 256 counts: lane l owns bins 4l .. 4l+3
      const uint4 c = reinterpret_cast<uint4*>(hist)[lane];
      const unsigned sum = c.x + c.y + c.z + c.w;
      const unsigned excl = wave_inclusive_scan(sum, lane) - sum;
      reinterpret_cast<uint4*>(hist)[lane] =
          make_uint4(excl, excl + c.x, excl + c.x + c.y, excl + c.x + c.y + c.z);
    }
    wave_lds_sync();
    if (pass == 0)
      wave_scatter<G>(key, buf, hist, n, shift, db, lane);
    else
      wave_scatter_in_order<G>(key, buf, hist, n, shift, db, lane);
    wave_lds_sync();
    shift += db;
  }
}

// Rows of the edges of a window of at most MAX edges, for one wave that walks the edges in groups of
// 64. mark: MAX / 32 + 2 words of LDS, 8-byte aligned; bit i is set where a row that is not empty
// starts at edge i, and nibble k of the last two words names the k-th such row: two instructions
// count the marks up to a lane, where a search of the row pointers is four dependent LDS reads.
template <int MAX>
struct EdgeRows {
  const uint32_t* mark;
  unsigned long long names;
  int rows;  // rows in front of the next group

  // rowStart: lane r holds row r's first edge (from the window's first one), lane 16 their number
  __device__ __forceinline__ void init(uint32_t* words, int rowStart, int lane) {
    static_assert(MAX % 64 == 0, "the row names are read as one 64-bit word");
    if (lane < MAX / 32 + 2) words[lane] = 0u;
    wave_lds_sync();
    const int next = __shfl_down(rowStart, 1);
    const unsigned filled = (unsigned)__ballot(lane < 16 && next > rowStart);
    if (lane < 16 && ((filled >> lane) & 1u)) {
      const int k = __popc(filled & ((1u << lane) - 1u));
      atomicOr(&words[rowStart >> 5], 1u << (rowStart & 31));
      atomicOr(&words[MAX / 32 + (k >> 3)], (uint32_t)lane << (4 * (k & 7)));
    }
    wave_lds_sync();
    mark = words;
    names = *reinterpret_cast<const unsigned long long*>(words + MAX / 32);
    rows = 0;
  }
  // row of this lane's edge in the group of 64 from `base` on (groups in order, each once), and
  // whether the edge is the first of its row
  __device__ __forceinline__ int next_group(int base, int lane, bool* starts) {
    const uint2 m = *reinterpret_cast<const uint2*>(mark + (base >> 5));
    const bool own = (((lane < 32 ? m.x : m.y) >> (lane & 31)) & 1u) != 0u;
    const int k = rows + (int)__builtin_amdgcn_mbcnt_hi(m.y, __builtin_amdgcn_mbcnt_lo(m.x, 0));
    rows += __popc(m.x) + __popc(m.y);
    *starts = own;
    return (int)(names >> (4 * (k - (own ? 0 : 1)))) & 15;
  }
};

// EdgeRows where only the rows are asked for: bit i - 1 is set where a row that is not empty starts at edge
// i > 0, so that the set bits below a lane are the rows that started before its edge, without the first one.
// Where no row is empty (every node has its own diagonal entry, for one) that number is the row.
template <int MAX>
struct RowMarks {
  uint32_t words;  // lane l holds word l of the marks
  unsigned long long names;
  int rows;
  bool named;  // some rows are empty

  // rowStart, mark: as for EdgeRows
  __device__ __forceinline__ void init(uint32_t* mark, int rowStart, int lane) {
    static_assert(MAX % 64 == 0 && MAX / 32 + 2 <= 64, "whole groups, a word per lane");
    if (lane < MAX / 32 + 2) mark[lane] = 0u;
    wave_lds_sync();
    const int next = __shfl_down(rowStart, 1);
    const unsigned filled = (unsigned)__ballot(lane < 16 && next > rowStart);
    named = filled != 0xFFFFu;
    if (lane < 16 && ((filled >> lane) & 1u)) {
      const int k = __popc(filled & ((1u << lane) - 1u));
      if (k > 0) atomicOr(&mark[(rowStart - 1) >> 5], 1u << ((rowStart - 1) & 31));
      if (named) atomicOr(&mark[MAX / 32 + (k >> 3)], (uint32_t)lane << (4 * (k & 7)));
    }
    wave_lds_sync();
    words = mark[min(lane, MAX / 32 + 1)];
    names = (unsigned long long)(unsigned)__builtin_amdgcn_readlane((int)words, MAX / 32) |
            (unsigned long long)(unsigned)__builtin_amdgcn_readlane((int)words, MAX / 32 + 1) << 32;
    rows = 0;
  }
  // row of this lane's edge in group u of 64 (groups in order, each once)
  __device__ __forceinline__ int next_group(int u) {
    const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)words, 2 * u);
    const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)words, 2 * u + 1);
    int k = (int)__builtin_amdgcn_mbcnt_hi(hi, __builtin_amdgcn_mbcnt_lo(lo, rows));
    rows += __popc(lo) + __popc(hi);
    if (named) k = (int)(names >> (4 * k)) & 15;
    return k;
  }
};

// The same job for graphs of at most 2^22 nodes, where a column id and the edge's position in the
// window (< kBinsMax) fit one 32-bit word. The columns' top ten bits spread the window's
// edges over 1024 bins (two 16-bit counters per word; one counting pass, one that hands out
// places), after which an edge shares its bin with one or two others and finds its place by
// comparing itself with its neighbours. The sorted words carry the edge positions along, so that the rank of
// every distinct column goes straight back to its edges. A window whose columns crowd into few bins
// (communities) is binned again, more finely around its middle; only one that crowds there too takes an LSD
// radix sort of the column bits, whose stable passes cost a ballot per bit.
//
// Bound by the issue of vector instructions: 885 of them for a window of 400 edges when every group of 64
// edges guarded its lanes, looked up its bins' ends and walked them. Groups that are known to be whole (by the
// window's size, six sizes) need no guards and immediate offsets, and the neighbours need no bin's ends. One
// LDS buffer: between its passes a window's words are in registers, so that a pass can scatter into the
// buffer it has read; 6 KiB and 71 registers, 26 waves per CU, where two buffers allowed 16. Preprocessing of
// a 61M-edge graph (149k such windows) 789 -> 646 us, of a 2.8M-edge R-MAT graph 112 -> 104, of community
// graphs of 15k to 200k nodes 53 -> 52 to 209 -> 163.
constexpr int kRankBins = 1024;
// A fuller bin makes a window a crowded one. At 12 R-MAT graphs, whose hub columns repeat up to 16 times, take
// that route: 2.8M edges 104 -> 121 us, 61M edges 646 -> 840; at 36 and 48 communities walk fuller bins: 60k
// nodes 58 -> 59 and 60.
constexpr int kRankCrowd = 24;
constexpr int kRankNear = 3;    // neighbours on each side that every word is compared with
constexpr int kRankStep = 4;    // ... and how many more at a time where bins are fuller
constexpr int kRankPad = 32;
static_assert(kRankPad >= kRankCrowd + kRankStep, "neighbours of the first and the last word");
struct alignas(16) RankBinsLds {  // of one wave
  uint32_t hist[kRankBins / 2];  // word i: bin i in the low half, bin 512 + i in the high one
  // the window's words from kRankPad on: words below them all in front, words above them all behind the last
  uint32_t words[kRankPad + kBinsMax + kRankPad];
  uint32_t mark[kBinsMax / 32 + 2];
};

constexpr int kRankIdxBits = 10;
static_assert(kBinsMax <= (1 << kRankIdxBits), "edge position must fit kRankIdxBits");

// Adjacency matrices commonly hold the diagonal: sixteen neighbouring columns in every window, of one bin, where
// every one of them compares itself with the others. So a window's own columns are spread over bins of their
// own: each moves a bin further than the one before, and the columns above all sixteen with them. The columns'
// order stays. (61M edges: 199 -> 176 us for the short windows, 77 -> 70 us for those of up to 4 096 edges.)
// Returns the window's first column, or one past all columns where the bins (1 << bits columns in all) have no
// room for that.
__device__ __forceinline__ int own_columns(int w, int64_t N, int shift, int bits) {
  return N + (17ll << shift) < (1ll << bits) ? w * 16 : 0x7FFFFFFF;
}
__device__ __forceinline__ uint32_t spread_column(uint32_t col, int own, int shift) {
  return col + ((uint32_t)min(max((int)col - own + 1, 0), 17) << shift);
}
// Back: exact except for the window's own columns, which all become the ninth of them.
__device__ __forceinline__ uint32_t gathered_column(uint32_t col, int own, int shift) {
  const int beyond = (int)col - own;
  return beyond < 0 ? col : (uint32_t)(own + max(beyond - (17 << shift), 8));
}

// Ranks of the distinct columns of n sorted words, collected in edge order and written as whole lines. Here and
// in rank_window_groups 64 (G - P) < n <= 64 G: the first G - P groups of 64 edges are whole, and only the
// others look at the edge's number.
template <int W, int G, int P>
__device__ __forceinline__ void rank_sorted_words(int w, uint32_t* buf, int n, int lane,
                                                  int32_t* __restrict__ blockPartition,
                                                  int32_t* __restrict__ ranks) {
  uint32_t word[G];
#pragma unroll
  for (int u = 0; u < G; u++) {
    if (u >= G - P && 64 * u >= n) continue;
    word[u] = buf[64 * u + lane];
  }
  wave_lds_sync();
  int nUniq = 0;
  uint32_t last = ~(uint32_t)__builtin_amdgcn_readfirstlane((int)word[0]);
#pragma unroll
  for (int u = 0; u < G; u++) {
    if (u >= G - P && 64 * u >= n) continue;
    const bool valid = u < G - P || lane < n - 64 * u;
    const uint32_t left =
        (uint32_t)__builtin_amdgcn_update_dpp((int)last, (int)word[u], 0x138, 0xf, 0xf, false);
    last = (uint32_t)__builtin_amdgcn_readlane((int)word[u], 63);
    const bool first = (left ^ word[u]) >= (1u << kRankIdxBits) && valid;
    const unsigned long long firsts = __ballot(first);
    const int below = (int)__builtin_amdgcn_mbcnt_hi(
        (unsigned)(firsts >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)firsts, nUniq));
    if (valid) buf[word[u] & ((1u << kRankIdxBits) - 1u)] = (uint32_t)(below - (first ? 0 : 1));
    nUniq += __popcll(firsts);
  }
  wave_lds_sync();
#pragma unroll
  for (int u = 0; u < G; u++) {
    if (u >= G - P && 64 * u >= n) continue;
    if (u < G - P || lane < n - 64 * u) ranks[64 * u + lane] = (int)buf[64 * u + lane];
  }
  if (lane == 0) blockPartition[w] = (nUniq + W - 1) / W;
}

// Counts of the bins into where each starts; whether some bin holds more than kRankCrowd. Lane l owns words
// 8 l .. 8 l + 7, both halves at once: no sum reaches 2^16.
__device__ __forceinline__ bool rank_bin_starts(uint32_t* hist, int lane) {
  uint4* h = reinterpret_cast<uint4*>(hist) + 2 * lane;
  const uint4 x = h[0], y = h[1];
  uint32_t v[8] = {x.x, x.y, x.z, x.w, y.x, y.y, y.z, y.w};
  uint32_t total = 0, full = 0;
#pragma unroll
  for (int k = 0; k < 8; k++) {
    full |= v[k] + 0x10001u * (0x7FFFu - kRankCrowd);  // bit 15 of a half: more than kRankCrowd
    total += v[k];
  }
  const uint32_t incl = wave_inclusive_scan(total, lane);
  uint32_t run = incl - total + ((uint32_t)__builtin_amdgcn_readlane((int)incl, 63) << 16);
#pragma unroll
  for (int k = 0; k < 8; k++) {
    const uint32_t start = run;
    run += v[k];
    v[k] = start;
  }
  h[0] = make_uint4(v[0], v[1], v[2], v[3]);
  h[1] = make_uint4(v[4], v[5], v[6], v[7]);
  const bool crowded = __ballot((full & 0x80008000u) != 0u) != 0ull;
  wave_lds_sync();
  return crowded;
}

// Places of the words of groups u0 .. u0 + B - 1 (those before `groups`) of the words that are in their bins'
// order: inside its bin, later ones that are smaller move a word up, earlier ones that are larger move it
// down, and words of other bins do neither. Three neighbours on each side are enough for bins of four; a group with
// a fuller bin goes on until no lane's next neighbour is of its bin. The groups' first neighbours are read
// together, as what a wave waits for here is one round of LDS reads after the other. sameBin: words of one
// bin differ by less in their exclusive or. wholeGroups: groups from 1 up to there are all words of the window, and so
// are the one before and the one behind.
template <int B>
__device__ __forceinline__ void rank_places(const uint32_t* buf, int u0, int groups, int wholeGroups, int lane,
                                            int n, uint32_t sameBin, uint32_t (&word)[B], uint32_t (&place)[B]) {
  uint32_t up[B][kRankNear], down[B][kRankNear];
#pragma unroll
  for (int b = 0; b < B; b++) {
    if (u0 + b >= groups) continue;
    const uint32_t* at = buf + 64 * (u0 + b) + lane;
    word[b] = at[0];
#pragma unroll
    for (int k = 0; k < kRankNear; k++) {
      up[b][k] = at[k + 1];
      down[b][k] = at[-k - 1];
    }
  }
  const auto more_in_bin = [&](int b, int k, uint32_t u, uint32_t d) {
    const int g = u0 + b;
    if (g > 0 && g < wholeGroups) return (u ^ word[b]) < sameBin || (d ^ word[b]) < sameBin;
    return ((u ^ word[b]) < sameBin && lane < n - 64 * g - k) ||
           ((d ^ word[b]) < sameBin && lane >= k - 64 * g && lane < n - 64 * g);
  };
  bool more = false;
#pragma unroll
  for (int b = 0; b < B; b++) {
    if (u0 + b >= groups) continue;
    int p = 64 * (u0 + b) + lane;
#pragma unroll
    for (int k = 0; k < kRankNear; k++) {
      p += up[b][k] < word[b] ? 1 : 0;
      p -= down[b][k] > word[b] ? 1 : 0;
    }
    place[b] = (uint32_t)p;
    more = more || more_in_bin(b, kRankNear, up[b][kRankNear - 1], down[b][kRankNear - 1]);
  }
  if (__ballot(more) != 0ull) {
#pragma unroll
    for (int b = 0; b < B; b++) {
      if (u0 + b >= groups) continue;
      const uint32_t* at = buf + 64 * (u0 + b) + lane;
      uint32_t u = up[b][kRankNear - 1], d = down[b][kRankNear - 1];
      for (int k = kRankNear; k < kRankCrowd; k += kRankStep) {
        if (__ballot(more_in_bin(b, k, u, d)) == 0ull) break;
#pragma unroll
        for (int j = 1; j <= kRankStep; j++) {
          u = at[k + j];
          d = at[-k - j];
          place[b] += u < word[b] ? 1u : 0u;
          place[b] -= d > word[b] ? 1u : 0u;
        }
      }
    }
  }
}

// False where columns crowd into few bins: the rows are written, the unsorted words are in lds.words, with the
// columns as they are, and the rest is left to the caller.
template <int W, int G, int P>
__device__ __forceinline__ bool rank_window_groups(
    int w, const int32_t* __restrict__ cols, int n, int rowStart, int N, int colBits, RankBinsLds& lds,
    int32_t* __restrict__ blockPartition, int32_t* __restrict__ ranks, int32_t* __restrict__ rows,
    int* __restrict__ error) {
  const int lane = threadIdx.x & 63;
  const int shift = colBits > 10 ? colBits - 10 : 0;
  uint32_t* buf = lds.words + kRankPad;
  uint32_t* hist = lds.hist;
  uint32_t col[G];  // columns, later (column, position) words, of edges 64 u + lane
#pragma unroll
  for (int u = 0; u < G; u++)
    col[u] = (uint32_t)cols[u < G - P ? 64 * u + lane : min(64 * u + lane, n - 1)];
  auto valid = [&](int u) { return u < G - P || lane < n - 64 * u; };
  RowMarks<kBinsMax> marks;
  marks.init(lds.mark, rowStart, lane);
#pragma unroll
  for (int k = 0; k < kRankBins / 2 / 256; k++)
    reinterpret_cast<uint4*>(hist)[lane + 64 * k] = make_uint4(0, 0, 0, 0);
  if (lane < kRankPad) {
    lds.words[lane] = 0u;
    buf[n + lane] = 0xFFFFFFFFu;
  }
  wave_lds_sync();
  // ---- rows
#pragma unroll
  for (int u = 0; u < G; u++) {
    const int row = marks.next_group(u);
    if (valid(u)) rows[64 * u + lane] = w * 16 + row;
  }
  // ---- how many edges fall into each bin
  uint32_t most = 0;
#pragma unroll
  for (int u = 0; u < G; u++) most = max(most, col[u]);
  if (__ballot(most >= (uint32_t)N) != 0ull) {
    *error = 1;
#pragma unroll
    for (int u = 0; u < G; u++) col[u] = col[u] < (uint32_t)N ? col[u] : 0u;
  }
  const int own = own_columns(w, N, shift, colBits);
#pragma unroll
  for (int u = 0; u < G; u++) col[u] = spread_column(col[u], own, shift);
  const uint32_t upper = 512u << shift;  // first column of the bins in high halves
#pragma unroll
  for (int u = 0; u < G; u++)
    if (valid(u)) atomicAdd(&hist[(col[u] >> shift) & 511u], col[u] < upper ? 1u : 0x10000u);
  wave_lds_sync();
  const bool crowded = rank_bin_starts(hist, lane);
  if (crowded) {
#pragma unroll
    for (int u = 0; u < G; u++)
      if (valid(u)) {
        const uint32_t c = (uint32_t)cols[64 * u + lane];
        buf[64 * u + lane] = ((c < (uint32_t)N ? c : 0u) << kRankIdxBits) | (uint32_t)(64 * u + lane);
      }
    wave_lds_sync();
    return false;
  }
  // ---- into the bins
  uint32_t at[G];
#pragma unroll
  for (int u = 0; u < G; u++) {
    const uint32_t half = col[u] < upper ? 0u : 16u;
    if (valid(u)) at[u] = (atomicAdd(&hist[(col[u] >> shift) & 511u], 1u << half) >> half) & 0xFFFFu;
  }
#pragma unroll
  for (int u = 0; u < G; u++)
    if (valid(u)) buf[at[u]] = (col[u] << kRankIdxBits) | (uint32_t)(64 * u + lane);
  wave_lds_sync();
  // ---- from the bins' order to the columns'
  constexpr int B = 2;
#pragma unroll
  for (int u = 0; u < G; u += B) {
    uint32_t word[B], place[B];
    rank_places<B>(buf, u, G, G - P - 1, lane, n, 1u << (kRankIdxBits + shift), word, place);
#pragma unroll
    for (int b = 0; b < B; b++) {
      if (u + b >= G) continue;
      col[u + b] = word[b];
      at[u + b] = place[b];
    }
  }
  wave_lds_sync();
#pragma unroll
  for (int u = 0; u < G; u++)
    if (valid(u)) buf[at[u]] = col[u];
  wave_lds_sync();
  rank_sorted_words<W, G, P>(w, buf, n, lane, blockPartition, ranks);
  return true;
}

// The rest of a window whose columns crowd into few bins, as those of a community do: half of the bins are spread
// over the columns around the window's middle edge (512 of them, or four bins' worth), the others over
// what lies below and above. Columns that crowd there as well take the radix sort. The columns are the true ones: a
// community around the window's own columns, spread like those, would lie in three pieces of which the middle
// holds one (500 communities of 200 nodes, 37 edges a node: 121 us a call instead of 97; 800 000 nodes in
// 1 000, 33 edges: 425 instead of 313; with no column spread at all 99 and 333).
template <int W, int G>
__device__ __forceinline__ void rank_crowded_window(int w, int n, int N, int colBits, RankBinsLds& lds, int lane,
                                                    int32_t* __restrict__ blockPartition,
                                                    int32_t* __restrict__ ranks) {
  const int shift = colBits > 10 ? colBits - 10 : 0;
  uint32_t* buf = lds.words + kRankPad;
  uint32_t* hist = lds.hist;
  // the last bin that starts at or before the middle edge
  uint32_t bin = 0;
#pragma unroll
  for (int k = 0; k < kRankBins / 128; k++) {
    const uint32_t v = hist[lane + 64 * k];
    bin += __popcll(__ballot((v & 0xFFFFu) <= (uint32_t)n / 2)) + __popcll(__ballot((v >> 16) <= (uint32_t)n / 2));
  }
  bin -= 1u;
  const int fine = shift > 7 ? shift - 7 : 0;
  const uint32_t span = 512u << fine;
  const uint32_t middle =
      gathered_column((2u * bin + 1u) << shift >> 1, own_columns(w, N, shift, colBits), shift);
  const uint32_t from = (middle > span / 2 ? middle - span / 2 : 0u) >> fine << fine;
  wave_lds_sync();
#pragma unroll
  for (int k = 0; k < kRankBins / 2 / 256; k++)
    reinterpret_cast<uint4*>(hist)[lane + 64 * k] = make_uint4(0, 0, 0, 0);
  wave_lds_sync();
  // bins 0..255: below, 256..767: around the middle, 768..1023: above
  auto bin_of = [&](uint32_t c) {
    const uint32_t coarse = (c >> (shift + 2)) + (c < from ? 0u : 768u);
    return c - from < span ? 256u + ((c - from) >> fine) : coarse;
  };
  uint32_t word[G], at[G];
#pragma unroll
  for (int u = 0; u < G; u++) {
    if (64 * u >= n) continue;
    word[u] = buf[64 * u + lane];
    const uint32_t b = bin_of(word[u] >> kRankIdxBits);
    if (lane < n - 64 * u) atomicAdd(&hist[b & 511u], b < 512u ? 1u : 0x10000u);
  }
  wave_lds_sync();
  if (rank_bin_starts(hist, lane)) {
    wave_radix_sort<kRankIdxBits, G>(buf, hist, n, colBits, lane);
  } else {
#pragma unroll
    for (int u = 0; u < G; u++) {
      if (64 * u >= n) continue;
      const uint32_t b = bin_of(word[u] >> kRankIdxBits);
      const uint32_t half = b < 512u ? 0u : 16u;
      if (lane < n - 64 * u)
        buf[(atomicAdd(&hist[b & 511u], 1u << half) >> half) & 0xFFFFu] = word[u];
    }
    wave_lds_sync();
#pragma unroll
    for (int u = 0; u < G; u++) {
      if (64 * u >= n) continue;
      const bool middleBin = (buf[64 * u + lane] >> kRankIdxBits) - from < span;
      uint32_t one[1], place[1];
      rank_places<1>(buf, u, G, 0, lane, n, 1u << (kRankIdxBits + (middleBin ? fine : shift + 2)), one, place);
      word[u] = one[0];
      at[u] = place[0];
    }
    wave_lds_sync();
#pragma unroll
    for (int u = 0; u < G; u++) {
      if (64 * u >= n) continue;
      if (lane < n - 64 * u) buf[at[u]] = word[u];
    }
    wave_lds_sync();
  }
  rank_sorted_words<W, G, G>(w, buf, n, lane, blockPartition, ranks);
}

template <int W>
__device__ __forceinline__ void rank_window_by_bins(
    int w, const int32_t* __restrict__ rowPtr, const int32_t* __restrict__ colIdx, int N,
    int colBits, const LongQueue& queue, RankBinsLds& lds, int32_t* __restrict__ blockPartition,
    int32_t* __restrict__ edgeToColumn, int32_t* __restrict__ edgeToRow,
    int* __restrict__ error) {
  const int lane = threadIdx.x & 63;
  int rowStart = rowPtr[min(w * 16 + min(lane, 16), N)];
  const int eS = __builtin_amdgcn_readlane(rowStart, 0);
  const int n = __builtin_amdgcn_readlane(rowStart, 16) - eS;
  rowStart -= eS;
  if (n == 0) {
    if (lane == 0) blockPartition[w] = 0;
    return;
  }
  if (n > kBinsMax) {  // left to another kernel
    if (lane == 0 && queue.counts) queue.add(w, n);
    return;
  }
  const int32_t* cols = colIdx + eS;
  int32_t *ranks = edgeToColumn + eS, *rows = edgeToRow + eS;
  bool done;
#define F3S_RANK_GROUPS(G, P)                                                                       \
  rank_window_groups<W, G, P>(w, cols, n, rowStart, N, colBits, lds, blockPartition, ranks, rows, error)
  if (n <= 64 * 2) {
    done = F3S_RANK_GROUPS(2, 2);
  } else if (n <= 64 * 4) {
    done = F3S_RANK_GROUPS(4, 2);
  } else if (n <= 64 * 6) {
    done = F3S_RANK_GROUPS(6, 2);
  } else if (n <= 64 * 8) {
    done = F3S_RANK_GROUPS(8, 2);
  } else if (n <= 64 * 11) {
    done = F3S_RANK_GROUPS(11, 3);
  } else {
    done = F3S_RANK_GROUPS(15, 4);
  }
#undef F3S_RANK_GROUPS
  if (done) return;
  if (n <= 64 * 4)
    rank_crowded_window<W, 4>(w, n, N, colBits, lds, lane, blockPartition, ranks);
  else
    rank_crowded_window<W, kBinsMax / 64>(w, n, N, colBits, lds, lane, blockPartition, ranks);
}
template <int W>
__global__ __launch_bounds__(64) void window_rank_bins_kernel(
    const int32_t* __restrict__ rowPtr, const int32_t* __restrict__ colIdx, int N, int colBits,
    LongQueue queue, int32_t* __restrict__ blockPartition, int32_t* __restrict__ edgeToColumn,
    int32_t* __restrict__ edgeToRow, int* __restrict__ error) {
  __shared__ RankBinsLds lds;
  rank_window_by_bins<W>((int)blockIdx.x, rowPtr, colIdx, N, colBits, queue, lds, blockPartition,
                         edgeToColumn, edgeToRow, error);
}

// One window by the whole workgroup, every edge's column against a bitset in LDS: range / 32 words
// of bits, then range / 128 group prefixes. Every thread of the workgroup calls this.
template <int W, int TB>
__device__ __forceinline__ void rank_window_by_bitset(
    int w, const int32_t* __restrict__ rowPtr, const int32_t* __restrict__ colIdx, int N,
    int range, int nPasses, int minEdges, uint32_t* bits, int32_t* __restrict__ blockPartition,
    int32_t* __restrict__ edgeToColumn, int32_t* __restrict__ edgeToRow,
    int* __restrict__ error) {
  uint32_t* pref = bits + (range >> 5);
  __shared__ int sRow[17];
  __shared__ unsigned sWaveTot[TB / 64];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  __syncthreads();  // the previous window's reads of sRow are done
  const int r0 = w * 16;
  if (tid < 17) sRow[tid] = rowPtr[min(r0 + tid, N)];
  __syncthreads();
  const int eS = sRow[0], eE = sRow[16];
  if (eE - eS <= minEdges) return;  // ranked by one wave
  const int nGroups = range >> 7;
  unsigned uniqueBefore = 0;
  for (int pass = 0; pass < nPasses; pass++) {
    const int lo = pass * range;
    for (int i = tid; i < nGroups; i += TB)
      reinterpret_cast<uint4*>(bits)[i] = make_uint4(0, 0, 0, 0);
    __syncthreads();
    // four edges per thread and step, loads first
    for (int e0 = eS + tid; e0 < eE; e0 += 4 * TB) {
      int cols[4];
#pragma unroll
      for (int u = 0; u < 4; u++) cols[u] = (e0 + u * TB < eE) ? colIdx[e0 + u * TB] : lo;
#pragma unroll
      for (int u = 0; u < 4; u++) {
        if (e0 + u * TB >= eE) continue;
        int col = cols[u];
        if ((unsigned)col >= (unsigned)N) {
          *error = 1;
          col = 0;
        }
        const unsigned rel = (unsigned)(col - lo);
        if (rel < (unsigned)range) atomicOr(&bits[rel >> 5], 1u << (rel & 31));
      }
    }
    __syncthreads();
    unsigned carry = uniqueBefore;
    for (int gb = 0; gb < nGroups; gb += TB) {
      const int gi = gb + tid;
      unsigned cnt = 0;
      if (gi < nGroups) {
        const uint4 v = reinterpret_cast<const uint4*>(bits)[gi];
        cnt = __popc(v.x) + __popc(v.y) + __popc(v.z) + __popc(v.w);
      }
      const unsigned incl = wave_inclusive_scan(cnt, lane);
      if (lane == 63) sWaveTot[wave] = incl;
      __syncthreads();
      unsigned waveOff = 0, tileTot = 0;
#pragma unroll
      for (int v = 0; v < TB / 64; v++) {
        const unsigned t = sWaveTot[v];
        if (v < wave) waveOff += t;
        tileTot += t;
      }
      if (gi < nGroups) pref[gi] = carry + waveOff + incl - cnt;
      carry += tileTot;
      __syncthreads();
    }
    for (int e0 = eS + tid; e0 < eE; e0 += 4 * TB) {
      int cols[4];
#pragma unroll
      for (int u = 0; u < 4; u++) cols[u] = (e0 + u * TB < eE) ? colIdx[e0 + u * TB] : -1;
#pragma unroll
      for (int u = 0; u < 4; u++) {
        if (e0 + u * TB >= eE) continue;
        const int col = (unsigned)cols[u] < (unsigned)N ? cols[u] : 0;
        const unsigned rel = (unsigned)(col - lo);
        if (rel < (unsigned)range) {
          // rank = set bits below this one: group prefix, then the whole 128-bit group read at
          // once and masked
          const unsigned wd = rel >> 5;
          const uint4 grp = reinterpret_cast<const uint4*>(bits)[wd >> 2];
          const unsigned words[4] = {grp.x, grp.y, grp.z, grp.w};
          unsigned rank = pref[wd >> 2];
#pragma unroll
          for (unsigned k = 0; k < 4; k++) {
            const unsigned keep = k < (wd & 3u) ? 0xFFFFFFFFu
                                  : (k == (wd & 3u) ? ((1u << (rel & 31)) - 1u) : 0u);
            rank += __popc(words[k] & keep);
          }
          edgeToColumn[e0 + u * TB] = (int)rank;
        }
        if (pass == 0) edgeToRow[e0 + u * TB] = r0 + row_of_edge(sRow, e0 + u * TB);
      }
    }
    uniqueBefore = carry;
    __syncthreads();
  }
  if (tid == 0) blockPartition[w] = (int)((uniqueBefore + W - 1) / W);
}

// LISTED: the large windows of the queue, of which those of more than minEdges edges are taken (graphs of
// mostly short windows); else workgroup b takes window b, if it is that long.
template <int W, int TB, bool LISTED>
__global__ __launch_bounds__(TB) void window_rank_kernel(
    const int32_t* __restrict__ rowPtr, const int32_t* __restrict__ colIdx, int N, int nRW,
    int range, int nPasses, int minEdges, LongQueue queue, int32_t* __restrict__ blockPartition,
    int32_t* __restrict__ edgeToColumn, int32_t* __restrict__ edgeToRow,
    int* __restrict__ error) {
  extern __shared__ __align__(16) uint32_t smem[];
  if constexpr (LISTED) {
    const int listed = queue.size(true);
    for (int k = blockIdx.x; k < listed; k += (int)gridDim.x)
      rank_window_by_bitset<W, TB>(queue.at(true, k), rowPtr, colIdx, N, range, nPasses, minEdges, smem,
                                   blockPartition, edgeToColumn, edgeToRow, error);
  } else {
    rank_window_by_bitset<W, TB>((int)blockIdx.x, rowPtr, colIdx, N, range, nPasses, minEdges,
                                 smem, blockPartition, edgeToColumn, edgeToRow, error);
  }
}

// Graphs of up to kFinSingleMax windows, most of them short: both kinds of window in one launch. The
// first longGroups workgroups look for the windows of more than kBinsMax edges and take one at a
// time with all of their waves, each wave of the others takes one window. One launch after the other
// meant that everything waited for the longest window twice (169k-node R-MAT graph, windows of up to
// 12 500 edges: 29 + 23 us).
template <int W, int TB>
__global__ __launch_bounds__(TB) void window_rank_all_kernel(
    const int32_t* __restrict__ rowPtr, const int32_t* __restrict__ colIdx, int N, int nRW,
    int colBits, int range, int longGroups, int32_t* __restrict__ blockPartition,
    int32_t* __restrict__ edgeToColumn, int32_t* __restrict__ edgeToRow,
    int* __restrict__ error) {
  extern __shared__ __align__(16) uint32_t smem[];
  constexpr int NW = TB / 64;
  if ((int)blockIdx.x >= longGroups) {
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int w = ((int)blockIdx.x - longGroups) * NW + wave;
    if (w < nRW)
      rank_window_by_bins<W>(w, rowPtr, colIdx, N, colBits, LongQueue{nullptr, nullptr, 0, 0},
                             reinterpret_cast<RankBinsLds*>(smem)[wave], blockPartition,
                             edgeToColumn, edgeToRow, error);
    return;
  }
  __shared__ int sList[TB];
  __shared__ int sListLen;
  for (int64_t first = 0; first < nRW; first += (int64_t)TB * longGroups) {
    const int found = find_windows(rowPtr, N, nRW, first, longGroups, kBinsMax, 0x7FFFFFFF, sList,
                                   &sListLen);
    for (int k = 0; k < found; k++)
      rank_window_by_bitset<W, TB>(sList[k], rowPtr, colIdx, N, range, 1, kBinsMax, smem, blockPartition,
                                   edgeToColumn, edgeToRow, error);
  }
}

// Windows too long for a wave on graphs whose column range needs several bitset passes (N >
// kRangeMax): one workgroup ranks the window's column ids among each other, instead of several passes over
// a 48 KiB bitset that such a window fills with a few thousand bits. The columns go into eight bins per
// thread, as in rank_window_groups; a thread keeps its columns and where it put them, finds their places
// among the sorted ones from their neighbours and marks the first of every column in a bitset of places, in
// which a rank is a count. Bound by the issue of vector instructions, and by latency where windows are few.
// Windows whose columns crowd into few bins take an LSD radix sort, eight bits per pass, and a binary search
// per edge. 256 threads for up to kMidMax edges, 24 waves per CU: most such windows have less than half of the 4 096
// edges that 512 threads hold, and each wave pays for the clearing, the scans and the guards of eight items
// (5 000 of 960 to 2 048 edges in a 61M-edge graph: 70 -> 54 us. A wave each, its state in LDS or in registers
// over thirty unrolled groups, took 63 to 97: too few waves, or code that the instruction cache does not hold.)
// 1024 threads for up to kFourMax and kLargeMax edges.
constexpr int kMidThreads = 256;
constexpr int kMidItems = 8;
constexpr int kMidMax = kMidThreads * kMidItems;
constexpr int kLargeThreads = 1024;
constexpr int kFourItems = 4;
constexpr int kFourMax = kLargeThreads * kFourItems;
constexpr int kLargeItems = 16;
constexpr int kLargeMax = kLargeThreads * kLargeItems;
constexpr int kSortCrowd = 32;  // a fuller bin sends the window to the radix sort
constexpr int kSortPad = 64;
static_assert(kSortPad >= kSortCrowd + kRankStep, "neighbours of the first and the last key");
template <int ITEMS, int THREADS>
constexpr size_t rank_sort_lds() {
  return ((size_t)THREADS * ITEMS + 2 * kSortPad + 4 * THREADS + 2 * (THREADS * ITEMS / 32)) * sizeof(uint32_t);
}

// The n distinct ones of a workgroup's keys, ascending, in sKeys and their number in *sUniq: an LSD radix
// sort, eight bits per pass, every wave on its own contiguous part of the keys, which it holds in registers
// while it scatters them back. Key u * THREADS + thread is key[u] of the thread. Every thread of the
// workgroup calls this.
template <int ITEMS, int THREADS>
__device__ __forceinline__ void rank_crowded_keys(const uint32_t (&key)[ITEMS], uint32_t* sKeys, uint32_t* sHist,
                                                  unsigned* sWaveTot, int n, int keyBits, int* sUniq) {
  constexpr int WAVES = THREADS / 64;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
#pragma unroll
  for (int u = 0; u < ITEMS; u++)
    if (tid < n - u * THREADS) sKeys[u * THREADS + tid] = key[u];
  // wave v sorts the keys [cb, cb + part) of every pass's input into their places of its output
  const int chunk = ((n + THREADS - 1) / THREADS) * 64;
  const int cb = min(n, wave * chunk), part = min(n - cb, chunk);
  uint32_t* hist = sHist + 256 * wave;
  uint32_t mine[ITEMS];
  for (int shift = 0; shift < keyBits; shift += 8) {
    __syncthreads();  // the keys of this pass are in place
#pragma unroll
    for (int u = 0; u < ITEMS; u++) {
      if (64 * u >= part) continue;
      mine[u] = lane < part - 64 * u ? sKeys[cb + 64 * u + lane] : 0u;
    }
#pragma unroll
    for (int k = 0; k < 4; k++) hist[lane + 64 * k] = 0;
    wave_lds_sync();
#pragma unroll
    for (int u = 0; u < ITEMS; u++) {
      if (64 * u >= part) continue;
      if (lane < part - 64 * u) atomicAdd(&hist[(mine[u] >> shift) & 255u], 1u);
    }
    __syncthreads();
    // thread d < 256: keys with a smaller digit, then this digit's keys of the waves in front
    unsigned c[WAVES], tot = 0, incl = 0;
    if (tid < 256) {
#pragma unroll
      for (int v = 0; v < WAVES; v++) {
        c[v] = sHist[256 * v + tid];
        tot += c[v];
      }
      incl = wave_inclusive_scan(tot, lane);
      if (lane == 63) sWaveTot[wave] = incl;
    }
    __syncthreads();
    if (tid < 256) {
      unsigned run = incl - tot;
#pragma unroll
      for (int v = 0; v < 4; v++)
        if (v < wave) run += sWaveTot[v];
#pragma unroll
      for (int v = 0; v < WAVES; v++) {
        sHist[256 * v + tid] = run;
        run += c[v];
      }
    }
    __syncthreads();
    if (shift == 0)
      wave_scatter<ITEMS>(mine, sKeys, hist, part, 0, 8, lane);
    else
      wave_scatter_in_order<ITEMS>(mine, sKeys, hist, part, shift, 8, lane);
  }
  __syncthreads();
  // distinct keys: first occurrences, a count with ballots, the waves' totals, then the stores
  unsigned cnt = 0, first = 0;  // bit u: key 64 u + lane of the part is one
#pragma unroll
  for (int u = 0; u < ITEMS; u++) {
    if (64 * u >= part) continue;
    const int i = cb + 64 * u + lane;
    const bool valid = lane < part - 64 * u;
    mine[u] = valid ? sKeys[i] : 0u;
    const bool is = valid && (i == 0 || sKeys[i - 1] != mine[u]);
    first |= is ? 1u << u : 0u;
    cnt += (unsigned)__popcll(__ballot(is));
  }
  if (lane == 0) sWaveTot[wave] = cnt;
  __syncthreads();
  unsigned pos = 0, all = 0;
#pragma unroll
  for (int v = 0; v < WAVES; v++) {
    const unsigned x = sWaveTot[v];
    if (v < wave) pos += x;
    all += x;
  }
#pragma unroll
  for (int u = 0; u < ITEMS; u++) {
    if (64 * u >= part) continue;
    const bool is = (first >> u) & 1u;
    const unsigned long long bal = __ballot(is);
    if (is) sKeys[pos + (unsigned)__popcll(bal & ((1ull << lane) - 1ull))] = mine[u];
    pos += (unsigned)__popcll(bal);
  }
  if (tid == 0) *sUniq = (int)all;
  __syncthreads();
}

// One window of at most THREADS * ITEMS edges by the whole workgroup; every thread calls this.
template <int W, int ITEMS, int THREADS>
__device__ __forceinline__ void rank_window_by_sort(
    int w, const int32_t* __restrict__ rowPtr, const int32_t* __restrict__ colIdx, int N, int colBits,
    uint32_t* sSort, int32_t* __restrict__ blockPartition, int32_t* __restrict__ edgeToColumn,
    int32_t* __restrict__ edgeToRow, int* __restrict__ error) {
  constexpr int WAVES = THREADS / 64;
  constexpr int CAP = THREADS * ITEMS;
  constexpr int BIN_BITS = THREADS == 256 ? 11 : 13;
  static_assert((1 << BIN_BITS) == 8 * THREADS, "eight bins per thread");
  static_assert(THREADS >= 256 && THREADS % 256 == 0, "the first 256 threads own one digit each");
  uint32_t* sKeys = sSort + kSortPad;  // CAP keys, room for kSortPad on each side
  uint32_t* sBins = sKeys + CAP + kSortPad;  // 16-bit counters, or the radix sort's digit counters
  uint32_t* sFirst = sBins + 4 * THREADS;  // bit per key: the first one of its column
  uint32_t* sBefore = sFirst + CAP / 32;  // such keys in front of a word of bits
  __shared__ int sRow[17];
  __shared__ unsigned sWaveTot[WAVES];
  __shared__ int sCrowded;
  __shared__ int sUniq;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // keys are columns plus one: 0 stands for none
  const int keyBits = colBits + (((int64_t)1 << colBits) <= (int64_t)N ? 1 : 0);
  const int shiftBins = keyBits > BIN_BITS ? keyBits - BIN_BITS : 0;
  const uint32_t sameBin = 1u << shiftBins;
  const int r0 = w * 16;
  __syncthreads();  // the window before this one has left the LDS arrays
  if (tid < 17) sRow[tid] = rowPtr[min(r0 + tid, N)];
  if (tid == 0) sCrowded = 0;
  reinterpret_cast<uint4*>(sBins)[tid] = make_uint4(0, 0, 0, 0);
  for (int i = tid; i < CAP / 32; i += THREADS) sFirst[i] = 0u;
  if (tid < kSortPad) sSort[tid] = 0u;
  __syncthreads();
  const int eS = uniform(sRow[0]);
  int n = uniform(sRow[16]) - eS;
  const int32_t* cols = colIdx + eS;
  int32_t *ranks = edgeToColumn + eS, *rows = edgeToRow + eS;
  // thread t's keys: of edges t + THREADS u
  uint32_t key[ITEMS], at[ITEMS];
#pragma unroll
  for (int u = 0; u < ITEMS; u++) {
    if (u * THREADS >= n) continue;
    key[u] = (uint32_t)cols[min(u * THREADS + tid, n - 1)];
  }
  if (tid < kSortPad) sKeys[n + tid] = 0xFFFFFFFFu;
  asm volatile("" : "+s"(n));
  const int own = own_columns(w, (int64_t)N + 1, shiftBins, keyBits);
  bool bad = false;
#pragma unroll
  for (int u = 0; u < ITEMS; u++) {
    if (u * THREADS >= n) continue;
    if (key[u] >= (uint32_t)N) {
      bad = true;
      key[u] = 0u;
    }
    key[u] = spread_column(key[u], own, shiftBins) + 1u;
    const uint32_t bin = key[u] >> shiftBins;
    if (tid < n - u * THREADS) {
      rows[u * THREADS + tid] = r0 + row_of_edge(sRow, eS + u * THREADS + tid);
      atomicAdd(&sBins[bin >> 1], 1u << ((bin & 1u) * 16u));
    }
  }
  if (bad) *error = 1;
  __syncthreads();
  {
    const uint4 x = reinterpret_cast<const uint4*>(sBins)[tid];
    uint32_t v[4] = {x.x, x.y, x.z, x.w};
    uint32_t total = 0, most = 0;
#pragma unroll
    for (int k = 0; k < 4; k++) {
      total += (v[k] & 0xFFFFu) + (v[k] >> 16);
      most = max(most, max(v[k] & 0xFFFFu, v[k] >> 16));
    }
    if (most > (uint32_t)kSortCrowd) sCrowded = 1;
    const unsigned incl = wave_inclusive_scan(total, lane);
    if (lane == 63) sWaveTot[wave] = incl;
    __syncthreads();
    unsigned run = incl - total;
#pragma unroll
    for (int u = 0; u < WAVES; u++)
      if (u < wave) run += sWaveTot[u];
#pragma unroll
    for (int k = 0; k < 4; k++) {
      const uint32_t mid = run + (v[k] & 0xFFFFu);
      const uint32_t start = run | (mid << 16);
      run = mid + (v[k] >> 16);
      v[k] = start;
    }
    reinterpret_cast<uint4*>(sBins)[tid] = make_uint4(v[0], v[1], v[2], v[3]);
  }
  __syncthreads();
  if (sCrowded) {
    rank_crowded_keys<ITEMS, THREADS>(key, sKeys, sBins, sWaveTot, n, keyBits, &sUniq);
    const int nUniq = sUniq;
#pragma unroll
    for (int u = 0; u < ITEMS; u++) {
      if (u * THREADS >= n) continue;
      int lo = 0, hi = nUniq - 1;  // the key is one of the window's distinct ones
      while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (sKeys[mid] < key[u])
          lo = mid + 1;
        else
          hi = mid;
      }
      if (tid < n - u * THREADS) ranks[u * THREADS + tid] = lo;
    }
    if (tid == 0) blockPartition[w] = (nUniq + W - 1) / W;
    return;
  }
  // into the bins (n is hidden from the compiler between the passes: sixteen comparisons with it, kept for
  // all of them, cost more vector registers than the keys. Within a pass the lane masks of the guarded items
  // still outnumber the scalar registers: 120 of them in window_rank_mid_kernel and 382 in the two forms of
  // window_rank_rest_kernel go to lanes of vector registers and back. None goes to memory.)
  asm volatile("" : "+s"(n));
#pragma unroll
  for (int u = 0; u < ITEMS; u++) {
    if (u * THREADS >= n) continue;
    const uint32_t bin = key[u] >> shiftBins, half = (bin & 1u) * 16u;
    at[u] = 0;
    if (tid < n - u * THREADS) {
      at[u] = (atomicAdd(&sBins[bin >> 1], 1u << half) >> half) & 0xFFFFu;
      sKeys[at[u]] = key[u];
    }
  }
  __syncthreads();
  asm volatile("" : "+s"(n));
  // Each key's place among the sorted ones: from its place in the bins' order, later keys that are smaller
  // move it up, earlier ones that are larger move it down, and keys of other bins do neither. An earlier
  // equal one says that this is not the first of its column.
#pragma unroll
  for (int u = 0; u < ITEMS; u++) {
    if (u * THREADS >= n) continue;
    const bool valid = tid < n - u * THREADS;
    const uint32_t* here = sKeys + at[u];
    uint32_t up = 0, down = 0;
    int place = (int)at[u];
    bool again = false;
#pragma unroll
    for (int k = 1; k <= kRankNear; k++) {
      up = here[k];
      down = here[-k];
      place += up < key[u] ? 1 : 0;
      place -= down > key[u] ? 1 : 0;
      again = again || down == key[u];
    }
    for (int k = kRankNear; k < kSortCrowd; k += kRankStep) {
      const bool more = valid && ((up ^ key[u]) < sameBin || ((down ^ key[u]) < sameBin && down != 0u));
      if (__ballot(more) == 0ull) break;
#pragma unroll
      for (int j = 1; j <= kRankStep; j++) {
        up = here[k + j];
        down = here[-k - j];
        place += up < key[u] ? 1 : 0;
        place -= down > key[u] ? 1 : 0;
        again = again || down == key[u];
      }
    }
    at[u] = (uint32_t)place;
    if (valid && !again) atomicOr(&sFirst[place >> 5], 1u << (place & 31));
  }
  __syncthreads();
  {
    static_assert(CAP / 32 <= THREADS, "a word of bits per thread");
    const uint32_t count = tid < CAP / 32 ? __popc(sFirst[tid]) : 0u;
    const uint32_t incl = wave_inclusive_scan(count, lane);
    if (lane == 63) sWaveTot[wave] = incl;
    __syncthreads();
    uint32_t run = incl - count;
#pragma unroll
    for (int u = 0; u < CAP / 32 / 64; u++)
      if (u < wave) run += sWaveTot[u];
    if (tid < CAP / 32) sBefore[tid] = run;
    if (tid == CAP / 32 - 1) blockPartition[w] = ((int)(run + count) + W - 1) / W;
  }
  __syncthreads();
  asm volatile("" : "+s"(n));
  // an edge's rank: the first keys at or in front of its place, without the column's own
#pragma unroll
  for (int u = 0; u < ITEMS; u++) {
    if (u * THREADS >= n) continue;
    if (tid >= n - u * THREADS) continue;
    const uint32_t bits = sFirst[at[u] >> 5] & ((2u << (at[u] & 31u)) - 1u);
    ranks[u * THREADS + tid] = (int)(sBefore[at[u] >> 5] + __popc(bits)) - 1;
  }
}

// The mid windows of the queue.
template <int W>
__global__ __launch_bounds__(kMidThreads, 6) void window_rank_mid_kernel(
    const int32_t* __restrict__ rowPtr, const int32_t* __restrict__ colIdx, int N, int colBits,
    LongQueue queue, int32_t* __restrict__ blockPartition, int32_t* __restrict__ edgeToColumn,
    int32_t* __restrict__ edgeToRow, int* __restrict__ error) {
  extern __shared__ __align__(16) uint32_t smem[];
  const int listed = queue.size(false);
  for (int k = blockIdx.x; k < listed; k += (int)gridDim.x)
    rank_window_by_sort<W, kMidItems, kMidThreads>(queue.at(false, k), rowPtr, colIdx, N, colBits, smem,
                                                   blockPartition, edgeToColumn, edgeToRow, error);
}

// The large windows of the queue, those of more than kLargeMax edges by the bitset in several passes. One launch:
// the handful of windows of thousands of edges would each keep a launch of its own waiting (61M edges, 414
// windows of 1 921 to 11 001 edges: 18 + 25 + 5 us as three launches, 29 as one).
constexpr size_t rank_rest_lds(size_t bitset) {
  constexpr size_t sort = rank_sort_lds<kLargeItems, kLargeThreads>();
  return bitset > sort ? bitset : sort;
}
template <int W>
__global__ __launch_bounds__(kLargeThreads) void window_rank_rest_kernel(
    const int32_t* __restrict__ rowPtr, const int32_t* __restrict__ colIdx, int N,
    int colBits, int range, int nPasses, LongQueue queue, int32_t* __restrict__ blockPartition,
    int32_t* __restrict__ edgeToColumn, int32_t* __restrict__ edgeToRow,
    int* __restrict__ error) {
  extern __shared__ __align__(16) uint32_t smem[];
  const int listed = queue.size(true);
  for (int k = blockIdx.x; k < listed; k += (int)gridDim.x) {
    const int w = uniform(queue.at(true, k));
    const int n = rowPtr[min(w * 16 + 16, N)] - rowPtr[w * 16];
    __syncthreads();
    if (n > kLargeMax)
      rank_window_by_bitset<W, kLargeThreads>(w, rowPtr, colIdx, N, range, nPasses, 0, smem, blockPartition,
                                              edgeToColumn, edgeToRow, error);
    else if (n > kFourMax)
      rank_window_by_sort<W, kLargeItems, kLargeThreads>(w, rowPtr, colIdx, N, colBits, smem, blockPartition,
                                                         edgeToColumn, edgeToRow, error);
    else
      rank_window_by_sort<W, kFourItems, kLargeThreads>(w, rowPtr, colIdx, N, colBits, smem, blockPartition,
                                                       edgeToColumn, edgeToRow, error);
  }
}

// ------------------------------------------------- scan + window ordering
constexpr int kFinBlock = 1024;
// windows up to which one workgroup scans the counts and order_chunk orders them
constexpr int kFinSingleMax = 16384;

// Exclusive prefix of the block counts into rowWindowOffset and their total, by one workgroup: every
// wave owns a contiguous chunk of the windows, all of its loads in flight together.
__device__ __forceinline__ void scan_windows(const int32_t* __restrict__ blockPartition, int nRW,
                                             int32_t* __restrict__ rowWindowOffset,
                                             long long* __restrict__ nTcb) {
  constexpr int NW = kFinBlock / 64;
  constexpr int G = kFinSingleMax / kFinBlock;  // groups of 64 windows per wave at most
  __shared__ unsigned sWaveSum[NW];
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int chunk = (((nRW + NW - 1) / NW) + 63) & ~63;
  const int cBegin = min(wave * chunk, nRW);
  const int cEnd = min(cBegin + chunk, nRW);
  unsigned v[G], sum = 0;
#pragma unroll
  for (int k = 0; k < G; k++) {
    const int i = cBegin + 64 * k + lane;
    v[k] = i < cEnd ? (unsigned)blockPartition[i] : 0u;
  }
#pragma unroll
  for (int k = 0; k < G; k++) sum += v[k];
  sum = wave_inclusive_scan(sum, lane);
  if (lane == 63) sWaveSum[wave] = sum;
  __syncthreads();
  unsigned carry = 0, total = 0;
#pragma unroll
  for (int k = 0; k < NW; k++) {
    const unsigned t = sWaveSum[k];
    if (k < wave) carry += t;
    total += t;
  }
#pragma unroll
  for (int k = 0; k < G; k++) {
    if (64 * k >= chunk) break;
    const int i = cBegin + 64 * k + lane;
    const unsigned incl = wave_inclusive_scan(v[k], lane);
    if (i < cEnd) rowWindowOffset[i + 1] = (int)(carry + incl);
    carry += (unsigned)__builtin_amdgcn_readlane((int)incl, 63);
  }
  if (threadIdx.x == 0) {
    rowWindowOffset[0] = 0;
    *nTcb = (long long)total;
  }
}

// Positions of windows first .. first + TB - 1 (first: a multiple of TB) in the order by descending
// block count, ties ascending, into sortedRowWindows, by one workgroup: the counts of all windows
// become a histogram in LDS (low half of a word: windows with that many blocks, high half: those in
// front of `first`), its sums from the top the places. No workgroup waits for another one, and
// nRW / TB of them share the work (a radix sort by one workgroup of 1024 threads took 21 us for
// 10 584 windows, 30 us for 14 561). hist: nBins words, a multiple of TB. blocks(i): window i's count,
// not negative.
// ROWS: more windows than 16 bits count, so the two halves are words of their own, hist 2 nBins of them;
// and the histogram of the first nBins - 1 counts is added up from `rows`, one per TB windows
// (finalize_partials_kernel): one after the other for all windows, the LDS additions of 153 000 windows
// take 60 us, of 64 lanes a handful of distinct counts.
// Counts from nBins - 1 on share the last bin; while it holds any, another round orders the windows
// of the next nBins - 1 counts, so a call takes as many rounds as its largest count asks for (at most
// nine: 32 769 blocks of 8 columns, 4096 bins); nearly every graph takes one. Wide windows that compare
// themselves with all others instead, one after the other in a wave, are slow where there are many:
// 100 000 nodes of 2 500 edges, 8-column blocks, 6 245 of 6 250 windows: a preprocessing call of 7.54
// instead of 7.01 ms; 262 000 nodes of 2 200 edges: 17.01 instead of 15.03 ms.
template <int TB, bool ROWS = false, typename BlocksOf>
__device__ __forceinline__ void order_chunk(const BlocksOf& blocks, int nRW, int first, int nBins,
                                            int32_t* __restrict__ sortedRowWindows, uint32_t* hist,
                                            const uint16_t* __restrict__ rows = nullptr) {
  static_assert(kFinSingleMax < 0x8000, "two counters of windows per word");
  constexpr int NW = TB / 64;
  constexpr int U = 4;  // counts of a thread in flight together
  __shared__ unsigned sBinTot[NW];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int top = nBins - 1;
  const int count = first + tid < nRW ? blocks(first + tid) : -1;
  uint32_t* const ahead = ROWS ? hist + nBins : hist;  // windows in front of `first`, then the places
  const auto windows_in = [&](int bin) { return ROWS ? hist[bin] : hist[bin] & 0xFFFFu; };
  for (int low = 0;; low += top) {  // windows of low .. low + top - 1 blocks
    if (ROWS && low == 0) {
      const int nRows = (nRW + TB - 1) / TB, own = first / TB;
      for (int b = tid; b < nBins; b += TB) {
        unsigned all = 0, front = 0;
#pragma unroll 16
        for (int r = 0; r < nRows; r++) {
          const unsigned n = rows[(size_t)r * nBins + b];
          all += n;
          front += r < own ? n : 0u;
        }
        hist[b] = all;
        ahead[b] = front;
      }
    } else {
      for (int i = tid; i < (ROWS ? 2 : 1) * nBins; i += TB) hist[i] = 0u;
      __syncthreads();
      for (int i0 = 0; i0 < nRW; i0 += U * TB) {
        int c[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
          const int i = i0 + u * TB + tid;
          c[u] = i < nRW ? min(blocks(i) - low, top) : -1;
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
          // counts cluster, and lanes that name the same bin are served one after the other: the lanes
          // that agree with the group's first one are counted with one ballot and added once
          const int c0 = __builtin_amdgcn_readfirstlane(c[u]);
          const bool front = i0 + u * TB + wave * 64 < first;
          const unsigned one = !ROWS && front ? 0x10001u : 1u;
          const unsigned long long same = __ballot(c[u] == c0);
          if (c[u] >= 0 && c[u] != c0) {
            atomicAdd(&hist[c[u]], one);
            if (ROWS && front) atomicAdd(&ahead[c[u]], 1u);
          }
          if (c0 >= 0 && lane == 0) {
            atomicAdd(&hist[c0], one * (unsigned)__popcll(same));
            if (ROWS && front) atomicAdd(&ahead[c0], (unsigned)__popcll(same));
          }
        }
      }
    }
    __syncthreads();
    const bool wider = windows_in(top) != 0u;  // windows left for the rounds to come
    {  // where each bin's windows of this chunk start; thread t owns nBins / TB bins from the top
      const int per = nBins / TB;
      unsigned total = 0;
      for (int k = 0; k < per; k++) total += windows_in(top - (tid * per + k));
      const unsigned incl = wave_inclusive_scan(total, lane);
      if (lane == 63) sBinTot[wave] = incl;
      __syncthreads();
      unsigned run = incl - total;
#pragma unroll
      for (int k = 0; k < NW; k++) run += k < wave ? sBinTot[k] : 0u;
      for (int k = 0; k < per; k++) {
        const int b = top - (tid * per + k);
        const uint32_t in = windows_in(b);
        ahead[b] = run + (ROWS ? ahead[b] : hist[b] >> 16);
        run += in;
      }
    }
    const int bin = count - low;
    const bool binned = bin >= 0 && bin < top;
    unsigned long long peers = __ballot(binned);
    for (int b = 0; (top >> b) != 0; b++) {
      const unsigned long long bal = __ballot((bin >> b) & 1);
      peers &= ((bin >> b) & 1) ? bal : ~bal;
    }
    for (int turn = 0; turn < NW; turn++) {  // ties go by window: one wave after the other
      __syncthreads();
      if (wave != turn) continue;
      const unsigned at = binned ? ahead[bin] : 0u;
      wave_lds_sync();
      if (binned) {
        sortedRowWindows[at + __popcll(peers & ((1ull << lane) - 1ull))] = first + tid;
        if ((peers >> lane) == 1ull) ahead[bin] = at + (unsigned)__popcll(peers);
      }
    }
    if (!wider) return;
    __syncthreads();  // the bins are free again
  }
}
// bins for the counts that the windows of a graph can have, within 16 KiB
constexpr int order_bins(int N, int W) {
  const int bins = ((N / W + 2) + 1023) & ~1023;
  return bins < 4096 ? bins : 4096;
}

__global__ __launch_bounds__(kFinBlock) void window_scan_kernel(
    const int32_t* __restrict__ blockPartition, int nRW, int32_t* __restrict__ rowWindowOffset,
    long long* __restrict__ nTcb) {
  scan_windows(blockPartition, nRW, rowWindowOffset, nTcb);
}

// workgroup 0 scans the counts, each of the others orders kFinBlock windows
__global__ __launch_bounds__(kFinBlock) void finalize_count_kernel(
    const int32_t* __restrict__ blockPartition, int nRW, int nBins,
    int32_t* __restrict__ rowWindowOffset, int32_t* __restrict__ sortedRowWindows,
    long long* __restrict__ nTcb) {
  extern __shared__ __align__(16) uint32_t finLds[];
  if (blockIdx.x == 0)
    scan_windows(blockPartition, nRW, rowWindowOffset, nTcb);
  else
    order_chunk<kFinBlock>([=](int i) { return blockPartition[i]; }, nRW,
                           ((int)blockIdx.x - 1) * kFinBlock, nBins, sortedRowWindows, finLds);
}

// The order alone, for attention calls without one. It only has to start the long windows first, so
// counts of 512 blocks and more share 64 bins an octave: 1024 bins in all, one round below
// 131 000 blocks. 4 to 6 us.
constexpr int kOrderOnlyBins = 1024;
constexpr int kOrderOnlyThreads = 512;
__global__ __launch_bounds__(kOrderOnlyThreads) void window_order_kernel(
    const int32_t* __restrict__ rowWindowOffset, int nRW, int32_t* __restrict__ order) {
  __shared__ uint32_t hist[kOrderOnlyBins];
  auto blocks = [=](int i) {
    // offsets that descend (not from preprocessing) stand for an empty window, as in the attention
    // kernels: every window has its place, whatever the caller's offsets hold
    const int c = max((int)((unsigned)rowWindowOffset[i + 1] - (unsigned)rowWindowOffset[i]), 0);
    const int octave = 31 - __builtin_clz((unsigned)c | 1u);
    return c < 512 ? c : 512 + (octave - 9) * 64 + ((c >> (octave - 6)) & 63);
  };
  order_chunk<kOrderOnlyThreads>(blocks, nRW, (int)blockIdx.x * kOrderOnlyThreads, kOrderOnlyBins,
                                 order, hist);
}

// ---- the same scan + stable sort spread over many workgroups, for graphs with many windows.
// Every WAVE of the grid owns a contiguous chunk of the windows (chunks in wave order), exactly as
// the waves of scan_windows do; what they exchange through LDS and block barriers
// goes through small global arrays and kernel boundaries here:
//   finalize_partials_kernel   per-wave sum and maximum of the block counts
//   finalize_scan_kernel       rowWindowOffset of the chunk (carry = sums of the earlier waves),
//                              total and maximum into the header, digit histogram of pass 0
//   finalize_scatter_kernel    one pass: start of (digit, wave) from every wave's histogram, then
//                              the in-order scatter of the chunk
//   finalize_histogram_kernel  digit histogram of the next pass (its input is the scattered
//                              order, complete only at the kernel boundary)
// The number of passes depends on the largest count, known on the device only: the host enqueues
// as many passes as the window count could need and the surplus kernels return at once.
constexpr int kFinDigitBits = 6;
constexpr int kFinBins = 1 << kFinDigitBits;

struct FinChunk {
  int begin, end;
};
__device__ __forceinline__ FinChunk fin_chunk(int nRW, int totalWaves, int gw) {
  const int chunk = (((nRW + totalWaves - 1) / totalWaves) + 63) & ~63;
  FinChunk c;
  c.begin = min(gw * chunk, nRW);
  c.end = min(c.begin + chunk, nRW);
  return c;
}
__device__ __forceinline__ unsigned long long fin_digit_peers(bool valid, int dgt) {
  unsigned long long peers = __ballot(valid);
#pragma unroll
  for (int b = 0; b < kFinDigitBits; b++) {
    const unsigned long long bal = __ballot((dgt >> b) & 1);
    peers &= ((dgt >> b) & 1) ? bal : ~bal;
  }
  return peers;
}
__device__ __forceinline__ int fin_passes(int maxC) {
  int nBits = 0;
  while ((maxC >> nBits) != 0) nBits++;
  return (nBits + kFinDigitBits - 1) / kFinDigitBits;
}

// With rows (not null: a wave's chunk is 512 windows then): the histogram of every kOrderRowWindows
// windows' counts as well, counts from kOrderRowBins - 1 on in the last bin, for order_chunk.
constexpr int kOrderRowWindows = 1024, kOrderRowBins = 1024;
__global__ __launch_bounds__(256) void finalize_partials_kernel(
    const int32_t* __restrict__ blockPartition, int nRW, int totalWaves,
    unsigned* __restrict__ waveSum, int* __restrict__ waveMax, uint16_t* __restrict__ rows) {
  constexpr int ROWS = 2048 / kOrderRowWindows;  // of a workgroup
  __shared__ uint32_t sHist[ROWS][kOrderRowBins];
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int gw = blockIdx.x * 4 + wave;
  const FinChunk c = fin_chunk(nRW, totalWaves, gw);  // empty if gw >= totalWaves
  if (rows) {
    for (int i = threadIdx.x; i < ROWS * kOrderRowBins; i += 256) sHist[0][i] = 0u;
    __syncthreads();
  }
  unsigned sum = 0;
  int mx = 0;
  for (int i = c.begin + lane; i < c.end; i += 64) {
    const int v = blockPartition[i];
    sum += (unsigned)v;
    mx = max(mx, v);
    if (rows) atomicAdd(&sHist[wave * ROWS / 4][min(v, kOrderRowBins - 1)], 1u);
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    sum += __shfl_xor(sum, off);
    mx = max(mx, __shfl_xor(mx, off));
  }
  if (lane == 0 && gw < totalWaves) {
    waveSum[gw] = sum;
    waveMax[gw] = mx;
  }
  if (rows) {
    __syncthreads();
    const int nRows = (nRW + kOrderRowWindows - 1) / kOrderRowWindows;
    for (int r = 0; r < ROWS; r++) {
      const int row = (int)blockIdx.x * ROWS + r;
      for (int i = threadIdx.x; row < nRows && i < kOrderRowBins; i += 256)
        rows[(size_t)row * kOrderRowBins + i] = (uint16_t)sHist[r][i];
    }
  }
}

// digit histogram of a wave's chunk into hist[gw * 64 + digit]; sBins: 64 LDS counters of the wave
__device__ __forceinline__ void fin_histogram(const int32_t* __restrict__ keys, bool fromCounts,
                                              int maxC, FinChunk c, int shift, int lane,
                                              unsigned* sBins, unsigned* __restrict__ histRow) {
  sBins[lane] = 0;
  wave_lds_sync();
  const unsigned long long ltMask = (1ull << lane) - 1ull;
  int keyNext = (c.begin + lane < c.end) ? keys[c.begin + lane] : 0;
  for (int base = c.begin; base < c.end; base += 64) {
    const int i = base + lane;
    const bool valid = i < c.end;
    const int raw = keyNext;
    keyNext = (i + 64 < c.end) ? keys[i + 64] : 0;
    const int key = fromCounts ? maxC - raw : raw;
    const int dgt = (key >> shift) & (kFinBins - 1);
    const unsigned long long peers = fin_digit_peers(valid, dgt);
    // the first lane of every group of equal digits adds the group to its bin
    if (valid && (peers & ltMask) == 0ull) sBins[dgt] += __popcll(peers);
  }
  wave_lds_sync();
  histRow[lane] = sBins[lane];
}

__global__ __launch_bounds__(256) void finalize_scan_kernel(
    const int32_t* __restrict__ blockPartition, int nRW, int totalWaves,
    const unsigned* __restrict__ waveSum, const int* __restrict__ waveMax,
    int32_t* __restrict__ rowWindowOffset, unsigned* __restrict__ hist,
    WsHeader* __restrict__ hdr, long long* __restrict__ nTcb) {
  __shared__ unsigned sBins[4][kFinBins];
  const int lane = threadIdx.x & 63;
  const int gw = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (gw >= totalWaves) return;
  const FinChunk c = fin_chunk(nRW, totalWaves, gw);
  unsigned carry = 0, total = 0;
  int maxC = 0;
#pragma unroll 4
  for (int k = lane; k < totalWaves; k += 64) {
    const unsigned t = waveSum[k];
    if (k < gw) carry += t;
    total += t;
    maxC = max(maxC, waveMax[k]);
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    carry += __shfl_xor(carry, off);
    total += __shfl_xor(total, off);
    maxC = max(maxC, __shfl_xor(maxC, off));
  }
  for (int base = c.begin; base < c.end; base += 64) {
    const int i = base + lane;
    const unsigned v = (i < c.end) ? (unsigned)blockPartition[i] : 0u;
    const unsigned incl = wave_inclusive_scan(v, lane);
    if (i < c.end) rowWindowOffset[i + 1] = (int)(carry + incl);
    carry += __shfl(incl, 63);
  }
  if (gw == 0 && lane == 0) {
    rowWindowOffset[0] = 0;
    *nTcb = (long long)total;
    hdr->maxCount = maxC;
  }
  if (hist)  // null: the order is not made here
    fin_histogram(blockPartition, true, maxC, c, 0, lane, sBins[threadIdx.x >> 6],
                  hist + (size_t)gw * kFinBins);
}

__global__ __launch_bounds__(256) void finalize_histogram_kernel(
    int nRW, int totalWaves, int pass, const int32_t* __restrict__ keysA,
    const int32_t* __restrict__ keysB, unsigned* __restrict__ hist,
    const WsHeader* __restrict__ hdr) {
  __shared__ unsigned sBins[4][kFinBins];
  const int lane = threadIdx.x & 63;
  const int gw = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (gw >= totalWaves) return;
  const int maxC = hdr->maxCount;
  const int nPass = fin_passes(maxC);
  if (pass >= nPass) return;
  // the keys this pass reads are the ones the previous pass wrote
  const bool prevToOut = ((nPass - pass) & 1) == 0;
  const int32_t* kSrc = prevToOut ? keysA : keysB;
  fin_histogram(kSrc, false, maxC, fin_chunk(nRW, totalWaves, gw), pass * kFinDigitBits, lane,
                sBins[threadIdx.x >> 6], hist + (size_t)gw * kFinBins);
}

__global__ __launch_bounds__(256) void finalize_scatter_kernel(
    const int32_t* __restrict__ blockPartition, int nRW, int totalWaves, int pass,
    int32_t* __restrict__ sortedRowWindows, int32_t* __restrict__ keysA,
    int32_t* __restrict__ keysB, int32_t* __restrict__ valsTmp, const unsigned* __restrict__ hist,
    const WsHeader* __restrict__ hdr) {
  __shared__ unsigned sPos[4][kFinBins];
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int gw = blockIdx.x * 4 + wave;
  if (gw >= totalWaves) return;
  const FinChunk c = fin_chunk(nRW, totalWaves, gw);
  const int maxC = hdr->maxCount;
  const int nPass = fin_passes(maxC);
  if (nPass == 0) {  // every window is empty: the order is the identity
    if (pass == 0)
      for (int i = c.begin + lane; i < c.end; i += 64) sortedRowWindows[i] = i;
    return;
  }
  if (pass >= nPass) return;
  const int shift = pass * kFinDigitBits;
  const bool toOut = ((nPass - 1 - pass) & 1) == 0;
  int32_t* kDst = toOut ? keysA : keysB;
  int32_t* vDst = toOut ? sortedRowWindows : valsTmp;
  const int32_t* kSrc = toOut ? keysB : keysA;
  const int32_t* vSrc = toOut ? valsTmp : sortedRowWindows;
  // start of (digit = lane, this wave): all smaller digits, then the same digit in earlier waves
  unsigned digitTotal = 0, before = 0;
#pragma unroll 8
  for (int k = 0; k < totalWaves; k++) {
    const unsigned cnt = hist[(size_t)k * kFinBins + lane];
    digitTotal += cnt;
    before += (k < gw) ? cnt : 0u;
  }
  const unsigned start = wave_inclusive_scan(digitTotal, lane) - digitTotal + before;
  sPos[wave][lane] = start;
  wave_lds_sync();
  const unsigned long long ltMask = (1ull << lane) - 1ull;
  auto load_key = [&](int i) {
    return (i < c.end) ? ((pass == 0) ? (maxC - blockPartition[i]) : kSrc[i]) : 0;
  };
  auto load_val = [&](int i) { return (i < c.end) ? ((pass == 0) ? i : vSrc[i]) : 0; };
  int keyNext = load_key(c.begin + lane);
  int valNext = load_val(c.begin + lane);
  for (int base = c.begin; base < c.end; base += 64) {
    const int i = base + lane;
    const bool valid = i < c.end;
    const int key = keyNext, val = valNext;
    keyNext = load_key(i + 64);
    valNext = load_val(i + 64);
    const int dgt = (key >> shift) & (kFinBins - 1);
    const unsigned long long peers = fin_digit_peers(valid, dgt);
    if (valid) {
      const unsigned pos = sPos[wave][dgt] + __popcll(peers & ltMask);
      kDst[pos] = key;
      vDst[pos] = val;
    }
    // the last peer moves the digit's running position (the wave's LDS accesses stay in order)
    if (valid && (peers >> lane) == 1ull) sPos[wave][dgt] += __popcll(peers);
  }
}

// ------------------------------------------------------------------ phase 2
// Any window, TC blocks at a time: rows may hold repeated or descending columns. sCnt
// ([TC * 16]) and sBm ([TC * WPT]) are the caller's LDS; sRow holds the window's 17 row pointers;
// *sUnsorted must be 0 on entry. Every thread of the workgroup calls this.
template <int W, int TB>
__device__ __forceinline__ void fill_window_generic(
    const int32_t* __restrict__ colIdx, const int32_t* __restrict__ edgeToColumn, int w, int base,
    int nb, const int TC, int32_t* __restrict__ tcblockRowid, uint8_t* __restrict__ tcblocktileId,
    int32_t* __restrict__ tcblockOffset, int32_t* __restrict__ sparseAToXidx,
    unsigned long long* __restrict__ bitmap, unsigned* sCnt, unsigned long long* sBm,
    const int* sRow, unsigned* sWaveTot, unsigned* sUnsortedPtr) {
  constexpr int WPT = 16 * W / 64;  // bitmap words per TC block
  constexpr int LOGW = (W == 16) ? 4 : 3;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int eS = sRow[0], eE = sRow[16];
  const unsigned long long ltMask = (1ull << lane) - 1ull;
  unsigned carry = (unsigned)eS;  // absolute edge position where the next TC block starts

  for (int tc0 = 0; tc0 < nb; tc0 += TC) {
    const int nt = min(TC, nb - tc0);
    for (int i = tid; i < nt * 16; i += TB) sCnt[i] = 0;
    for (int i = tid; i < nt * WPT; i += TB) sBm[i] = 0ull;
    __syncthreads();
    // four edges per thread and step, loads first: the LDS atomics of one edge then overlap the
    // memory latency of the next ones
    for (int e0 = eS + tid; e0 < eE; e0 += 4 * TB) {
      int ecs[4], cols[4];
#pragma unroll
      for (int u = 0; u < 4; u++) {
        const int e = e0 + u * TB;
        ecs[u] = (e < eE) ? edgeToColumn[e] : -1;
        cols[u] = (e < eE) ? colIdx[e] : 0;
      }
      if (tc0 == 0) {
        // once per window: which rows are strictly ascending (every edge against its left
        // neighbour in the same row)
#pragma unroll
        for (int u = 0; u < 4; u++) {
          const int e = e0 + u * TB;
          if (e < eE && e > eS) {
            const int r = row_of_edge(sRow, e);
            if (e > sRow[r] && colIdx[e - 1] >= cols[u]) atomicOr(sUnsortedPtr, 1u << r);
          }
        }
      }
#pragma unroll
      for (int u = 0; u < 4; u++) {
        const int e = e0 + u * TB;
        const int ec = ecs[u];
        const int t = (ec >> LOGW) - tc0;
        if (ec >= 0 && (unsigned)t < (unsigned)nt) {
          const int r = row_of_edge(sRow, e);
          const int cl = ec & (W - 1);
          atomicAdd(&sCnt[t * 16 + r], 1u);
          // 8x8 sub-blocks in column-major order, row-major and MSB-first inside
          const int sub = (cl >> 3) * (W / 8) + (r >> 3);
          atomicOr(&sBm[t * WPT + sub], 1ull << (63 - ((r & 7) * 8 + (cl & 7))));
          sparseAToXidx[(int64_t)(base + tc0 + t) * W + cl] = cols[u];
        }
      }
    }
    __syncthreads();
    for (int tb = 0; tb < nt; tb += TB) {
      const int t = tb + tid;
      unsigned nnz = 0;
      if (t < nt) {
#pragma unroll
        for (int r = 0; r < 16; r++) nnz += sCnt[t * 16 + r];
      }
      const unsigned incl = wave_inclusive_scan(nnz, lane);
      if (lane == 63) sWaveTot[wave] = incl;
      __syncthreads();
      unsigned waveOff = 0, tileTot = 0;
#pragma unroll
      for (int v = 0; v < TB / 64; v++) {
        const unsigned x = sWaveTot[v];
        if (v < wave) waveOff += x;
        tileTot += x;
      }
      if (t < nt) {
        const int64_t gt = (int64_t)base + tc0 + t;
        unsigned run = carry + waveOff + incl - nnz;
        tcblockOffset[gt] = (int)run;
        tcblockRowid[gt] = w;
        if (*sUnsortedPtr == 0u) {
          // Every row of the window is strictly ascending, so the block's tile ids are its set
          // bits read row by row, left to right (src/utils.cu:213-223 walks the edges in that
          // order): this thread writes them all, next to the previous block's.
          unsigned long long words[WPT];
#pragma unroll
          for (int k = 0; k < WPT; k++) words[k] = sBm[t * WPT + k];
          walk_tile_ids<W>(words, tcblocktileId, run);
        }
#pragma unroll
        for (int r = 0; r < 16; r++) {
          const unsigned c = sCnt[t * 16 + r];
          sCnt[t * 16 + r] = run;
          run += c;
        }
        // bitmap words out; a compacted slot that no edge named keeps column id 0
        unsigned colMask = 0;  // bit cl set <=> slot cl holds a column
#pragma unroll
        for (int k = 0; k < WPT; k++) {
          const unsigned long long word = sBm[t * WPT + k];
          bitmap[gt * WPT + k] = word;
          unsigned long long x = word;
          x |= x >> 32;
          x |= x >> 16;
          x |= x >> 8;
          const unsigned rowOr = (unsigned)(x & 0xFFull);  // bit (7 - cl%8)
          const int colHalf = (W == 16) ? (k >> 1) : 0;
#pragma unroll
          for (int b = 0; b < 8; b++)
            if (rowOr & (0x80u >> b)) colMask |= 1u << (colHalf * 8 + b);
        }
#pragma unroll
        for (int cl = 0; cl < W; cl++)
          if (!((colMask >> cl) & 1u)) sparseAToXidx[gt * W + cl] = 0;
      }
      carry += tileTot;
      __syncthreads();
    }
    // Windows with some row that is not strictly ascending. Tile ids sit in CSR edge order
    // inside a TC block (src/utils.cu:213-223): position = start of (block, row) + number of
    // earlier edges of that row in the block. In a strictly ascending row those are exactly the
    // bits left of the edge's own bit in the block's bitmap row, so every edge of such a row
    // finds its place on its own; the other rows are replayed in order below.
    const unsigned unsorted = *sUnsortedPtr;
    for (int e = eS + tid; unsorted != 0u && e < eE; e += TB) {
      const int ec = edgeToColumn[e];
      const int t = (ec >> LOGW) - tc0;
      if ((unsigned)t >= (unsigned)nt) continue;
      const int r = row_of_edge(sRow, e);
      if ((unsorted >> r) & 1u) continue;
      const int cl = ec & (W - 1);
      const int shift = 8 * (7 - (r & 7));
      unsigned before = 0;
      if (W == 16 && cl >= 8)
        before = __popc((unsigned)(sBm[t * WPT + (r >> 3)] >> shift) & 0xFFu);
      const unsigned own =
          (unsigned)(sBm[t * WPT + (cl >> 3) * (W / 8) + (r >> 3)] >> shift) & 0xFFu;
      before += __popc(own >> (8 - (cl & 7)));
      tcblocktileId[sCnt[t * 16 + r] + before] = (uint8_t)(r * W + cl);
    }
    // rows with repeated or descending columns: a wave replays the whole row in order
    for (int r = wave; r < 16; r += TB / 64) {
      if (!((unsorted >> r) & 1u)) continue;
      const int rs = sRow[r], re = sRow[r + 1];
      int ecNext = (rs + lane < re) ? edgeToColumn[rs + lane] : 0;
      for (int eb = rs; eb < re; eb += 64) {
        const int e = eb + lane;
        const bool valid = e < re;
        const int ec = ecNext;
        ecNext = (e + 64 < re) ? edgeToColumn[e + 64] : 0;  // next batch, in flight during this one
        const int t = (ec >> LOGW) - tc0;
        const bool inr = valid && (unsigned)t < (unsigned)nt;
        unsigned long long peers = __ballot(inr);
        if (peers == 0ull) continue;
        // lanes whose edges fall into the same block: agree on every bit of t (t < TC)
        for (int b = 0; ((TC - 1) >> b) != 0; b++) {
          const unsigned long long bal = __ballot((t >> b) & 1);
          peers &= ((t >> b) & 1) ? bal : ~bal;
        }
        unsigned pos = 0;
        if (inr) pos = sCnt[t * 16 + r] + __popcll(peers & ltMask);
        if (inr) tcblocktileId[pos] = (uint8_t)(r * W + (ec & (W - 1)));
        // the highest peer lane advances the running position of (block, row)
        if (inr && (peers >> lane) == 1ull) sCnt[t * 16 + r] += __popcll(peers);
      }
    }
    __syncthreads();
  }
}


// One workgroup (or one wave) per window. Windows whose rows are all strictly ascending (every
// CSR that is sorted and free of repeated entries) take the short way: every edge sets its bit in
// the LDS bitmaps and drops its column id into the LDS copy of the block's id slots; a block's
// non-zero count is then the population count of its bitmap, its tile ids are its set bits read
// row by row (src/utils.cu:213-223 walks the edges in exactly that order), and bitmaps and ids
// leave LDS as contiguous runs. A window with a repeated or descending column is handed to
// fill_window_generic. TC blocks of LDS at a time on the short way, TCG on the general one.
// LDS of fill_one_window: sRaw
template <int W>
constexpr size_t fill_lds_bytes(int tc, int tcg) {
  const size_t fast = (size_t)tc * (2 * W + 4 * W), generic = (size_t)tcg * (64 + 2 * W);
  return fast > generic ? fast : generic;
}
template <int W, int TB, int TC, int TCG>
__device__ __forceinline__ void fill_one_window(
    int w, int base, int nb, const int32_t* __restrict__ rowPtr,
    const int32_t* __restrict__ colIdx, int N, int E, const int32_t* __restrict__ edgeToColumn,
    unsigned char* sRaw, int32_t* __restrict__ tcblockRowid,
    uint8_t* __restrict__ tcblocktileId, int32_t* __restrict__ tcblockOffset,
    int32_t* __restrict__ sparseAToXidx, unsigned long long* __restrict__ bitmap) {
  constexpr int WPT = 16 * W / 64;  // bitmap words per TC block
  constexpr int LOGW = (W == 16) ? 4 : 3;
  __shared__ int sRow[17];
  __shared__ unsigned sWaveTot[TB / 64];
  __shared__ unsigned sUnsorted;  // bit r: row r's columns are not strictly ascending
  unsigned long long* sBm = reinterpret_cast<unsigned long long*>(sRaw);       // [TC * WPT]
  int32_t* sIds = reinterpret_cast<int32_t*>(sRaw + TC * WPT * 8);             // [TC * W]

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  if (tid == 0) sUnsorted = 0u;
  if (nb == 0) return;
  const int r0 = w * 16;
  if (tid < 17) sRow[tid] = rowPtr[min(r0 + tid, N)];
  __syncthreads();
  const int eS = sRow[0], eE = sRow[16];
  unsigned carry = (unsigned)eS;  // absolute edge position where the next TC block starts

  for (int tc0 = 0; tc0 < nb; tc0 += TC) {
    const int nt = min(TC, nb - tc0);
    for (int i = tid; i < nt * WPT; i += TB) sBm[i] = 0ull;
    for (int i = tid; i < nt * W; i += TB) sIds[i] = 0;
    __syncthreads();
    // Four CONSECUTIVE edges per thread (one 16-byte load of ranks, one of column ids, from a
    // 16-byte aligned index). Consecutive edges of a row fall into the same bitmap byte (row r
    // of an 8-column sub-block) up to eight at a time, so a thread first ORs its edges' bits
    // together per byte and then issues one 32-bit LDS atomic per distinct byte.
    unsigned* sBmWords = reinterpret_cast<unsigned*>(sBm);
    for (int e0 = (eS & ~3) + 4 * tid; e0 < eE; e0 += 4 * TB) {
      int ecs[4], cols[4];
      if (e0 + 4 <= E) {
        const int4 a = *reinterpret_cast<const int4*>(edgeToColumn + e0);
        const int4 b = *reinterpret_cast<const int4*>(colIdx + e0);
        ecs[0] = a.x; ecs[1] = a.y; ecs[2] = a.z; ecs[3] = a.w;
        cols[0] = b.x; cols[1] = b.y; cols[2] = b.z; cols[3] = b.w;
      } else {
#pragma unroll
        for (int u = 0; u < 4; u++) {
          ecs[u] = (e0 + u < E) ? edgeToColumn[e0 + u] : 0;
          cols[u] = (e0 + u < E) ? colIdx[e0 + u] : 0;
        }
      }
      int left = (tc0 == 0 && e0 > eS) ? colIdx[e0 - 1] : -1;
      const int eLo = e0 > eS ? e0 : eS;
      const int eHi = (e0 + 3 < eE - 1) ? e0 + 3 : eE - 1;
      const int rLo = row_of_edge(sRow, eLo);
      const int rHi = row_of_edge(sRow, eHi);
      int curKey = -1;
      unsigned curMask = 0;
#pragma unroll
      for (int u = 0; u < 4; u++) {
        const int e = e0 + u;
        const bool valid = e >= eS && e < eE;
        const int r = (rLo == rHi) ? rLo : (valid ? row_of_edge(sRow, e) : rLo);
        // once per window: is every edge right of its left neighbour in the same row?
        if (tc0 == 0 && valid && e > sRow[r] && left >= cols[u]) atomicOr(&sUnsorted, 1u << r);
        left = cols[u];
        const int t = (ecs[u] >> LOGW) - tc0;
        if (valid && (unsigned)t < (unsigned)nt) {
          const int cl = ecs[u] & (W - 1);
          sIds[t * W + cl] = cols[u];
          // 8x8 sub-blocks in column-major order; byte 7 - r%8 of the sub-block's word is row
          // r%8, MSB first
          const int sub = (cl >> 3) * (W / 8) + (r >> 3);
          const int key = (t * WPT + sub) * 8 + 7 - (r & 7);
          const unsigned m8 = 0x80u >> (cl & 7);
          if (key == curKey) {
            curMask |= m8;
          } else {
            if (curKey >= 0) atomicOr(&sBmWords[curKey >> 2], curMask << (8 * (curKey & 3)));
            curKey = key;
            curMask = m8;
          }
        }
      }
      if (curKey >= 0) atomicOr(&sBmWords[curKey >> 2], curMask << (8 * (curKey & 3)));
    }
    __syncthreads();
    if (sUnsorted != 0u) break;  // known after the first pass over the window's edges
    for (int tb = 0; tb < nt; tb += TB) {
      const int t = tb + tid;
      unsigned long long words[WPT];
      unsigned nnz = 0;
      if (t < nt) {
#pragma unroll
        for (int k = 0; k < WPT; k++) {
          words[k] = sBm[t * WPT + k];
          nnz += __popcll(words[k]);
        }
      }
      const unsigned incl = wave_inclusive_scan(nnz, lane);
      if (lane == 63) sWaveTot[wave] = incl;
      __syncthreads();
      unsigned waveOff = 0, tileTot = 0;
#pragma unroll
      for (int v = 0; v < TB / 64; v++) {
        const unsigned x = sWaveTot[v];
        if (v < wave) waveOff += x;
        tileTot += x;
      }
      if (t < nt) {
        const int64_t gt = (int64_t)base + tc0 + t;
        unsigned pos = carry + waveOff + incl - nnz;
        tcblockOffset[gt] = (int)pos;
        tcblockRowid[gt] = w;
        // tile ids: the block's set bits read row by row (each lane walks its own block; the
        // byte stores of neighbouring lanes fall next to each other)
        walk_tile_ids<W>(words, tcblocktileId, pos);
      }
      carry += tileTot;
      __syncthreads();
    }
    // bitmaps and column ids of the chunk as contiguous runs (unused id slots stay 0)
    {
      unsigned long long* bmDst = bitmap + ((int64_t)base + tc0) * WPT;
      for (int i = tid; i < nt * WPT; i += TB) bmDst[i] = sBm[i];
      int32_t* idDst = sparseAToXidx + ((int64_t)base + tc0) * W;
      for (int i = tid; i < nt * W; i += TB) idDst[i] = sIds[i];
    }
    __syncthreads();
  }
  if (sUnsorted != 0u) {
    // repeated or descending columns somewhere in the window: start over on the general way
    __syncthreads();
    if (tid == 0) sUnsorted = 0u;
    __syncthreads();
    unsigned* gCnt = reinterpret_cast<unsigned*>(sRaw);                                  // [TCG*16]
    unsigned long long* gBm = reinterpret_cast<unsigned long long*>(sRaw + TCG * 64);    // [TCG*WPT]
    fill_window_generic<W, TB>(colIdx, edgeToColumn, w, base, nb, TCG, tcblockRowid,
                               tcblocktileId, tcblockOffset, sparseAToXidx, bitmap, gCnt, gBm, sRow,
                               sWaveTot, &sUnsorted);
  }
}

// Windows of at most kBinsMax edges: one wave per window, everything in its LDS slice. Every edge sets
// its bit in the window's bitmaps and drops its column into the ids; two lanes per TC block then walk
// the set bits row by row (a block of a sparse graph has 17, most of a walk's time is the fullest
// dword among the lanes), and bitmaps, ids and tile ids leave as whole words. Bound by the issue of
// vector instructions. Workgroups of one wave, 27 per CU (of four: 260 instead of 220 us for the 149k
// such windows of a 61M-edge graph).
template <int W>
struct alignas(16) FillShortLds {  // of one wave
  static constexpr int MAXB = (kBinsMax + W - 1) / W;  // TC blocks of a window at most
  unsigned long long bm[MAXB * (16 * W / 64)];
  uint32_t ids[MAXB * W];  // later the tile ids, kBinsMax + 8 bytes
  alignas(8) uint32_t mark[kBinsMax / 32 + 2];
};
template <int W>
__device__ __forceinline__ void fill_short_window(
    int w, int base, int nb, const int32_t* __restrict__ rowPtr,
    const int32_t* __restrict__ colIdx, int N, const int32_t* __restrict__ edgeToColumn,
    const LongQueue& queue, FillShortLds<W>& lds, int32_t* __restrict__ tcblockRowid, uint8_t* __restrict__ tcblocktileId,
    int32_t* __restrict__ tcblockOffset, int32_t* __restrict__ sparseAToXidx,
    unsigned long long* __restrict__ bitmap) {
  constexpr int WPT = 16 * W / 64;
  constexpr int LOGW = (W == 16) ? 4 : 3;
  constexpr int MAXB = FillShortLds<W>::MAXB;
  constexpr int U = 4;  // groups of 64 edges in flight together
  static_assert(MAXB * 8 <= MAXB * W, "edges per (block, row), two counters per word, fit ids");
  const int lane = threadIdx.x & 63;
  int rowStart = rowPtr[min(w * 16 + min(lane, 16), N)];
  const int eS = __builtin_amdgcn_readlane(rowStart, 0);
  const int n = __builtin_amdgcn_readlane(rowStart, 16) - eS;
  rowStart -= eS;
  if (n > kBinsMax && queue.counts && lane == 0) queue.add(w, n);
  if (n == 0 || n > kBinsMax || nb > MAXB) return;  // long ones: fill_one_window
  if (nb < 1) return;  // no block to write: every column of the window lay outside [0, N)
  unsigned long long* bm = lds.bm;
  uint32_t* ids = lds.ids;
  RowMarks<kBinsMax> marks;
  marks.init(lds.mark, rowStart, lane);
  for (int i = lane; i < nb * WPT / 2; i += 64)
    reinterpret_cast<uint4*>(bm)[i] = make_uint4(0, 0, 0, 0);
  for (int i = nb * W - W + lane; i < nb * W; i += 64) ids[i] = 0u;  // unused slots hold 0
  wave_lds_sync();
  bool rough = false;  // some row's columns do not strictly ascend: nor do its (row, rank) pairs
  int before = -1;
  for (int e0 = 0; e0 < n; e0 += 64 * U) {
    int rank[U], col[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int i = min(e0 + 64 * u + lane, n - 1);
      rank[u] = edgeToColumn[eS + i];
      col[u] = colIdx[eS + i];
    }
#pragma unroll
    for (int u = 0; u < U; u++)  // all of them in flight before the first one is used
      asm volatile("" : "+v"(rank[u]), "+v"(col[u]));
#pragma unroll
    for (int u = 0; u < U; u++) {
      if (e0 + 64 * u >= n) break;
      const int row = marks.next_group((e0 >> 6) + u);
      const int pair = (row << 16) | rank[u];
      const int left = __builtin_amdgcn_update_dpp(before, pair, 0x138, 0xf, 0xf, false);
      before = __builtin_amdgcn_readlane(pair, 63);
      if (e0 + 64 * u + lane < n && (unsigned)rank[u] < (unsigned)(nb * W)) {
        rough = rough || left >= pair;
        ids[rank[u]] = (uint32_t)col[u];
        // Byte 7 - row % 8 of word 2 (rank >> 3) + (row >> 3) is the row, MSB first (see window_rank_fill_kernel):
        // in dwords, the halves of a word change places.
        atomicOr(&reinterpret_cast<unsigned*>(bm)[((rank[u] & ~7) >> 1) + ((row >> 2) ^ 1)],
                 0x80000000u >> ((((unsigned)row << 3) | ((unsigned)rank[u] & 7u)) & 31u));
      }
    }
  }
  wave_lds_sync();
  for (int i = lane; i < nb * WPT / 2; i += 64)
    store_streaming(reinterpret_cast<uint4*>(bitmap + (int64_t)base * WPT) + i,
                    reinterpret_cast<const uint4*>(bm)[i]);
  for (int i = lane; i < nb * W / 4; i += 64)
    store_streaming(reinterpret_cast<uint4*>(sparseAToXidx + (int64_t)base * W) + i,
                    reinterpret_cast<const uint4*>(ids)[i]);
  if (__ballot(rough) == 0ull) {
    static_assert(kBinsMax + 8 <= sizeof(lds.ids), "tile ids where the ids were");
    uint8_t* stage = reinterpret_cast<uint8_t*>(ids);
    wave_lds_sync();  // the ids are out
    const unsigned skew = (unsigned)((uintptr_t)(tcblocktileId + eS) & 3u);
    unsigned carry = 0;
    for (int k = 0; k < 2 * nb; k += 64) {
      const int t = (k + lane) >> 1, half = lane & 1;
      unsigned long long left = 0, right = 0;
      if (t < nb) {
        left = bm[t * WPT + half];
        if constexpr (W == 16) right = bm[t * WPT + 2 + half];
      }
      const unsigned nnz = __popcll(left) + __popcll(right);
      const unsigned incl = wave_inclusive_scan(nnz, lane);
      const unsigned at = carry + incl - nnz;
      carry += (unsigned)__builtin_amdgcn_readlane((int)incl, 63);
      if (t < nb && half == 0) {
        tcblockOffset[base + t] = eS + (int)at;
        tcblockRowid[base + t] = w;
      }
      walk_half_block<W>(left, right, half, stage, at + skew);
    }
    wave_lds_sync();
    uint8_t* dst = tcblocktileId + eS - skew;  // the dword that holds the window's first tile id
    const int end = n + (int)skew;
    for (int i = 4 * lane; i < end; i += 256) {
      if (i >= (int)skew && i + 4 <= end) {
        *reinterpret_cast<uint32_t*>(dst + i) = *reinterpret_cast<const uint32_t*>(stage + i);
      } else {
        for (int j = 0; j < 4; j++)
          if (i + j >= (int)skew && i + j < end) dst[i + j] = stage[i + j];
      }
    }
    return;
  }
  // Repeated or descending columns: tile ids sit in edge order inside a block. The edges of every
  // (block, row) are counted (two 16-bit counters per word, where the ids were), the counts turned
  // into places and the rows replayed in order (src/utils.cu:173-224).
  uint32_t* cnt = ids;
  wave_lds_sync();
  EdgeRows<kBinsMax> edgeRows;
  edgeRows.init(lds.mark, rowStart, lane);
  for (int i = lane; i < nb * 8; i += 64) cnt[i] = 0u;
  wave_lds_sync();
  for (int e0 = 0; e0 < n; e0 += 64) {
    bool starts;
    const int row = edgeRows.next_group(e0, lane, &starts);
    const int rank = e0 + lane < n ? edgeToColumn[eS + e0 + lane] : -1;
    if ((unsigned)rank < (unsigned)(nb * W)) {
      const int c = (rank >> LOGW) * 16 + row;
      atomicAdd(&cnt[c >> 1], 1u << ((c & 1) * 16));
    }
  }
  wave_lds_sync();
  unsigned carry = 0;
  for (int k = 0; k < nb; k += 64) {
    const int t = k + lane;
    unsigned nnz = 0;
    for (int q = 0; q < 8; q++) {
      const uint32_t v = t < nb ? cnt[t * 8 + q] : 0u;
      nnz += (v & 0xFFFFu) + (v >> 16);
    }
    const unsigned incl = wave_inclusive_scan(nnz, lane);
    unsigned run = carry + incl - nnz;
    carry += (unsigned)__builtin_amdgcn_readlane((int)incl, 63);
    if (t < nb) {
      tcblockOffset[base + t] = eS + (int)run;
      tcblockRowid[base + t] = w;
      for (int q = 0; q < 8; q++) {
        const uint32_t v = cnt[t * 8 + q], lo = run + (v & 0xFFFFu);
        cnt[t * 8 + q] = run | (lo << 16);
        run = lo + (v >> 16);
      }
    }
  }
  wave_lds_sync();
  const unsigned long long ltMask = (1ull << lane) - 1ull;
  for (int row = 0; row < 16; row++) {
    const int rs = __builtin_amdgcn_readlane(rowStart, row);
    const int re = __builtin_amdgcn_readlane(rowStart, row + 1);
    for (int e0 = rs; e0 < re; e0 += 64) {
      const int rank = e0 + lane < re ? edgeToColumn[eS + e0 + lane] : -1;
      const bool valid = (unsigned)rank < (unsigned)(nb * W);
      const int t = rank >> LOGW;
      unsigned long long peers = __ballot(valid);  // lanes whose edges fall into the same block
      for (int bit = 0; (MAXB >> bit) != 0; bit++) {
        const unsigned long long bal = __ballot((t >> bit) & 1);
        peers &= ((t >> bit) & 1) ? bal : ~bal;
      }
      const int c = t * 16 + row, sh = (c & 1) * 16;
      if (valid)
        tcblocktileId[eS + ((cnt[c >> 1] >> sh) & 0xFFFFu) + __popcll(peers & ltMask)] =
            (uint8_t)(row * W + (rank & (W - 1)));
      wave_lds_sync();
      // the row's blocks have a word each: the last lane of a block moves its counter
      if (valid && (peers >> lane) == 1ull)
        atomicAdd(&cnt[c >> 1], (uint32_t)__popcll(peers) << sh);
      wave_lds_sync();
    }
  }
}

template <int W>
__global__ __launch_bounds__(64) void window_fill_short_kernel(
    const int32_t* __restrict__ rowPtr, const int32_t* __restrict__ colIdx, int N, int E, int nRW,
    const int32_t* __restrict__ edgeToColumn, const int32_t* __restrict__ rowWindowOffset,
    LongQueue queue, int32_t* __restrict__ tcblockRowid, uint8_t* __restrict__ tcblocktileId,
    int32_t* __restrict__ tcblockOffset, int32_t* __restrict__ sparseAToXidx,
    unsigned long long* __restrict__ bitmap) {
  __shared__ FillShortLds<W> lds;
  // the last windows first: what the ranking wrote last is still in the memory-side cache (61M edges: 204 -> 198 us)
  const int w = nRW - 1 - (int)blockIdx.x;
  const int base = __builtin_amdgcn_readfirstlane(rowWindowOffset[w]);
  const int nb = __builtin_amdgcn_readfirstlane(rowWindowOffset[w + 1]) - base;
  if (w == nRW - 1 && threadIdx.x == 0) tcblockOffset[base + nb] = E;
  fill_short_window<W>(w, base, nb, rowPtr, colIdx, N, edgeToColumn, queue, lds, tcblockRowid,
                       tcblocktileId, tcblockOffset, sparseAToXidx, bitmap);
}

template <int W, int TB, int TC, int TCG>
__global__ __launch_bounds__(TB) void window_fill_kernel(
    const int32_t* __restrict__ rowPtr, const int32_t* __restrict__ colIdx, int N, int E,
    const int32_t* __restrict__ edgeToColumn, const int32_t* __restrict__ rowWindowOffset,
    int32_t* __restrict__ tcblockRowid,
    uint8_t* __restrict__ tcblocktileId, int32_t* __restrict__ tcblockOffset,
    int32_t* __restrict__ sparseAToXidx, unsigned long long* __restrict__ bitmap) {
  extern __shared__ __align__(16) unsigned char sRawDyn[];
  const int w = blockIdx.x;
  if (w == 0 && threadIdx.x == 0) tcblockOffset[rowWindowOffset[gridDim.x]] = E;
  const int base = rowWindowOffset[w];
  fill_one_window<W, TB, TC, TCG>(w, base, rowWindowOffset[w + 1] - base, rowPtr, colIdx, N, E,
                                  edgeToColumn, sRawDyn, tcblockRowid, tcblocktileId, tcblockOffset,
                                  sparseAToXidx, bitmap);
}

// The windows that window_fill_short_kernel leaves out: those of its queue (the large ones if LARGE, else
// the mid ones), or, where the caller has no memory for one, those of more than minEdges and at most
// maxEdges edges (find_windows). Two sizes: 256 threads and 320 TC blocks of LDS at a time for windows of
// up to kFillMid edges (five workgroups per CU), 1024 threads and 1280 blocks for longer ones, which would
// otherwise each keep one small workgroup busy long after the others are done (31 700 edges:
// 190 us).
// LARGE: the first orderGroups workgroups order the windows instead, TB of them each: the launch holds a
// handful of windows, so most of the CUs would be idle, and nothing else of the call waits for the
// order.
template <int W, int TB, int TC, bool LARGE>
__global__ __launch_bounds__(TB) void window_fill_long_kernel(
    const int32_t* __restrict__ rowPtr, const int32_t* __restrict__ colIdx, int N, int E, int nRW,
    const int32_t* __restrict__ edgeToColumn, const int32_t* __restrict__ rowWindowOffset,
    LongQueue queue, int minEdges, int maxEdges, int orderGroups,
    const int32_t* __restrict__ blockPartition, const uint16_t* __restrict__ orderRows,
    int32_t* __restrict__ sortedRowWindows, int32_t* __restrict__ tcblockRowid,
    uint8_t* __restrict__ tcblocktileId, int32_t* __restrict__ tcblockOffset,
    int32_t* __restrict__ sparseAToXidx, unsigned long long* __restrict__ bitmap) {
  extern __shared__ __align__(16) unsigned char sRawDyn[];
  __shared__ int sList[TB];
  __shared__ int sListLen;
  if constexpr (LARGE) {
    if ((int)blockIdx.x < orderGroups) {
      static_assert(TB == kOrderRowWindows, "a row of the histogram per workgroup");
      order_chunk<TB, true>([=](int i) { return blockPartition[i]; }, nRW, (int)blockIdx.x * TB,
                            kOrderRowBins, sortedRowWindows, reinterpret_cast<uint32_t*>(sRawDyn),
                            orderRows);
      return;
    }
  }
  const int group = (int)blockIdx.x - (LARGE ? orderGroups : 0);
  const int groups = (int)gridDim.x - (LARGE ? orderGroups : 0);
  const auto fill = [&](int w) {
    __syncthreads();  // the window before this one has left the LDS arrays
    const int base = rowWindowOffset[w];
    fill_one_window<W, TB, TC, TC>(w, base, rowWindowOffset[w + 1] - base, rowPtr, colIdx, N, E,
                                   edgeToColumn, sRawDyn, tcblockRowid, tcblocktileId, tcblockOffset,
                                   sparseAToXidx, bitmap);
  };
  if (queue.counts) {
    const int listed = queue.size(LARGE);
    for (int k = group; k < listed; k += groups) fill(queue.at(LARGE, k));
    return;
  }
  for (int64_t first = 0; first < nRW; first += (int64_t)TB * groups) {
    const int found = find_windows(rowPtr, N, nRW, first + group - (int)blockIdx.x, groups, minEdges,
                                   maxEdges, sList, &sListLen);
    for (int k = 0; k < found; k++) fill(sList[k]);
  }
}

// Sum of counts[0 .. n) by the whole workgroup; every thread calls this and gets the sum.
template <int TB>
__device__ __forceinline__ int sum_counts(const int32_t* __restrict__ counts, int n) {
  __shared__ unsigned sSum[TB / 64];
  unsigned sum = 0;
  for (int i = threadIdx.x; i < n; i += TB) sum += (unsigned)counts[i];
  sum = wave_inclusive_scan(sum, threadIdx.x & 63);
  __syncthreads();  // the reads of the call before this one are done
  if ((threadIdx.x & 63) == 63) sSum[threadIdx.x >> 6] = sum;
  __syncthreads();
  unsigned total = 0;
#pragma unroll
  for (int k = 0; k < TB / 64; k++) total += sSum[k];
  return (int)total;
}

// Phase 2 of a graph of up to kFinSingleMax windows, most of them short, in one launch like
// window_rank_all_kernel: workgroups that look for the long windows, then some that make the window
// order (unless orderGroups is 0), which nothing else of the call waits for, then those of the short
// windows. 169k-node R-MAT graph: 17 + 25 us as two launches, 29 us together. Eight waves: preprocessing
// calls on 34 R-MAT, power-law and even graphs take up to 23 % longer with four and 28 % with sixteen.
// As many blocks of a long window at a time as let three workgroups share a CU (53 760 bytes of LDS each),
// which the short windows' LDS does too since a window's tile ids are staged where its ids were (two
// workgroups and 576 blocks before: power-law, 50k nodes, 1300 edges a window: 107 -> 98 us, 250k nodes, 700:
// 195 -> 173; R-MAT, 250k nodes, 200: 115 -> 109; power-law, 130k nodes, 100, whose longest windows fall
// between 528 and 576 blocks: 74 -> 78).
// SELF: no scan was launched before; every workgroup adds up the counts in front of its windows itself
// and the short ones' write rowWindowOffset and the total. That is one launch (4 us) less where the sums
// are short, a few counts per thread: up to kSelfScanMax windows.
constexpr int kFillAllThreads = 512;
template <int W>
constexpr int kFillAllChunk = W == 16 ? 528 : 640;
constexpr int kSelfScanMax = 2048;
template <int W, bool SELF>
__global__ __launch_bounds__(kFillAllThreads) void window_fill_all_kernel(
    const int32_t* __restrict__ rowPtr, const int32_t* __restrict__ colIdx, int N, int E, int nRW,
    const int32_t* __restrict__ edgeToColumn, const int32_t* __restrict__ blockPartition,
    int longGroups, int orderGroups, int nBins, int32_t* __restrict__ rowWindowOffset,
    int32_t* __restrict__ sortedRowWindows, long long* __restrict__ nTcb,
    int32_t* __restrict__ tcblockRowid, uint8_t* __restrict__ tcblocktileId,
    int32_t* __restrict__ tcblockOffset, int32_t* __restrict__ sparseAToXidx,
    unsigned long long* __restrict__ bitmap) {
  extern __shared__ __align__(16) unsigned char sRawDyn[];
  constexpr int TB = kFillAllThreads, NW = TB / 64;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int group = (int)blockIdx.x - longGroups - orderGroups;
  if (group >= 0) {
    const int w = group * NW + wave;
    int base, nb;
    if constexpr (SELF) {
      base = sum_counts<TB>(blockPartition, group * NW);
      if (w >= nRW) return;
      const unsigned c = lane <= wave ? (unsigned)blockPartition[group * NW + lane] : 0u;
      nb = __builtin_amdgcn_readlane((int)c, wave);
      base += __builtin_amdgcn_readlane((int)wave_inclusive_scan(c, lane), 63) - nb;
      if (lane == 0) {
        if (w == 0) rowWindowOffset[0] = 0;
        rowWindowOffset[w + 1] = base + nb;
        if (w == nRW - 1) *nTcb = base + nb;
      }
    } else {
      if (w >= nRW) return;
      base = __builtin_amdgcn_readfirstlane(rowWindowOffset[w]);
      nb = __builtin_amdgcn_readfirstlane(rowWindowOffset[w + 1]) - base;
    }
    if (w == nRW - 1 && lane == 0) tcblockOffset[base + nb] = E;
    fill_short_window<W>(w, base, nb, rowPtr, colIdx, N, edgeToColumn,
                         LongQueue{nullptr, nullptr, 0, 0},
                         reinterpret_cast<FillShortLds<W>*>(sRawDyn)[wave], tcblockRowid,
                         tcblocktileId, tcblockOffset, sparseAToXidx, bitmap);
    return;
  }
  if ((int)blockIdx.x >= longGroups) {
    order_chunk<TB>([=](int i) { return blockPartition[i]; }, nRW,
                    ((int)blockIdx.x - longGroups) * TB, nBins, sortedRowWindows,
                    reinterpret_cast<uint32_t*>(sRawDyn));
    return;
  }
  __shared__ int sList[TB];
  __shared__ int sListLen;
  for (int64_t first = 0; first < nRW; first += (int64_t)TB * longGroups) {
    const int found = find_windows(rowPtr, N, nRW, first, longGroups, kBinsMax, 0x7FFFFFFF, sList,
                                   &sListLen);
    for (int k = 0; k < found; k++) {
      __syncthreads();  // the window before this one has left the LDS arrays
      const int w = sList[k];
      int base, nb;
      if constexpr (SELF) {
        base = sum_counts<TB>(blockPartition, w);
        nb = blockPartition[w];
      } else {
        base = rowWindowOffset[w];
        nb = rowWindowOffset[w + 1] - base;
      }
      fill_one_window<W, TB, kFillAllChunk<W>, kFillAllChunk<W>>(
          w, base, nb, rowPtr, colIdx, N, E, edgeToColumn, sRawDyn, tcblockRowid, tcblocktileId,
          tcblockOffset, sparseAToXidx, bitmap);
    }
  }
}
template <int W>
constexpr size_t fill_all_lds(int nBins) {
  size_t lds = (kFillAllThreads / 64) * sizeof(FillShortLds<W>);
  if (lds < fill_lds_bytes<W>(kFillAllChunk<W>, kFillAllChunk<W>))
    lds = fill_lds_bytes<W>(kFillAllChunk<W>, kFillAllChunk<W>);
  return lds > nBins * sizeof(uint32_t) ? lds : nBins * sizeof(uint32_t);
}

// ------------------------------------------------------------------ both phases, one call
// Graphs of long windows whose column range fits one bitset (N <= kRangeMax) when the caller has
// sized the block arrays by an upper bound instead of waiting for the count: the window's bitset
// is built twice (window_count_kernel for the block counts, window_rank_fill_kernel after the
// scan) and everything else happens while it sits in LDS, so edgeToColumn is written once and
// never read back and the column ids are read from memory once (the second and third reads of a
// window's 30 KB come from the L2).
//
// Neither kernel is bound by memory alone: on a 115 M-edge graph of 233 k nodes the second one takes
// 577 us for 2.2 GB that it cannot do without, and the vector ALUs are busy half of that. So both are
// written for few instructions per edge: a window's edges are split into whole groups of four
// consecutive edges from a 4-aligned index (no per-edge range checks, 16-byte loads and stores) and at
// most six edges at the window's two ends, which single threads handle one by one, as they do the
// (at most fifteen) groups in which a row starts. On that graph: such groups out of the main loop, ids
// collected in LDS instead of enumerated from the bitset, 16-bit prefixes (which make the room for
// them) and the first loads in front of the clearing 738 -> 610 us; outputs past the caches, which
// leaves the column ids there for their second and third reading, 610 -> 577 us and the count kernel
// 129 -> 88 us.

// Workgroup barrier that orders LDS traffic only: unlike __syncthreads() it does not wait for the
// wave's outstanding global loads and stores, which then overlap the next phase. For phases that
// talk to each other through LDS and never through global memory.
__device__ __forceinline__ void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// The window's edges [eS, eE) as whole 4-aligned groups [gA, gB) plus the edges in front of and
// behind them (at most three each).
struct EdgeSplit {
  int gA, gB;      // whole groups: e0 = gA, gA + 4, ... < gB
  int headEnd;     // loose edges [eS, headEnd) and [tailBegin, eE)
  int tailBegin;
};
__device__ __forceinline__ EdgeSplit split_edges(int eS, int eE) {
  EdgeSplit sp;
  const int up = (eS + 3) & ~3, down = eE & ~3;
  sp.headEnd = min(up, eE);
  sp.tailBegin = max(down, sp.headEnd);
  sp.gA = up;
  sp.gB = max(down, up);
  return sp;
}
// the i-th loose edge (i = 0..5), or -1
__device__ __forceinline__ int loose_edge(const EdgeSplit& sp, int eS, int eE, int i) {
  const int nHead = sp.headEnd - eS;
  const int e = i < nHead ? eS + i : sp.tailBegin + (i - nHead);
  return (i < 6 && e < eE) ? e : -1;
}

// The groups of a thread's step, from e0 on: U of them, TB apart. A group past the end repeats the first
// one (its bits are set already).
template <int TB, int U>
__device__ __forceinline__ void load_groups(const int32_t* __restrict__ colIdx, const EdgeSplit& sp,
                                            int e0, int4 (&c)[U]) {
#pragma unroll
  for (int g = 0; g < U; g++) {
    const int e = e0 + 4 * g * TB < sp.gB ? e0 + 4 * g * TB : e0;
    c[g] = *reinterpret_cast<const int4*>(colIdx + e);
  }
}

// Sets the bits of the window's column ids in `bits` (32-bit words). c: the thread's first step, which
// the caller has requested before it cleared the bits. Returns false (for the calling thread) when it
// met a column outside [0, N); such a column sets the bit of N - 1.
template <int TB, int U>
__device__ __forceinline__ bool set_column_bits(const int32_t* __restrict__ colIdx, int eS, int eE,
                                                const EdgeSplit& sp, unsigned N, uint32_t* bits,
                                                int4 (&c)[U]) {
  const int tid = threadIdx.x;
  unsigned most = 0;
  const auto set = [&](unsigned col) {
    most = max(most, col);
    col = min(col, N - 1u);
    atomicOr(&bits[col >> 5], 1u << (col & 31));
  };
  for (int e0 = sp.gA + 4 * tid; e0 < sp.gB;) {
#pragma unroll
    for (int g = 0; g < U; g++) {
      set((unsigned)c[g].x);
      set((unsigned)c[g].y);
      set((unsigned)c[g].z);
      set((unsigned)c[g].w);
    }
    e0 += 4 * U * TB;
    if (e0 < sp.gB) load_groups<TB, U>(colIdx, sp, e0, c);
  }
  const int e = loose_edge(sp, eS, eE, tid);
  if (e >= 0) set((unsigned)colIdx[e]);
  return most < N;
}

template <int W, int TB>
__global__ __launch_bounds__(TB) void window_count_kernel(
    const int32_t* __restrict__ rowPtr, const int32_t* __restrict__ colIdx, int N, int range,
    int32_t* __restrict__ blockPartition, WsHeader* __restrict__ hdr, int* __restrict__ error) {
  extern __shared__ __align__(16) uint32_t smem[];
  uint32_t* bits = smem;  // range/32 words
  __shared__ unsigned sWaveTot[TB / 64];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int w = blockIdx.x;
  const int eS = rowPtr[min(w * 16, N)], eE = rowPtr[min(w * 16 + 16, N)];
  if (eE <= eS) {
    if (tid == 0) blockPartition[w] = 0;
    return;
  }
  const EdgeSplit sp = split_edges(eS, eE);
  int4 c[4];
  if (sp.gA + 4 * tid < sp.gB) load_groups<TB, 4>(colIdx, sp, sp.gA + 4 * tid, c);
  const int nGroups = range >> 7;
  for (int i = tid; i < nGroups; i += TB)
    reinterpret_cast<uint4*>(bits)[i] = make_uint4(0, 0, 0, 0);
  lds_barrier();
  if (!set_column_bits<TB, 4>(colIdx, eS, eE, sp, (unsigned)N, bits, c)) {
    hdr->error = 1;  // window_rank_fill_kernel asks here, the host over there
    *error = 1;
  }
  lds_barrier();
  unsigned cnt = 0;
  for (int gi = tid; gi < nGroups; gi += TB) {
    const uint4 v = reinterpret_cast<const uint4*>(bits)[gi];
    cnt += __popc(v.x) + __popc(v.y) + __popc(v.z) + __popc(v.w);
  }
  const unsigned incl = wave_inclusive_scan(cnt, lane);
  if (lane == 63) sWaveTot[wave] = incl;
  lds_barrier();
  if (tid == 0) {
    unsigned total = 0;
#pragma unroll
    for (int v = 0; v < TB / 64; v++) total += sWaveTot[v];
    blockPartition[w] = (int)((total + W - 1) / W);
  }
}

constexpr int kRankFillThreads = 768;
// 64-bit bitset words per thread of window_rank_fill_kernel at the largest column range
constexpr int kRankFillPerMax = (kRangeMax / 64 + kRankFillThreads - 1) / kRankFillThreads;
// bytes of bitset and prefixes (16 bits per 64-bit word), a multiple of 16
constexpr int rank_fill_bitset_bytes(int range) { return (range / 64 * 10 + 15) & ~15; }

// Dynamic LDS: bitset (range/64 64-bit words) | set bits before each word (range/64 16-bit words)
// | chunkBytes: the window's TC-block bitmaps, then the low halves of its column ids, in rank order; a
// window with more blocks than both have room for there (or whose prefixes need more than 16 bits, see
// `big`) takes its blocks in chunks of bitmaps and enumerates its ids from the bitset. A window with a
// repeated or descending column is handed to fill_window_generic once its edgeToColumn entries are
// written, with the whole of the dynamic LDS as that routine's arrays.
// Registers: 60 vector ones of the 80 that two workgroups per CU leave; of the scalar ones (pointers, lane
// masks) about 40 go to lanes of vector registers, none to memory.
template <int W, int TB>
__global__ __launch_bounds__(TB) __attribute__((amdgpu_waves_per_eu(6, 6)))
void window_rank_fill_kernel(
    const int32_t* __restrict__ rowPtr, const int32_t* __restrict__ colIdx, int N, int E,
    int range, int chunkBytes, const int32_t* __restrict__ rowWindowOffset,
    const int32_t* __restrict__ order, const WsHeader* __restrict__ hdr, int32_t* edgeToColumn,
    int32_t* __restrict__ edgeToRow,
    int32_t* __restrict__ tcblockRowid, uint8_t* __restrict__ tcblocktileId,
    int32_t* __restrict__ tcblockOffset, int32_t* __restrict__ sparseAToXidx,
    unsigned long long* __restrict__ bitmap) {
  constexpr int WPT = 16 * W / 64;  // bitmap words per TC block
  constexpr int LOGW = (W == 16) ? 4 : 3;
  constexpr int NWAVE = TB / 64;
  constexpr int PER = kRankFillPerMax;
  constexpr int HIGH = (kRangeMax + 65535) >> 16;  // values of a column id's upper half
  static_assert(TB == kRankFillThreads, "PER is computed for this workgroup size");
  extern __shared__ __align__(16) uint32_t smem[];
  const int nW64 = range >> 6;  // even: range is a multiple of 128
  unsigned long long* bits64 = reinterpret_cast<unsigned long long*>(smem);
  uint32_t* bits = smem;
  uint16_t* pref = reinterpret_cast<uint16_t*>(smem + 2 * nW64);
  const int bitsetBytes = rank_fill_bitset_bytes(range);
  unsigned long long* sBm = reinterpret_cast<unsigned long long*>(smem + bitsetBytes / 4);
  __shared__ int sRow[17];
  __shared__ unsigned sWaveTot[NWAVE];
  __shared__ unsigned sTot[PER * NWAVE];     // set bits per (round, wave)
  __shared__ unsigned sBefore[PER * NWAVE];  // and in front of it
  __shared__ unsigned sHigh[HIGH];        // distinct columns below 65536 h
  __shared__ unsigned sUnsorted;          // bit r: row r's columns are not strictly ascending

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = uniform(tid >> 6);
  // windows start in the heavy-first order that the scan kernel has just written: the longest
  // ones first, so that none of them is still running alone when the others are done
  const int w = order[blockIdx.x];
  if (hdr->error) return;  // a column index outside [0, N): the caller gets the error, no output
  if (w == 0 && tid == 0) tcblockOffset[rowWindowOffset[gridDim.x]] = E;
  const int base = rowWindowOffset[w];
  const int nb = rowWindowOffset[w + 1] - base;
  const int r0 = w * 16;
  const int eS = rowPtr[min(r0, N)], eE = rowPtr[min(r0 + 16, N)];
  if (eE <= eS) return;
  const EdgeSplit sp = split_edges(eS, eE);
  constexpr int U = 2;  // groups of a thread in flight together
  {
    // ---- the window's distinct columns as a bitset (validated by window_count_kernel)
    int4 c[U];
    if (sp.gA + 4 * tid < sp.gB) load_groups<TB, U>(colIdx, sp, sp.gA + 4 * tid, c);
    if (tid < 17) sRow[tid] = rowPtr[min(r0 + tid, N)];
    if (tid < HIGH) sHigh[tid] = 0xFFFFFFFFu;
    if (tid == 0) sUnsorted = 0u;
    for (int i = tid; i < (nW64 >> 1); i += TB)
      reinterpret_cast<uint4*>(bits)[i] = make_uint4(0, 0, 0, 0);
    lds_barrier();
    set_column_bits<TB, U>(colIdx, eS, eE, sp, (unsigned)N, bits, c);
  }
  lds_barrier();

  // ---- set bits before every 64-bit word. Thread t owns the words t, t + TB, ... (neighbouring lanes,
  // neighbouring words): a wave-level scan per round, then every wave scans the (round, wave) totals.
  const int per = (nW64 + TB - 1) / TB;  // <= PER
  unsigned before[PER];  // within the wave's 64 words
#pragma unroll
  for (int k = 0; k < PER; k++) {
    if (k < per) {
      const int i = k * TB + tid;
      const unsigned cnt = i < nW64 ? (unsigned)__popcll(bits64[i]) : 0u;
      const unsigned incl = wave_inclusive_scan(cnt, lane);
      before[k] = incl - cnt;
      if (lane == 63) sTot[k * NWAVE + wave] = incl;
    }
  }
  lds_barrier();
  unsigned pairIncl, pairBoth, pairFirst;  // lane l: pair l of the totals
  {
    static_assert(PER * NWAVE <= 128, "two totals per lane");
    const int n = per * NWAVE;
    pairFirst = (2 * lane < n) ? sTot[2 * lane] : 0u;
    const unsigned second = (2 * lane + 1 < n) ? sTot[2 * lane + 1] : 0u;
    pairBoth = pairFirst + second;
    pairIncl = wave_inclusive_scan(pairBoth, lane);
    if (wave == 0 && 2 * lane < n) sBefore[2 * lane] = pairIncl - pairBoth;
    if (wave == 0 && 2 * lane + 1 < n) sBefore[2 * lane + 1] = pairIncl - second;
  }
  const unsigned nCols = (unsigned)__builtin_amdgcn_readlane((int)pairIncl, 63);
  // more distinct columns than a 16-bit prefix can name: the prefixes stay relative to their wave's 64
  // words and sBefore is added on every use
  const bool big = nCols > 0xFFFFu;
  const bool idsInLds = nb * (WPT * 8 + W * 2) <= chunkBytes && !big;
#pragma unroll
  for (int k = 0; k < PER; k++) {
    if (k < per) {
      const int i = k * TB + tid;
      const int at = k * NWAVE + wave;
      unsigned front = (unsigned)__builtin_amdgcn_readlane((int)(pairIncl - pairBoth), at >> 1);
      if (at & 1) front += (unsigned)__builtin_amdgcn_readlane((int)pairFirst, at >> 1);
      const unsigned pos = front + before[k];
      if (i < nW64) pref[i] = (uint16_t)(big ? before[k] : pos);
      if (idsInLds) {
        if ((i & 1023) == 0 && i < nW64) sHigh[i >> 10] = pos;
      } else if (i < nW64) {
        // the compacted column ids, which are the set bits in ascending order, 32 bits at a time, with a
        // 32-bit byte offset from the window's first id slot
        char* idBytes = reinterpret_cast<char*>(sparseAToXidx + (int64_t)base * W);
        const unsigned long long x = bits64[i];
        unsigned off = pos * 4u;
#pragma unroll
        for (int h = 0; h < 2; h++) {
          unsigned half = h ? (unsigned)(x >> 32) : (unsigned)x;
          const int idBase = i * 64 + 32 * h;
          while (half) {
            *reinterpret_cast<int32_t*>(idBytes + off) = idBase + __builtin_ctz(half);
            off += 4u;
            half &= half - 1u;
          }
        }
      }
    }
  }
  if (!idsInLds)  // the slots that the last block leaves unused hold 0
    for (int i = (int)nCols + tid; i < nb * W; i += TB) sparseAToXidx[(int64_t)base * W + i] = 0;

  // ---- ranks, rows and bitmaps. The first chunk of TC blocks also writes edgeToColumn / edgeToRow;
  // a window of several chunks ranks its edges again per chunk (the bitset stays in LDS).
  const auto rank_of = [&](int col) -> int {
    const unsigned wd = (unsigned)col >> 6;
    const unsigned long long upTo = bits64[wd] << (~col & 63);  // the column's own bit on top
    unsigned rank = pref[wd] + (unsigned)__popcll(upTo) - 1u;
    if (big) rank += sBefore[wd >> 6];
    return (int)rank;
  };
  unsigned* sBmWords = reinterpret_cast<unsigned*>(sBm);
  // the window's edges against the blocks [tc0, tc0 + nt): bitmap bits, with `ids` the ids' low halves
  // as well, and edgeToColumn / edgeToRow where tc0 = 0. ids: one chunk holds all blocks.
  const auto rank_edges = [&](auto ids, int tc0, int nt) {
    constexpr bool IDS = decltype(ids)::value;
    const bool first = IDS || tc0 == 0;
    uint16_t* sId = reinterpret_cast<uint16_t*>(sBm + nt * WPT);
    // one edge: rank, row, bit (the window's loose ends and the groups that straddle rows)
    const auto one_edge = [&](int e, int col, int r) {
      const int ec = rank_of(col);
      if (first) {
        edgeToColumn[e] = ec;
        edgeToRow[e] = r0 + r;
        if (e > sRow[r] && colIdx[e - 1] >= col) atomicOr(&sUnsorted, 1u << r);
      }
      const int t = (ec >> LOGW) - tc0;
      if (IDS || (unsigned)t < (unsigned)nt) {
        const int cl = ec & (W - 1);
        const int sub = (cl >> 3) * (W / 8) + (r >> 3);
        const int key = (t * WPT + sub) * 8 + 7 - (r & 7);
        atomicOr(&sBmWords[key >> 2], (0x80u >> (cl & 7)) << (8 * (key & 3)));
        if constexpr (IDS) sId[ec] = (uint16_t)col;
      }
    };
    // a whole group of four edges of one row; left: the column in front of it
    const auto group = [&](int e0, const int4& c4, int left) {
      const int cols[4] = {c4.x, c4.y, c4.z, c4.w};
      const int r = row_of_edge(sRow, e0);
      if (e0 + 3 >= sRow[r + 1]) return;  // it straddles rows: edge by edge below
      int ecs[4];
#pragma unroll
      for (int u = 0; u < 4; u++) ecs[u] = rank_of(cols[u]);
      if (first) {
#ifndef F3S_PROBE_PRE_NO_EDGE_STORES
        store_streaming(reinterpret_cast<uint4*>(edgeToColumn + e0),
                        make_uint4(ecs[0], ecs[1], ecs[2], ecs[3]));
        store_streaming(reinterpret_cast<uint4*>(edgeToRow + e0),
                        make_uint4(r0 + r, r0 + r, r0 + r, r0 + r));
#endif
        const bool bad = (e0 > sRow[r] && left >= cols[0]) || cols[0] >= cols[1] ||
                         cols[1] >= cols[2] || cols[2] >= cols[3];
        if (bad) atomicOr(&sUnsorted, 1u << r);
      }
      if constexpr (IDS) {
#pragma unroll
        for (int u = 0; u < 4; u++) sId[ecs[u]] = (uint16_t)cols[u];
      }
      // Bits of one row. A TC block's bitmap is WPT 64-bit words, one per 8x8 sub-block (column
      // halves first); byte 7 - r%8 of a word is row r%8, MSB first. With rank = 16 t + cl (or
      // 8 t + cl) the 64-bit word of (t, cl, r) is 2 (rank >> 3) + (r >> 3) for both widths, and
      // the bit inside the row's byte is 0x80 >> (rank & 7). Consecutive edges of a row fall into
      // the same byte up to eight at a time: OR the bits of equal bytes together, then one
      // 32-bit LDS atomic per byte.
      const int byte = 7 - (r & 7);
      const int wordBias = (r >> 3) * 2 + (byte >> 2) - tc0 * (WPT * 2);  // in 32-bit words
      const unsigned rowBit = 0x80u << (8 * (byte & 3));
      int word[4];
      unsigned m[4];
#pragma unroll
      for (int u = 0; u < 4; u++) {
        word[u] = (ecs[u] >> 3) * 4 + wordBias;
        m[u] = rowBit >> (ecs[u] & 7);
        if (!IDS && (unsigned)((ecs[u] >> LOGW) - tc0) >= (unsigned)nt) m[u] = 0u;
      }
#pragma unroll
      for (int u = 1; u < 4; u++) {
        if (word[u] == word[u - 1]) {
          m[u] |= m[u - 1];
          m[u - 1] = 0u;
        }
      }
#pragma unroll
      for (int u = 0; u < 4; u++)
        if (m[u])
          atomicOr(&sBmWords[word[u]], m[u]);
    };
    // two groups per thread and step, loads first. A group's left neighbour is the last edge of the lane
    // before, whose group lies directly in front; the wave's first lane fetches its own.
#ifdef F3S_PROBE_PRE_NO_FILL
    if (nb < 0)
#endif
    for (int e0 = sp.gA + 4 * tid; e0 < sp.gB; e0 += 4 * U * TB) {
      int4 c[U];
      load_groups<TB, U>(colIdx, sp, e0, c);
      int left[U];
#pragma unroll
      for (int g = 0; g < U; g++) {
        const int e = e0 + 4 * g * TB;
        left[g] = -1;
        if (first && lane == 0 && e > eS && e < sp.gB) left[g] = colIdx[e - 1];
      }
#pragma unroll
      for (int g = 0; g < U; g++) {
        left[g] = __builtin_amdgcn_update_dpp(left[g], c[g].w, 0x138, 0xf, 0xf, false);  // wave_shr:1
        if (e0 + 4 * g * TB < sp.gB) group(e0 + 4 * g * TB, c[g], left[g]);
      }
    }
    // Edge by edge: the groups with a row boundary inside (lanes 4 k - 4 .. 4 k - 1 of the first wave take
    // the group around the start of row k, unless row k - 1 starts inside it too) and the loose ends
    // (the second wave). Inside the loop above such a group would hold up its whole wave.
    if (tid < 128) {
      int e = -1;
      if (tid < 64) {
        const int k = (tid >> 2) + 1;
        const int start = sRow[k];
        const int g = start & ~3;
        if (k < 16 && start != g && g >= sp.gA && g < sp.gB && sRow[k - 1] <= g) e = g + (tid & 3);
      } else {
        e = loose_edge(sp, eS, eE, tid - 64);
      }
      if (e >= 0) one_edge(e, colIdx[e], row_of_edge(sRow, e));
    }
  };

  unsigned carry = (unsigned)eS;  // absolute edge position where the next TC block starts
  const int stageBytes = (bitsetBytes / NWAVE) & ~15;
  const int TC = idsInLds ? nb : chunkBytes / (WPT * 8);
  for (int tc0 = 0; tc0 < nb; tc0 += TC) {
    const int nt = min(TC, nb - tc0);
    const bool lastChunk = tc0 + TC >= nb;
    if (tc0 > 0) lds_barrier();  // the previous chunk is out
    for (int i = tid; i < nt * WPT; i += TB) sBm[i] = 0ull;
    lds_barrier();  // ranks are read after the prefixes are written
    if (idsInLds)
      rank_edges(std::true_type{}, 0, nt);
    else
      rank_edges(std::false_type{}, tc0, nt);
    lds_barrier();
    if (sUnsorted != 0u) break;  // known after the first pass over the window's edges
    for (int tb = 0; tb < nt; tb += TB) {
      const int t = tb + tid;
      unsigned long long words[WPT];
      unsigned nnz = 0;
      if (t < nt) {
#pragma unroll
        for (int k = 0; k < WPT; k++) {
          words[k] = sBm[t * WPT + k];
          nnz += __popcll(words[k]);
        }
      }
      const unsigned inc = wave_inclusive_scan(nnz, lane);
      if (lane == 63) sWaveTot[wave] = inc;
      lds_barrier();
      unsigned waveOff = 0, tileTot = 0;
#pragma unroll
      for (int v = 0; v < NWAVE; v++) {
        const unsigned x = sWaveTot[v];
        if (v < wave) waveOff += x;
        tileTot += x;
      }
      // tile ids: a block's set bits read row by row (src/utils.cu:213-223 walks the edges of a
      // window with ascending rows in exactly that order). In the window's last chunk the bitset
      // is no longer needed: each wave then collects the bytes of its 64 blocks in its slice of
      // that LDS and writes them out as whole dwords.
      const unsigned waveTot = __shfl(inc, 63);
      const unsigned wavePos0 = carry + waveOff;
      const unsigned a0 = wavePos0 & ~3u;
      const bool staged = lastChunk && waveTot + 3u <= (unsigned)stageBytes;
      uint8_t* stage = reinterpret_cast<uint8_t*>(smem) + wave * stageBytes;
      if (t < nt) {
        const int64_t gt = (int64_t)base + tc0 + t;
        const unsigned pos = wavePos0 + inc - nnz;
        tcblockOffset[gt] = (int)pos;
        tcblockRowid[gt] = w;
        // two calls, so that each store knows its address space (LDS or global)
#ifndef F3S_PROBE_PRE_NO_TILEIDS
        if (staged)
          walk_tile_ids<W>(words, stage, pos - a0);
        else
          walk_tile_ids<W>(words, tcblocktileId, pos);
#endif
      }
      if (staged && waveTot != 0u) {
        wave_lds_sync();
        const unsigned end = wavePos0 + waveTot;
        const unsigned d0 = min((wavePos0 + 3u) & ~3u, end);  // first whole dword
        const unsigned d1 = max(end & ~3u, d0);                // end of the whole dwords
        for (unsigned i = wavePos0 + lane; i < d0; i += 64) tcblocktileId[i] = stage[i - a0];
        for (unsigned i = d0 + 4u * lane; i < d1; i += 256u)
          *reinterpret_cast<uint32_t*>(tcblocktileId + i) =
              *reinterpret_cast<const uint32_t*>(stage + (i - a0));
        for (unsigned i = d1 + lane; i < end; i += 64) tcblocktileId[i] = stage[i - a0];
        wave_lds_sync();
      }
      carry += tileTot;
      lds_barrier();
    }
    {
      unsigned long long* bmDst = bitmap + ((int64_t)base + tc0) * WPT;
      for (int i = tid; i < nt * WPT; i += TB) __builtin_nontemporal_store(sBm[i], bmDst + i);
    }
    if (idsInLds) {
      // The ids, four per thread and step, their upper halves from the ranks at which those change (mostly
      // not within a wave's step); the slots that the last block leaves unused hold 0.
      const uint2* lows = reinterpret_cast<const uint2*>(sBm + nt * WPT);
      uint4* idDst = reinterpret_cast<uint4*>(sparseAToXidx + (int64_t)base * W);
      unsigned from[HIGH];
#pragma unroll
      for (int h = 1; h < HIGH; h++) from[h] = (unsigned)uniform((int)sHigh[h]);
      for (int i = tid; i < nt * (W / 4); i += TB) {
        const uint2 low = lows[i];
        const unsigned first = 4u * i, last = first + 3u;
        unsigned high = 0, highLast = 0;
#pragma unroll
        for (int h = 1; h < HIGH; h++) {
          high += first >= from[h] ? 1u : 0u;
          highLast += last >= from[h] ? 1u : 0u;
        }
        high <<= 16;
        uint4 id = make_uint4((low.x & 0xFFFFu) | high, (low.x >> 16) | high,
                              (low.y & 0xFFFFu) | high, (low.y >> 16) | high);
        if (high != highLast << 16 || last >= nCols) {
          unsigned v[4] = {low.x & 0xFFFFu, low.x >> 16, low.y & 0xFFFFu, low.y >> 16};
#pragma unroll
          for (int u = 0; u < 4; u++) {
#pragma unroll
            for (int h = 1; h < HIGH; h++) v[u] += first + u >= from[h] ? 0x10000u : 0u;
            if (first + u >= nCols) v[u] = 0u;
          }
          id = make_uint4(v[0], v[1], v[2], v[3]);
        }
        store_streaming(idDst + i, id);
      }
    }
  }
  if (sUnsorted != 0u) {
    // repeated or descending columns somewhere in the window: the general way, from the
    // edgeToColumn entries written above (visible to the whole workgroup after the barrier)
    __syncthreads();
    if (tid == 0) sUnsorted = 0u;
    __syncthreads();
    const int dynBytes = bitsetBytes + chunkBytes;
    const int tcg = dynBytes / (64 + WPT * 8);
    unsigned* gCnt = reinterpret_cast<unsigned*>(smem);                                // [tcg*16]
    unsigned long long* gBm = reinterpret_cast<unsigned long long*>(smem + tcg * 16);  // [tcg*WPT]
    fill_window_generic<W, TB>(colIdx, edgeToColumn, w, base, nb, tcg, tcblockRowid,
                               tcblocktileId, tcblockOffset, sparseAToXidx, bitmap, gCnt, gBm, sRow,
                               sWaveTot, &sUnsorted);
  }
}

__global__ void set_tail_kernel(int32_t* tcblockOffset, long long nTcb, int E) {
  tcblockOffset[nTcb] = E;
}

__global__ void clear_header_kernel(WsHeader* hdr) { *hdr = WsHeader{}; }

size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

}  // namespace

// waves of the multi-workgroup finalize (0: the single-workgroup kernel is used)
int finalize_waves(int nRW) {
  if (nRW <= kFinSingleMax) return 0;
  const int w = (nRW + 511) / 512;
  return w < 4096 ? w : 4096;
}

size_t preprocess_workspace_bytes(int N, int /*E*/) {
  const size_t nRW = (size_t)(N + kWinRows - 1) / kWinRows;
  const size_t fin = (size_t)finalize_waves((int)nRW) * (2 + kFinBins) * sizeof(int32_t);
  return kWsHeaderBytes + 3 * align256(nRW * sizeof(int32_t)) + align256(fin);
}

namespace {

// long windows on average: a workgroup per window instead of a wave
bool long_windows(int nRW, int64_t E) { return E >= (int64_t)nRW * 2048; }

// Kernels of more than 64 KiB of LDS have to be told.
template <typename KernelT>
int allow_lds(KernelT kernel, size_t bytes) {
  if (bytes > 64 * 1024)
    F3S_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                      hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes));
  return 0;
}

// Scan of the block counts and (unless it is made beside the fill, see order_beside_fill) the window
// order, after the kernels that write blockPartition.
int enqueue_finalize(int N, int W, const int32_t* blockPartition, int32_t* rowWindowOffset,
                     int32_t* sortedRowWindows, bool order, char* ws, long long* nTcb,
                     hipStream_t stream) {
  const int nRW = (N + kWinRows - 1) / kWinRows;
  WsHeader* hdr = reinterpret_cast<WsHeader*>(ws);
  const size_t seg = align256((size_t)nRW * sizeof(int32_t));
  int32_t* keysA = reinterpret_cast<int32_t*>(ws + kWsHeaderBytes);
  int32_t* keysB = reinterpret_cast<int32_t*>(ws + kWsHeaderBytes + seg);
  int32_t* valsTmp = reinterpret_cast<int32_t*>(ws + kWsHeaderBytes + 2 * seg);
  const int finWaves = finalize_waves(nRW);
  if (finWaves == 0) {
    const int nBins = order_bins(N, W);
    hipLaunchKernelGGL(finalize_count_kernel,
                       dim3(1 + (unsigned)((nRW + kFinBlock - 1) / kFinBlock)), dim3(kFinBlock),
                       nBins * sizeof(uint32_t), stream, blockPartition, nRW, nBins,
                       rowWindowOffset, sortedRowWindows, nTcb);
    F3S_HIP_CHECK(hipGetLastError());
    return 0;
  }
  unsigned* waveSum = reinterpret_cast<unsigned*>(ws + kWsHeaderBytes + 3 * seg);
  int* waveMax = reinterpret_cast<int*>(waveSum + finWaves);
  unsigned* hist = waveSum + 2 * (size_t)finWaves;
  const dim3 grid((unsigned)((finWaves + 3) / 4)), block(256);
  hipLaunchKernelGGL(finalize_partials_kernel, grid, block, 0, stream, blockPartition, nRW,
                     finWaves, waveSum, waveMax,
                     order ? nullptr : reinterpret_cast<uint16_t*>(keysB));
  hipLaunchKernelGGL(finalize_scan_kernel, grid, block, 0, stream, blockPartition, nRW, finWaves,
                     waveSum, waveMax, rowWindowOffset, order ? hist : nullptr, hdr, nTcb);
  F3S_HIP_CHECK(hipGetLastError());
  if (!order) return 0;
  // a window holds at most ceil(N / W) blocks: that bounds the passes that can be needed
  int maxBits = 0;
  while ((((int64_t)N + W - 1) / W >> maxBits) != 0) maxBits++;
  const int maxPass = (maxBits + kFinDigitBits - 1) / kFinDigitBits;
  for (int pass = 0; pass < (maxPass > 0 ? maxPass : 1); pass++) {
    if (pass > 0)
      hipLaunchKernelGGL(finalize_histogram_kernel, grid, block, 0, stream, nRW, finWaves, pass,
                         keysA, keysB, hist, hdr);
    hipLaunchKernelGGL(finalize_scatter_kernel, grid, block, 0, stream, blockPartition, nRW,
                       finWaves, pass, sortedRowWindows, keysA, keysB, valsTmp, hist, hdr);
  }
  F3S_HIP_CHECK(hipGetLastError());
  return 0;
}

// Workgroups that look for the windows of more than minEdges edges: one for each that there can be, so
// that the device deals them out as workgroups end (a fixed 1024 of them met up to 13 of the 4 272
// windows of a 61M-edge graph, 4.2 on average: 200 instead of 149 us), within `most`.
unsigned long_grid(int nRW, int E, int minEdges, int most) {
  int grid = E / (minEdges + 1) + 1;
  if (grid > nRW) grid = nRW;
  return (unsigned)(grid > most ? most : grid);
}

// Graphs whose short and long windows share a launch in both phases. Above kFinSingleMax windows the
// workgroups of one wave are the better ones: with more than four rounds of windows on every CU the
// LDS that a finished wave keeps until its workgroup ends costs more than the overlap gives.
bool one_launch(int nRW, int64_t E) { return nRW <= kFinSingleMax && !long_windows(nRW, E); }
// Their workgroups for windows of more than kBinsMax edges, one for each that there can be; where such windows
// are the exception 512 or 1024, as most look in vain and the short windows wait for their slots. 1024, so
// that fewer meet two long ones, where long windows are to be expected (512 -> 1024, means of six orders of
// the nodes; R-MAT, 130k nodes, 420 edges a window: 110 -> 103 us, power-law, 250k nodes, 420: 136 -> 125;
// even, 65k nodes, 200, none of them long: 59.4 -> 61).
constexpr int64_t kLongGroupsEdges = 1250000;
unsigned all_long_groups(int nRW, int E) {
  const int mean = E / nRW;
  const int most = mean > kBinsMax / 2 ? kFinSingleMax
                   : mean >= kBinsMax / 4 && E >= kLongGroupsEdges ? 1024 : 512;
  return long_grid(nRW, E, kBinsMax, most);
}

// Above kFinSingleMax windows the order is made in the last launch of the fill, where most CUs are idle:
// nRW / 1024 workgroups add up the rows of a histogram that the scan's first kernel leaves. A radix sort
// between the phases is five launches; a call's time in us with it and without: 17 000 windows 153 ->
// 117, 69 000 250 -> 212, 153 000 815 -> 763, 262 000 625 -> 573, 500 000 2140 -> 2077. Beyond, the
// workgroups' readings (nRW^2 / 512 bytes) grow faster than the sort.
constexpr int kOrderBesideMax = 524288;
bool order_beside_fill(int nRW, int64_t E) {
  return nRW > kFinSingleMax && nRW <= kOrderBesideMax && !long_windows(nRW, E);
}

// Eight waves or four: of eight, the few long windows of a skewed graph are done sooner, and where there are
// several rounds of short ones the chip starts fewer workgroups; four keep LDS for the rest of a workgroup
// less long and take more long windows at once where those are many (four -> eight waves, call in us; R-MAT
// of 130k nodes and 200, 340, 420 edges a window: 86 -> 83, 109 -> 99, 118 -> 104; power-law, 250k nodes, 340:
// 138 -> 119; even, 250k nodes, 260: 91 -> 89; but even, 65k nodes, 260: 60.6 -> 62, power-law, 130k
// nodes, 700: 124 -> 129).
constexpr int64_t kRankWideEdges = 1250000;
constexpr int kRankWideWindows = 8000;
bool rank_all_wide(int nRW, int64_t E) {
  return E / nRW <= kBinsMax / 2 && (E >= kRankWideEdges || nRW >= kRankWideWindows);
}
template <int W, int TB>
int launch_rank_all(const int32_t* rowPtr, const int32_t* colIdx, int N, int nRW, int colBits, int range,
                    unsigned longGroups, int32_t* blockPartition, int32_t* edgeToColumn,
                    int32_t* edgeToRow, int* error, hipStream_t stream) {
  constexpr int NW = TB / 64;
  const size_t bins = NW * sizeof(RankBinsLds);
  const size_t bitset = (size_t)(range / 32 + range / 128) * sizeof(uint32_t);
  const size_t lds = bins > bitset ? bins : bitset;
  auto kernel = window_rank_all_kernel<W, TB>;
  if (int rc = allow_lds(kernel, lds)) return rc;
  hipLaunchKernelGGL(kernel, dim3(longGroups + (unsigned)((nRW + NW - 1) / NW)), dim3(TB), lds, stream, rowPtr,
                     colIdx, N, nRW, colBits, range, (int)longGroups, blockPartition, edgeToColumn,
                     edgeToRow, error);
  F3S_HIP_CHECK(hipGetLastError());
  return 0;
}

// Enqueues the kernels that rank the windows' columns and count their TC blocks. sortedRowWindows holds
// the lists of long windows until the order is written.
template <int W>
int enqueue_rank(const int32_t* rowPtr, const int32_t* colIdx, int N, int E, char* ws,
                 int32_t* sortedRowWindows, int32_t* blockPartition, int32_t* edgeToColumn, int32_t* edgeToRow, int* error,
                 hipStream_t stream) {
  const int nRW = (N + kWinRows - 1) / kWinRows;
  if (nRW == 0) return 0;
  int range = ((N + 127) / 128) * 128;
  if (range > kRangeMax) range = kRangeMax;
  const int nPasses = (N + range - 1) / range;
  const size_t lds = (size_t)(range / 32 + range / 128) * sizeof(uint32_t);
  // short windows: packed (column, position) words when the column ids leave room for the
  // position, else the bitonic network on bare column ids
  int colBits = 0;
  while (colBits < 31 && ((int64_t)1 << colBits) < (int64_t)N) colBits++;
  if (one_launch(nRW, E)) {
    const unsigned groups = all_long_groups(nRW, E);
    auto launch = rank_all_wide(nRW, E) ? launch_rank_all<W, 512> : launch_rank_all<W, 256>;
    return launch(rowPtr, colIdx, N, nRW, colBits, range, groups, blockPartition, edgeToColumn, edgeToRow,
                  error, stream);
  }
  int shortMax = kBinsMax;
  WsHeader* hdr = reinterpret_cast<WsHeader*>(ws);
  LongQueue queue = {nullptr, nullptr, 0, 0};
  if (!long_windows(nRW, E)) {
    queue = {&hdr->rank, sortedRowWindows, nRW, nPasses >= 2 ? kMidMax : 0};
    hipLaunchKernelGGL(clear_header_kernel, dim3(1), dim3(1), 0, stream, hdr);
  }
  if (colBits <= 22) {
    hipLaunchKernelGGL(window_rank_bins_kernel<W>, dim3(nRW), dim3(64), 0, stream, rowPtr,
                       colIdx, N, colBits, queue, blockPartition, edgeToColumn, edgeToRow, error);
  } else {
    shortMax = kSortMax;
    hipLaunchKernelGGL(window_rank_small_kernel<W>, dim3(nRW), dim3(64), 0, stream, rowPtr, colIdx, N,
                       nRW, queue, blockPartition, edgeToColumn, edgeToRow, error);
  }
  F3S_HIP_CHECK(hipGetLastError());
  if (long_windows(nRW, E)) {
    hipLaunchKernelGGL((window_rank_kernel<W, 512, false>), dim3(nRW), dim3(512), lds, stream,
                       rowPtr, colIdx, N, nRW, range, nPasses, shortMax, queue, blockPartition,
                       edgeToColumn, edgeToRow, error);
    F3S_HIP_CHECK(hipGetLastError());
    return 0;
  }
  // The longer ones, from the lists. On a graph that needs several bitset passes, windows of a few thousand edges
  // are sorted instead of walking every pass: up to kMidMax edges by 256 threads each, and those of up to kLargeMax
  // by 1024, in one launch with the longer ones, which do walk the passes.
  if (nPasses >= 2) {
    auto rest = window_rank_rest_kernel<W>;
    const size_t restLds = rank_rest_lds(lds);
    if (int rc = allow_lds(rest, restLds)) return rc;
    constexpr size_t midLds = rank_sort_lds<kMidItems, kMidThreads>();
    hipLaunchKernelGGL(window_rank_mid_kernel<W>, dim3(long_grid(nRW, E, shortMax, 8192)), dim3(kMidThreads),
                       midLds, stream, rowPtr, colIdx, N, colBits, queue, blockPartition, edgeToColumn,
                       edgeToRow, error);
    hipLaunchKernelGGL(rest, dim3(long_grid(nRW, E, kMidMax, 1024)), dim3(kLargeThreads), restLds, stream,
                       rowPtr, colIdx, N, colBits, range, nPasses, queue, blockPartition, edgeToColumn,
                       edgeToRow, error);
    F3S_HIP_CHECK(hipGetLastError());
    return 0;
  }
  // sixteen waves per window: what counts is how soon the longest one is done (169k-node R-MAT graph,
  // windows of up to 12 500 edges: 31 us with four)
  hipLaunchKernelGGL((window_rank_kernel<W, 1024, true>), dim3(long_grid(nRW, E, shortMax, 512)),
                     dim3(1024), lds, stream, rowPtr, colIdx, N, nRW, range, nPasses, shortMax, queue,
                     blockPartition, edgeToColumn, edgeToRow, error);
  F3S_HIP_CHECK(hipGetLastError());
  return 0;
}
int enqueue_rank(const int32_t* rowPtr, const int32_t* colIdx, int N, int E, int W, char* ws,
                 int32_t* sortedRowWindows, int32_t* blockPartition, int32_t* edgeToColumn,
                 int32_t* edgeToRow, int* error, hipStream_t stream) {
  return W == 16 ? enqueue_rank<16>(rowPtr, colIdx, N, E, ws, sortedRowWindows, blockPartition,
                                    edgeToColumn, edgeToRow, error, stream)
                 : enqueue_rank<8>(rowPtr, colIdx, N, E, ws, sortedRowWindows, blockPartition,
                                   edgeToColumn, edgeToRow, error, stream);
}

// Enqueues every kernel of phase 1 on `stream`, the window order only if `order`; `ws` is device scratch
// of preprocess_workspace_bytes(N, E) bytes.
int enqueue_count(const int32_t* rowPtr, const int32_t* colIdx, int N, int E, int W,
                  int32_t* blockPartition, int32_t* edgeToColumn, int32_t* edgeToRow,
                  int32_t* rowWindowOffset, int32_t* sortedRowWindows, bool order, char* ws,
                  const ResultPtr& result, hipStream_t stream) {
  if (int rc = enqueue_rank(rowPtr, colIdx, N, E, W, ws, sortedRowWindows, blockPartition,
                            edgeToColumn, edgeToRow, result.error, stream))
    return rc;
  return enqueue_finalize(N, W, blockPartition, rowWindowOffset, sortedRowWindows, order, ws,
                          result.nTcb, stream);
}

// Pinned host memory for the results of calls that wait for the device: a slot per call in progress,
// taken from pages of 64 slots that stay with the library (one page unless more than 64 host
// threads preprocess at a time). The free slots are a list through the slots themselves, so that
// neither taking one nor giving it back can run out of host memory and throw through the C ABI.
struct HostResult {
  long long nTcb;
  int error;
  HostResult* next;  // of the free list
  int pad[10];
};
static_assert(sizeof(HostResult) == 64, "a line of its own");
class HostResultLease {
 public:
  int take() {
    std::lock_guard<std::mutex> lock(mutex_);
    if (!free_) {
      void* page = nullptr;
      F3S_HIP_CHECK(hipHostMalloc(&page, 64 * sizeof(HostResult), hipHostMallocPortable));
      for (int i = 0; i < 64; i++) give_back(static_cast<HostResult*>(page) + i);
    }
    slot_ = free_;
    free_ = slot_->next;
    slot_->nTcb = 0;
    slot_->error = 0;
    return 0;
  }
  ~HostResultLease() {
    if (!slot_) return;
    std::lock_guard<std::mutex> lock(mutex_);
    give_back(slot_);
  }
  // The host could not wait for the stream (a stream under capture, a lost device): kernels that hold
  // the slot's address may still run, so nobody else gets it.
  void abandon() { slot_ = nullptr; }
  ResultPtr pointers() const { return {&slot_->nTcb, &slot_->error}; }
  // after the stream is done
  const volatile HostResult& value() const { return *slot_; }

 private:
  static void give_back(HostResult* slot) {  // under the lock
    slot->next = free_;
    free_ = slot;
  }
  static std::mutex mutex_;
  static HostResult* free_;
  HostResult* slot_ = nullptr;
};
std::mutex HostResultLease::mutex_;
HostResult* HostResultLease::free_ = nullptr;

int check_count_args(const char* who, int N, int E, int H, int W) {
  if (H != 16 || (W != 16 && W != 8))
    return fail(-2, "%s: block %dx%d unsupported (16x16 or 16x8)", who, H, W);
  if (N < 0 || E < 0) return fail(-2, "%s: negative size", who);
  return 0;
}

}  // namespace

int launch_preprocess_count(const int32_t* rowPtr, const int32_t* colIdx, int N, int E, int H,
                            int W, int32_t* blockPartition, int32_t* edgeToColumn,
                            int32_t* edgeToRow, int32_t* rowWindowOffset,
                            int32_t* sortedRowWindows, void* workspace, size_t wsBytes,
                            int64_t* nTcbHost, hipStream_t stream) {
  if (int rc = check_count_args("f3s_preprocess_count", N, E, H, W)) return rc;
  if (wsBytes < preprocess_workspace_bytes(N, E))
    return fail(-2, "f3s_preprocess_count: workspace %zu B < required %zu B", wsBytes,
                preprocess_workspace_bytes(N, E));
  HostResultLease result;
  if (int rc = result.take()) return rc;
  int rc = enqueue_count(rowPtr, colIdx, N, E, W, blockPartition, edgeToColumn, edgeToRow,
                         rowWindowOffset, sortedRowWindows, true, static_cast<char*>(workspace),
                         result.pointers(), stream);
  // also after a failed launch: the slot must not be written to any more when it is given back
  const hipError_t done = hipStreamSynchronize(stream);
  if (done != hipSuccess) result.abandon();
  if (rc != 0) return rc;
  F3S_HIP_CHECK(done);
  if (result.value().error)
    return fail(-4, "f3s_preprocess_count: column index outside [0, %d)", N);
  *nTcbHost = result.value().nTcb;
  return 0;
}

// ------------------------------------------------------- phase 1 without any allocation
// The scratch is the file-scope array `scratch` at the top of this file; host code reaches it
// through the per-device address hipGetSymbolAddress returns, looked up once per device.
constexpr size_t kStaticScratchBytes = kF3sStaticScratchBytes;

namespace {

constexpr int kMaxDevices = 64;
std::mutex g_scratchMutex;
void* g_scratchPtr[kMaxDevices] = {};

int static_scratch(char** out) {
  int dev = -1;
  F3S_HIP_CHECK(hipGetDevice(&dev));
  if (dev < 0 || dev >= kMaxDevices)
    return fail(-2, "f3s_preprocess_count_static: device index %d out of range", dev);
  std::lock_guard<std::mutex> lock(g_scratchMutex);
  if (!g_scratchPtr[dev]) {
    void* ptr = nullptr;
    F3S_HIP_CHECK(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
    g_scratchPtr[dev] = ptr;
  }
  *out = static_cast<char*>(g_scratchPtr[dev]);
  return 0;
}

__global__ void clear_result_kernel(long long* result) {
  result[0] = 0;
  result[1] = 0;
}

}  // namespace

size_t preprocess_static_scratch_bytes() { return kStaticScratchBytes; }

int launch_preprocess_count_static(const int32_t* rowPtr, const int32_t* colIdx, int N, int E,
                                   int H, int W, int32_t* blockPartition, int32_t* edgeToColumn,
                                   int32_t* edgeToRow, int32_t* rowWindowOffset,
                                   int32_t* sortedRowWindows, int64_t* resultDev,
                                   hipStream_t stream) {
  if (int rc = check_count_args("f3s_preprocess_count_static", N, E, H, W)) return rc;
  if (preprocess_workspace_bytes(N, E) > kStaticScratchBytes)
    return fail(-5, "f3s_preprocess_count_static: a graph of %d nodes needs %zu B of scratch, the "
                    "library's own buffer holds %zu B; use f3s_preprocess_count with a workspace",
                N, preprocess_workspace_bytes(N, E), kStaticScratchBytes);
  char* ws = nullptr;
  if (int rc = static_scratch(&ws)) return rc;
  // every kernel below overwrites whatever it reads of the buffer, so nothing of an earlier call
  // survives into this one
  auto* result = reinterpret_cast<long long*>(resultDev);
  hipLaunchKernelGGL(clear_result_kernel, dim3(1), dim3(1), 0, stream, result);
  F3S_HIP_CHECK(hipGetLastError());
  // the error flag is the low half of the second value
  return enqueue_count(rowPtr, colIdx, N, E, W, blockPartition, edgeToColumn, edgeToRow,
                       rowWindowOffset, sortedRowWindows, true, ws,
                       {result, reinterpret_cast<int*>(result + 1)}, stream);
}

namespace {

// Enqueues phase 2. With sortedRowWindows (not null: order_beside_fill) the window order is written
// too, from blockPartition; with nTcb (not null: at most kSelfScanMax windows) rowWindowOffset and the
// total as well. ws: the workspace of phase 1, or null (the long windows are then looked for).
template <int W>
int enqueue_fill(const int32_t* rowPtr, const int32_t* colIdx, int N, int E,
                 const int32_t* edgeToColumn, int32_t* rowWindowOffset,
                 const int32_t* blockPartition, int32_t* sortedRowWindows, long long* nTcb, char* ws,
                 int32_t* tcblockRowid, uint8_t* tcblocktileId, int32_t* tcblockOffset,
                 int32_t* sparseAToXidx, uint64_t* bitmap, hipStream_t stream) {
  const int nRW = (N + kWinRows - 1) / kWinRows;
  auto bm = reinterpret_cast<unsigned long long*>(bitmap);
  // Graphs of windows with thousands of edges: eight waves per window.
  if (long_windows(nRW, E)) {
    auto kernel = window_fill_kernel<W, 512, kFillChunk, kFillChunkGeneric>;
    constexpr size_t lds = fill_lds_bytes<W>(kFillChunk, kFillChunkGeneric);
    hipLaunchKernelGGL(kernel, dim3(nRW), dim3(512), lds, stream, rowPtr, colIdx, N, E,
                       edgeToColumn, rowWindowOffset, tcblockRowid, tcblocktileId, tcblockOffset,
                       sparseAToXidx, bm);
    F3S_HIP_CHECK(hipGetLastError());
    return 0;
  }
  if (one_launch(nRW, E)) {
    const unsigned longGroups = all_long_groups(nRW, E);
    const unsigned orderGroups =
        sortedRowWindows ? (unsigned)((nRW + kFillAllThreads - 1) / kFillAllThreads) : 0;
    constexpr int NW = kFillAllThreads / 64;
    const unsigned grid = longGroups + orderGroups + (unsigned)((nRW + NW - 1) / NW);
    const int nBins = order_bins(N, W);
    const size_t lds = fill_all_lds<W>(nBins);
    auto kernel = nTcb ? window_fill_all_kernel<W, true> : window_fill_all_kernel<W, false>;
    if (int rc = allow_lds(kernel, lds)) return rc;
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(kFillAllThreads), lds, stream, rowPtr, colIdx, N, E,
                       nRW, edgeToColumn, blockPartition, (int)longGroups, (int)orderGroups, nBins,
                       rowWindowOffset, sortedRowWindows, nTcb, tcblockRowid, tcblocktileId,
                       tcblockOffset, sparseAToXidx, bm);
    F3S_HIP_CHECK(hipGetLastError());
    return 0;
  }
  // few long windows (at most kFillFewLong, and as windows have at most half of kBinsMax edges on
  // average, commonly far fewer): the large workgroups take all of them, which saves a launch
  const bool few = E / kBinsMax <= kFillFewLong && E / nRW <= kBinsMax / 2;
  LongQueue queue = {nullptr, nullptr, 0, 0};
  const uint16_t* orderRows = nullptr;
  if (ws) {  // phase 1 has cleared the counts and is done with the keys behind the header
    queue = {&reinterpret_cast<WsHeader*>(ws)->fill, reinterpret_cast<int32_t*>(ws + kWsHeaderBytes), nRW,
             few ? 0 : kFillMid};
    const size_t seg = align256((size_t)nRW * sizeof(int32_t));
    orderRows = reinterpret_cast<const uint16_t*>(ws + kWsHeaderBytes + seg);
  }
  hipLaunchKernelGGL((window_fill_short_kernel<W>), dim3(nRW), dim3(64), 0, stream, rowPtr, colIdx, N,
                     E, nRW, edgeToColumn, rowWindowOffset, queue, tcblockRowid, tcblocktileId,
                     tcblockOffset, sparseAToXidx, bm);
  F3S_HIP_CHECK(hipGetLastError());
  int minEdges = kBinsMax;
  if (!few) {
    auto mid = window_fill_long_kernel<W, 256, kFillChunkMid, false>;
    constexpr size_t lds = fill_lds_bytes<W>(kFillChunkMid, kFillChunkMid);
    hipLaunchKernelGGL(mid, dim3(long_grid(nRW, E, minEdges, 8192)), dim3(256), lds, stream, rowPtr,
                       colIdx, N, E, nRW, edgeToColumn, rowWindowOffset, queue, minEdges, kFillMid, 0,
                       nullptr, nullptr, nullptr, tcblockRowid, tcblocktileId, tcblockOffset, sparseAToXidx, bm);
    F3S_HIP_CHECK(hipGetLastError());
    minEdges = kFillMid;
  }
  auto kernel = window_fill_long_kernel<W, 1024, kFillChunkLong, true>;
  constexpr size_t lds = fill_lds_bytes<W>(kFillChunkLong, kFillChunkLong);
  static_assert(lds >= 2 * kOrderRowBins * sizeof(uint32_t), "order_chunk's arrays");
  if (int rc = allow_lds(kernel, lds)) return rc;
  const unsigned orderGroups =
      sortedRowWindows ? (unsigned)((nRW + kOrderRowWindows - 1) / kOrderRowWindows) : 0;
  hipLaunchKernelGGL(kernel, dim3(orderGroups + long_grid(nRW, E, minEdges, 255)), dim3(1024), lds,
                     stream, rowPtr, colIdx, N, E, nRW, edgeToColumn, rowWindowOffset, queue, minEdges,
                     0x7FFFFFFF, (int)orderGroups, blockPartition, orderRows, sortedRowWindows,
                     tcblockRowid, tcblocktileId, tcblockOffset, sparseAToXidx, bm);
  F3S_HIP_CHECK(hipGetLastError());
  return 0;
}
int enqueue_fill(const int32_t* rowPtr, const int32_t* colIdx, int N, int E, int W,
                 const int32_t* edgeToColumn, int32_t* rowWindowOffset,
                 const int32_t* blockPartition, int32_t* sortedRowWindows, long long* nTcb, char* ws,
                 int32_t* tcblockRowid, uint8_t* tcblocktileId, int32_t* tcblockOffset,
                 int32_t* sparseAToXidx, uint64_t* bitmap, hipStream_t stream) {
  return W == 16 ? enqueue_fill<16>(rowPtr, colIdx, N, E, edgeToColumn, rowWindowOffset,
                                    blockPartition, sortedRowWindows, nTcb, ws, tcblockRowid,
                                    tcblocktileId, tcblockOffset, sparseAToXidx, bitmap, stream)
                 : enqueue_fill<8>(rowPtr, colIdx, N, E, edgeToColumn, rowWindowOffset,
                                   blockPartition, sortedRowWindows, nTcb, ws, tcblockRowid,
                                   tcblocktileId, tcblockOffset, sparseAToXidx, bitmap, stream);
}

}  // namespace

int launch_preprocess_fill(const int32_t* rowPtr, const int32_t* colIdx, int N, int E, int H,
                           int W, const int32_t* edgeToColumn, const int32_t* rowWindowOffset,
                           int64_t nTcb, int32_t* tcblockRowid, uint8_t* tcblocktileId,
                           int32_t* tcblockOffset, int32_t* sparseAToXidx, uint64_t* bitmap,
                           hipStream_t stream) {
  if (H != 16 || (W != 16 && W != 8))
    return fail(-2, "f3s_preprocess_fill: block %dx%d unsupported (16x16 or 16x8)", H, W);
  const int nRW = (N + kWinRows - 1) / kWinRows;
  if (nRW == 0) {
    hipLaunchKernelGGL(set_tail_kernel, dim3(1), dim3(1), 0, stream, tcblockOffset,
                       (long long)nTcb, E);
    F3S_HIP_CHECK(hipGetLastError());
    return 0;
  }
  // the offsets are only read: without nTcb nothing writes them
  return enqueue_fill(rowPtr, colIdx, N, E, W, edgeToColumn, const_cast<int32_t*>(rowWindowOffset),
                      nullptr, nullptr, nullptr, nullptr, tcblockRowid, tcblocktileId, tcblockOffset,
                      sparseAToXidx, bitmap, stream);
}

int launch_window_order(const int32_t* rowWindowOffset, int nRW, int32_t* order,
                        hipStream_t stream) {
  if (nRW < 0 || nRW > kFinSingleMax)
    return fail(-2, "f3s_window_order: %d windows out of range (0..%d)", nRW, kFinSingleMax);
  if (nRW == 0) return 0;
  hipLaunchKernelGGL(window_order_kernel,
                     dim3((unsigned)((nRW + kOrderOnlyThreads - 1) / kOrderOnlyThreads)),
                     dim3(kOrderOnlyThreads), 0, stream, rowWindowOffset, nRW, order);
  F3S_HIP_CHECK(hipGetLastError());
  return 0;
}

// ------------------------------------------------------- both phases behind one call
int64_t preprocess_capacity(int N, int64_t E, int W) {
  // a window of e edges names at most e distinct columns: ceil(e / W) <= e / W + 1 blocks
  const int64_t nRW = ((int64_t)N + kWinRows - 1) / kWinRows;
  return (E + W - 1) / W + nRW;
}

namespace {

// Both phases, with nothing of the host in between.
int enqueue_preprocess(const int32_t* rowPtr, const int32_t* colIdx, int N, int E, int W,
                       int32_t* blockPartition, int32_t* edgeToColumn, int32_t* edgeToRow,
                       int32_t* rowWindowOffset, int32_t* sortedRowWindows, int32_t* tcblockRowid,
                       uint8_t* tcblocktileId, int32_t* tcblockOffset, int32_t* sparseAToXidx,
                       uint64_t* bitmap, char* ws, const ResultPtr& result, hipStream_t stream) {
  const int nRW = (N + kWinRows - 1) / kWinRows;
  const bool aligned16 =
      ((reinterpret_cast<uintptr_t>(colIdx) | reinterpret_cast<uintptr_t>(edgeToColumn) |
        reinterpret_cast<uintptr_t>(edgeToRow) | reinterpret_cast<uintptr_t>(sparseAToXidx) |
        reinterpret_cast<uintptr_t>(tcblocktileId)) & 15u) == 0;
  // long windows, one bitset pass: the kernels that keep a window's bitset in LDS for both phases
  if (nRW > 0 && long_windows(nRW, E) && N <= kRangeMax && aligned16) {
    WsHeader* hdr = reinterpret_cast<WsHeader*>(ws);
    const int range = ((N + 127) / 128) * 128;
    const int bitsetBytes = rank_fill_bitset_bytes(range);
    // two workgroups of twelve waves per CU (registers allow no more): half of the CU's LDS each
    int chunkBytes = (160 * 1024) / 2 - 1024 - bitsetBytes;
    chunkBytes &= ~255;
    const size_t ldsCount = (size_t)(range / 32) * 4;
    const size_t ldsFill = (size_t)bitsetBytes + chunkBytes;
    hipLaunchKernelGGL(clear_header_kernel, dim3(1), dim3(1), 0, stream, hdr);
#define F3S_ONECALL(WW)                                                                        \
  do {                                                                                         \
    auto rankFill = window_rank_fill_kernel<WW, kRankFillThreads>;                             \
    if (int rc = allow_lds(rankFill, ldsFill)) return rc;                                      \
    hipLaunchKernelGGL((window_count_kernel<WW, 512>), dim3(nRW), dim3(512), ldsCount, stream, \
                       rowPtr, colIdx, N, range, blockPartition, hdr, result.error);           \
    F3S_HIP_CHECK(hipGetLastError());                                                          \
    if (int rc = enqueue_finalize(N, W, blockPartition, rowWindowOffset, sortedRowWindows,     \
                                  true, ws, result.nTcb, stream))                              \
      return rc;                                                                               \
    hipLaunchKernelGGL(rankFill, dim3(nRW), dim3(kRankFillThreads), ldsFill, stream, rowPtr,   \
                       colIdx, N, E, range, chunkBytes, rowWindowOffset, sortedRowWindows,     \
                       hdr, edgeToColumn, edgeToRow, tcblockRowid, tcblocktileId,              \
                       tcblockOffset, sparseAToXidx,                                           \
                       reinterpret_cast<unsigned long long*>(bitmap));                         \
    F3S_HIP_CHECK(hipGetLastError());                                                          \
  } while (0)
    if (W == 16) F3S_ONECALL(16); else F3S_ONECALL(8);
#undef F3S_ONECALL
    return 0;
  }
  // At most the scan stands between the phases; the order is made beside the fill (as its own launch in
  // between it took 23 us of the 219 of a call on 169k nodes).
  if (nRW > 0 && one_launch(nRW, E)) {
    if (int rc = enqueue_rank(rowPtr, colIdx, N, E, W, ws, sortedRowWindows, blockPartition,
                              edgeToColumn, edgeToRow, result.error, stream))
      return rc;
    const bool self = nRW <= kSelfScanMax;
    if (!self) {
      hipLaunchKernelGGL(window_scan_kernel, dim3(1), dim3(kFinBlock), 0, stream, blockPartition,
                         nRW, rowWindowOffset, result.nTcb);
      F3S_HIP_CHECK(hipGetLastError());
    }
    return enqueue_fill(rowPtr, colIdx, N, E, W, edgeToColumn, rowWindowOffset, blockPartition,
                        sortedRowWindows, self ? result.nTcb : nullptr, ws, tcblockRowid,
                        tcblocktileId, tcblockOffset, sparseAToXidx, bitmap, stream);
  }
  const bool beside = order_beside_fill(nRW, E);
  if (int rc = enqueue_count(rowPtr, colIdx, N, E, W, blockPartition, edgeToColumn, edgeToRow,
                             rowWindowOffset, sortedRowWindows, !beside, ws, result, stream))
    return rc;
  if (nRW == 0) {
    hipLaunchKernelGGL(set_tail_kernel, dim3(1), dim3(1), 0, stream, tcblockOffset, 0ll, E);
    F3S_HIP_CHECK(hipGetLastError());
    return 0;
  }
  return enqueue_fill(rowPtr, colIdx, N, E, W, edgeToColumn, rowWindowOffset, blockPartition,
                      beside ? sortedRowWindows : nullptr, nullptr, ws, tcblockRowid, tcblocktileId,
                      tcblockOffset, sparseAToXidx, bitmap, stream);
}

}  // namespace

int launch_preprocess(const int32_t* rowPtr, const int32_t* colIdx, int N, int E, int H, int W,
                      int32_t* blockPartition, int32_t* edgeToColumn, int32_t* edgeToRow,
                      int32_t* rowWindowOffset, int32_t* sortedRowWindows, int64_t capacity,
                      int32_t* tcblockRowid, uint8_t* tcblocktileId, int32_t* tcblockOffset,
                      int32_t* sparseAToXidx, uint64_t* bitmap, void* workspace, size_t wsBytes,
                      int64_t* nTcbHost, hipStream_t stream) {
  if (int rc = check_count_args("f3s_preprocess", N, E, H, W)) return rc;
  if (wsBytes < preprocess_workspace_bytes(N, E))
    return fail(-2, "f3s_preprocess: workspace %zu B < required %zu B", wsBytes,
                preprocess_workspace_bytes(N, E));
  if (capacity < preprocess_capacity(N, E, W))
    return fail(-2, "f3s_preprocess: block arrays sized for %lld TC blocks, the bound for this "
                    "graph is %lld (f3s_preprocess_capacity)",
                (long long)capacity, (long long)preprocess_capacity(N, E, W));
  HostResultLease result;
  if (int rc = result.take()) return rc;
  const int rc = enqueue_preprocess(rowPtr, colIdx, N, E, W, blockPartition, edgeToColumn,
                                    edgeToRow, rowWindowOffset, sortedRowWindows, tcblockRowid,
                                    tcblocktileId, tcblockOffset, sparseAToXidx, bitmap,
                                    static_cast<char*>(workspace), result.pointers(), stream);
  // also after a failed launch: the slot must not be written to any more when it is given back
  const hipError_t done = hipStreamSynchronize(stream);
  if (done != hipSuccess) result.abandon();
  if (rc != 0) return rc;
  F3S_HIP_CHECK(done);
  if (result.value().error) return fail(-4, "f3s_preprocess: column index outside [0, %d)", N);
  *nTcbHost = result.value().nTcb;
  return 0;
}

}  // namespace f3s
