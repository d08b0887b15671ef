// The inner loop of the fused SDDMM -> online softmax -> SpMM kernels for gfx950 (MI355X),
// wave64: one wave walks a run of consecutive TC blocks of one 16-row window, two 16x16 blocks
// (a "pair", 32 keys) per step, with running (m, l, O) in registers. Every kernel of the library
// (workgroup per window, wave per (window, column slice) unit, waves and workgroups mixed, 16x8
// blocks, multi-head, timed) is this loop plus its own prologue and epilogue.
//
// Replaces the loop bodies of f3sKernel1tb1rw / ...Scheduled / ...ScheduledPermutedQKV[ScaleQK],
// f2sKernel1tb1rw and f3sKernel1tb1tcb (src/F3S_kernel.cu:1414-1558, 1040-1150, 2040-2160,
// 2230-2310, 702-853).
//
// Data path of one step (lane = 16*g + c, g in 0..3, c in 0..15):
//   metadata   column ids and bitmaps of four steps at a time: one 16-byte load per lane straight
//              into LDS (global_load_lds), 512 bytes of ids followed by 256 bytes of bitmaps.
//   K, V rows  gathered whole with 16 bytes per lane (D/8 adjacent lanes cover one row: every
//              HBM/L2 access is a full row) straight into this wave's LDS ring, K tile and V tile
//              of a pair side by side, 16-byte chunks XOR-swizzled by the choice of which chunk a
//              lane fetches. Nothing passes through registers on the way in, so the ring, not
//              the register file, holds the loads in flight.
//   S^T = K Q^T  v_mfma_f32_16x16x32, A = K rows read from LDS with one 16-byte read per k-step
//              and block (lane: key slot c, features 32i+8g..+7), B = Q, held in registers for
//              the whole window. The accumulator leaves S[q = c][slot 4g+i], i < 4, in this lane.
//   mask       this lane's 4 + 4 bits sit in one bitmap dword per block; a sign-extending bit
//              field extract turns each into an AND mask.
//   softmax    exponentials are taken against the running maximum m of the lane's row WITHOUT
//              looking for a new maximum first; m (which starts at 0 like the reference's) only
//              moves when a lane's sum of new exponentials exceeds 2^12, i.e. when some score
//              lies more than 12 (log2 units) above it. Then, and when an unmasked score is
//              exactly 0 (which the reference drops, see below), the wave takes the slow path:
//              true row maximum over the four lanes of a row, rescale of l and O, exact zero
//              test. The result is the same softmax (the shift cancels in O / l); P stays below
//              2^12 and keeps fp16's relative precision.
//   O^T += V^T P^T  v_mfma_f32_16x16x32 over the 32 keys of the pair; contraction index 8g+k <->
//              (block A, slot 4g+k) for k < 4, (block B, slot 4g+k-4) for k >= 4, so the B operand
//              is the 8 probabilities this lane already holds. A = V^T comes from LDS through
//              ds_read_b64_tr_b16, which hands lane (g, c) column 16j+c of four consecutive key
//              rows. Lane (g, c) accumulates O[q = c][16j + 4g .. +3] for output tile j.
//
// Numerics follow the reference kernel (src/F3S_kernel.cu:1402-1406,1447-1451,1487-1499,938-945,
// 1560-1561): masked entries do not contribute, an unmasked score that is exactly 0 is dropped
// like a masked one, the row sum uses un-rounded fp32 exponentials while P is rounded to fp16 for
// the second product, empty rows give 0. bf16 inputs (beyond the reference): P is split into a
// bf16 head and a bf16 tail (two products per tile), which keeps 16 bits of P, more than the
// reference's fp16.
#pragma once
#include "f3s_common.h"

namespace f3s {
namespace pipe {

typedef float float4v __attribute__((ext_vector_type(4)));
typedef int int4v __attribute__((ext_vector_type(4)));
typedef int int2v __attribute__((ext_vector_type(2)));
typedef short short4v __attribute__((ext_vector_type(4)));

#define F3S_LDS __attribute__((address_space(3)))

// probe builds can drop one part of a step (results are then wrong on purpose)
#ifdef F3S_PROBE_NO_READ
#define F3S_ABL_READ(x) op = Operands{}
#else
#define F3S_ABL_READ(x) x
#endif
#ifdef F3S_PROBE_NO_GATHER
#define F3S_ABL_GATHER(x) (void)0
#else
#define F3S_ABL_GATHER(x) x
#endif
#ifdef F3S_PROBE_NO_COMPUTE
#define F3S_ABL_COMPUTE(x) consume(op)
#else
#define F3S_ABL_COMPUTE(x) x
#endif

template <typename ET, int L>
struct Vec {
  typedef ET type __attribute__((ext_vector_type(L)));
};
template <typename ET>
__device__ __forceinline__ float4v mfma_16x16x32(typename Vec<ET, 8>::type a,
                                                 typename Vec<ET, 8>::type b, float4v acc);
template <>
__device__ __forceinline__ float4v mfma_16x16x32<_Float16>(Vec<_Float16, 8>::type a,
                                                           Vec<_Float16, 8>::type b,
                                                           float4v acc) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, acc, 0, 0, 0);
}
template <>
__device__ __forceinline__ float4v mfma_16x16x32<__bf16>(Vec<__bf16, 8>::type a,
                                                         Vec<__bf16, 8>::type b, float4v acc) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, acc, 0, 0, 0);
}

constexpr float kLog2e = 1.4426950408889634f;
// a lane's sum of new exponentials above this sends the wave to the slow path (new row maximum)
constexpr float kLazyLimit = 4096.0f;

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }
__device__ __forceinline__ int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }

// max / sum over the four lanes {c, c+16, c+32, c+48} that share a query row
__device__ __forceinline__ float row_max4(float v) {
  v = fmaxf(v, __shfl_xor(v, 16));
  v = fmaxf(v, __shfl_xor(v, 32));
  return v;
}
__device__ __forceinline__ float row_sum4(float v) {
  v += __shfl_xor(v, 16);
  v += __shfl_xor(v, 32);
  return v;
}

// ---- LDS accesses the compiler does not see as memory operations. It orders every LDS access
// it knows about after ALL outstanding direct-to-LDS loads (a full vmcnt(0)), which would
// serialise the ring; these are issued by hand and completed by lds_wait().
template <int OFFSET>
__device__ __forceinline__ int4v lds_read_b128(unsigned byteAddr) {
  int4v v;
  asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(v) : "v"(byteAddr), "n"(OFFSET) : "memory");
  return v;
}
template <int OFFSET0, int OFFSET1>  // offsets in dwords, 0..255
__device__ __forceinline__ int2v lds_read2_b32(unsigned byteAddr) {
  int2v v;
  asm volatile("ds_read2_b32 %0, %1 offset0:%2 offset1:%3"
               : "=v"(v)
               : "v"(byteAddr), "n"(OFFSET0), "n"(OFFSET1)
               : "memory");
  return v;
}
// 4 x 16 bit per lane, transposed inside each group of 16 lanes: lane 4e+x of a group addresses
// elements 4x..4x+3 of row e of a 4 x 16 matrix of 16-bit values and receives column 4e+x.
template <int OFFSET>
__device__ __forceinline__ short4v lds_read_tr16_b64(unsigned byteAddr) {
  short4v v;
  asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2"
               : "=v"(v)
               : "v"(byteAddr), "n"(OFFSET)
               : "memory");
  return v;
}
__device__ __forceinline__ void lds_wait() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }
template <typename T>
__device__ __forceinline__ void pin(T& v) {
  asm volatile("" : "+v"(v));
}

// s_waitcnt vmcnt(N) only (expcnt / lgkmcnt unconstrained), N <= 63
template <int N>
__device__ __forceinline__ void vm_wait() {
  static_assert(N >= 0 && N <= 63, "vmcnt is a 6-bit counter");
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_waitcnt(0x0F70 | (N & 15) | ((N >> 4) << 14));
  __builtin_amdgcn_sched_barrier(0);
}

// ---- geometry of the per-wave LDS ring
// D: head dimension, any multiple of 32 up to 256 (the reference takes embeddingDim at run time,
// src/F3S_kernel.cu:601-604,1424,1522). A tile is the 32 rows of a pair, D elements each, one behind the
// other: a gather instruction's 64 lanes fetch 64 chunks of 16 bytes that follow each other in it. At
// the powers of two those are whole rows. At 96, 160, 192 and 224 a row may begin in one instruction and
// end in the next; the ring holds no unused bytes and every lane of every gather works: 6, 10, 12, 14
// instructions a tile. Rows at the pitch of the next power of two, the lanes beyond the row idle, need 8, 16, 16,
// 16 and rings a third larger. What bounds such calls is the vector memory path, in instructions as well as
// lines; us a call, that pitch -> rows one behind the other (blocks a window in brackets):
//   sliced, 50 000 nodes (109)             d =  96 165 -> 154, 160 328 -> 255, 192 347 -> 280, 224 390 -> 363
//   sliced, 233 000 nodes, bf16 (188)      1352 -> 1324, 2611 -> 2371, 2804 -> 2577, 3565 -> 3436
//   mixed, R-MAT 100 000 nodes (22)        98.5 -> 96.0, 167 -> 151, 173 -> 158, 203 -> 200
//   mixed, 40 000 nodes (39)               73.8 -> 70.8, 115 -> 103, 120 -> 111, 146 -> 140
//   windows, 20 000 nodes, bf16 (6)        27.6 -> 27.1, 39.8 -> 37.2, 42.0 -> 39.3, 45.0 -> 43.3
//   16x8 blocks, R-MAT 100 000 nodes (12)  83.9 -> 81.9, 139 -> 122
// (More waves in what the smaller rings leave free, units in workgroups of one or two waves: sliced calls at
// d = 96 1 to 2 % faster or slower, at 160 up to 14 % slower: the rows of more units at a time
// do not stay in the L2s.)
// STAGES: pairs of the ring in flight per wave (the kernels choose: two stages where a wave is alone
// with a long run of blocks, one stage and more waves where runs are short and what has to be
// hidden is the chain of loads in front of the first gather).
template <int D, int STAGES>
struct Geo {
  static_assert(D % 32 == 0 && D >= 32 && D <= 256, "head dimension: a multiple of 32 up to 256");
  static constexpr int T = D / 16;         // output tiles
  static constexpr int KS = D / 32;        // k-steps of the score product
  static constexpr int TG = D / 16;        // gather instructions per 32-row tile
  static constexpr int ROW = D * 2;        // bytes of a K / V row, in memory and in LDS
  static constexpr int CPR = D / 8;        // 16-byte chunks per row
  static constexpr int TILE = 32 * ROW;    // K (or V) rows of one pair
  static constexpr int STAGE = 2 * TILE;   // one pair: K tile, then V tile
  static constexpr int NS = STAGES;  // stages of the ring
  static constexpr int META_SLOT = 768;    // metadata of four steps: 512 B ids, 256 B bitmaps
  static constexpr int META = 2 * META_SLOT;
  static constexpr int WAVE_BYTES = NS * STAGE + META;
};

// rows that straddle gather instructions (above), and the number of rows after which a row starts where
// an instruction does again: that many rows, and instructions, later a lane's chunk has the same place in its row
template <int D>
constexpr bool straddling() {
  return (D & (D - 1)) != 0;
}
template <int D>
constexpr int rows_of_period() {
  return D % 64 == 0 ? 8 : 16;
}
template <int D>
constexpr int gathers_of_period() {
  return rows_of_period<D>() * D / 512;
}
// Row of the tile that lane `lane` fetches a chunk of in gather instruction i, and the chunk's place in it.
template <int D>
__device__ __forceinline__ constexpr int gather_row(int i, int lane) {
  return (i * 64 + lane) / (D / 8);
}
template <int D>
__device__ __forceinline__ constexpr int gather_pos(int i, int lane) {
  return (i * 64 + lane) % (D / 8);
}
// Which of the pair's 32 key slots lies in which row of the tile, and the inverse. Powers of two: such that
// the slots a lane fetches are groups of four consecutive dwords of the metadata (one 16-byte LDS read
// yields four of its row ids); D >= 64: slot = 4 * (rho + RPI * (i / 4)) + i % 4 in lane-row rho of instruction
// i, RPI rows an instruction. Straddling rows: slot by slot.
template <int D>
__device__ __forceinline__ constexpr int slot_of_row(int row) {
  if constexpr (straddling<D>()) return row;
  if constexpr (D == 32) return 4 * ((row & 15) >> 1) + 2 * (row >> 4) + (row & 1);
  constexpr int RPI = 512 / D;
  const int i = row / RPI, rho = row % RPI;
  return 4 * (rho + RPI * (i >> 2)) + (i & 3);
}
template <int D>
__device__ __forceinline__ constexpr int lds_row_of(int s) {
  if constexpr (straddling<D>()) return s;
  if constexpr (D == 32) return ((s & 3) >> 1) * 16 + 2 * (s >> 2) + (s & 1);
  constexpr int RPI = 512 / D;
  const int rho = (s >> 2) & (RPI - 1);
  const int q = (s >> 2) / RPI;
  return ((s & 3) + 4 * q) * RPI + rho;
}
// XOR applied to the 16-byte chunk index of slot s inside its LDS row: the K tile is read with
// one 16-byte read per lane (16 consecutive slots by 4 chunks), the V tile with transposing
// 8-byte reads (8 consecutive slots by 32 bytes in each half of the lanes); each pattern wants its 256
// bytes on different banks.
template <int D>
__device__ __forceinline__ constexpr int swz_k(int s) {
  const int c = s & 15;
  if constexpr (D == 32) return ((c >> 1) & 1) | ((((c >> 2) ^ (c >> 3)) & 1) << 1);
  if constexpr (D == 64) return (c & 3) | ((((c >> 2) ^ (c >> 3)) & 1) << 2);
  if constexpr (D == 192) return c >> 1;  // every other row begins on the same bank
  if constexpr (straddling<D>()) return c >> 2;  // every fourth row
  return c;
}
template <int D>
__device__ __forceinline__ constexpr int swz_v(int s) {
  if constexpr (D == 32) return ((s >> 1) & 1) << 1;
  if constexpr (D == 64) return (s & 3) << 1;
  if constexpr (D == 192) return ((s >> 1) & 3) << 1;
  if constexpr (straddling<D>()) return ((s >> 2) & 1) << 1;
  return (s & 7) << 1;
}
// The chunk a lane fetches in gather instruction i depends on i only through i % NK (K) and
// i % NV (V), so that many byte offsets are kept per lane.
template <int D>
constexpr int distinct_k_offsets() {
  if (D == 192) return 2 * gathers_of_period<D>();
  if (straddling<D>()) return gathers_of_period<D>();
  return D == 32 ? 2 : D == 256 ? 8 : 4;
}
template <int D>
constexpr int distinct_v_offsets() {
  if (straddling<D>()) return gathers_of_period<D>();
  return D == 32 ? 2 : 4;
}
// Likewise the operand reads: k-step i reads at address i % KA plus i / KA of its stride, tile j at j % VA
// plus j / VA. KA k-steps (64 bytes each) and VA tiles (32 bytes each) span the chunks an XOR moves within.
template <int D>
constexpr int distinct_k_reads() {
  if (D == 192) return 2;
  if (straddling<D>()) return 1;
  return D / 32 < 4 ? D / 32 : 4;
}
template <int D>
constexpr int distinct_v_reads() {
  if (D == 192) return 4;
  if (straddling<D>()) return 2;
  return D / 16 < 8 ? (D == 32 ? 2 : 4) : 8;
}
template <int D>
constexpr bool gather_offsets_periodic() {
  for (int i = 0; i < D / 16; i++)
    for (int lane = 0; lane < 64; lane++) {
      const int s = slot_of_row<D>(gather_row<D>(i, lane));
      const int ik = i % distinct_k_offsets<D>(), iv = i % distinct_v_offsets<D>();
      if (gather_pos<D>(i, lane) != gather_pos<D>(ik, lane) || gather_pos<D>(i, lane) != gather_pos<D>(iv, lane))
        return false;
      if (swz_k<D>(s) != swz_k<D>(slot_of_row<D>(gather_row<D>(ik, lane)))) return false;
      if (swz_v<D>(s) != swz_v<D>(slot_of_row<D>(gather_row<D>(iv, lane)))) return false;
      if ((gather_pos<D>(i, lane) ^ swz_k<D>(s)) >= D / 8 || (gather_pos<D>(i, lane) ^ swz_v<D>(s)) >= D / 8)
        return false;
    }
  return true;
}
// the two maps of rows and slots are inverse to each other, and the second half of a tile lies a fixed
// distance behind the first
template <int D>
constexpr bool slot_maps_consistent() {
  for (int row = 0; row < 32; row++) {
    const int s = slot_of_row<D>(row);
    if (s < 0 || s >= 32 || lds_row_of<D>(s) != row) return false;
  }
  for (int s = 0; s < 16; s++)
    if (lds_row_of<D>(s + 16) - lds_row_of<D>(s) != lds_row_of<D>(16) - lds_row_of<D>(0) ||
        swz_k<D>(s + 16) != swz_k<D>(s) || swz_v<D>(s + 16) != swz_v<D>(s))
      return false;
  return true;
}
// what the lanes of one group (K: 16 slots, V: 8 slots by two chunks) read lies in different chunks of the
// 256 bytes that the banks span, and each k-step and tile where its address and stride say
template <int D>
constexpr bool operand_reads_consistent() {
  constexpr int KA = distinct_k_reads<D>(), VA = distinct_v_reads<D>(), C = D / 8;
  for (int i = 0; i < D / 32; i++)
    for (int g = 0; g < 4; g++) {
      unsigned banks = 0;
      for (int s = 0; s < 16; s++) {
        const int chunk = (4 * i + g) ^ swz_k<D>(s);
        banks |= 1u << ((lds_row_of<D>(s) * C + chunk) & 15);
        if (chunk >= C || chunk != ((4 * (i % KA) + g) ^ swz_k<D>(s)) + i / KA * KA * 4) return false;
      }
      if (banks != 0xFFFFu) return false;
    }
  for (int j = 0; j < D / 16; j++)
    for (int s0 = 0; s0 < 16; s0 += 8) {
      unsigned banks = 0;
      for (int s = s0; s < s0 + 8; s++)
        for (int x = 0; x < 2; x++) {
          const int chunk = (2 * j + x) ^ swz_v<D>(s);
          banks |= 1u << ((lds_row_of<D>(s) * C + chunk) & 15);
          if (chunk >= C || chunk != ((2 * (j % VA) + x) ^ swz_v<D>(s)) + j / VA * VA * 2) return false;
        }
      if (banks != 0xFFFFu) return false;
    }
  return true;
}
template <int D>
constexpr bool maps_consistent() {
  return gather_offsets_periodic<D>() && slot_maps_consistent<D>() && operand_reads_consistent<D>();
}
static_assert(maps_consistent<32>() && maps_consistent<64>() && maps_consistent<96>() &&
                  maps_consistent<128>() && maps_consistent<160>() && maps_consistent<192>() &&
                  maps_consistent<224>() && maps_consistent<256>(),
              "tile maps");

// Problem description shared by every kernel.
template <typename ET>
struct Problem {
  const int32_t* __restrict__ sparseAToXidx;
  const uint8_t* __restrict__ bitmapBytes;
  const ET* __restrict__ Q;
  const ET* __restrict__ K;
  const ET* __restrict__ V;
  int N;
  float scaleLog2;   // log2(e) / scalingFactor (1.0 without softmax)
  int pitchIn;       // row pitch of K/V in elements (D for the single-head layout)
  int pitchQ;        // row pitch of Q in elements
  int64_t nTcb;      // TC blocks in sparseAToXidx / bitmapBytes (bounds of the metadata loads)
  float* __restrict__ sddmm;  // 16x8 structure only: masked unscaled scores, or null
};

// ET: _Float16 or __bf16. HEADS: pitched rows (row offset by 24-bit multiply). W8: the structure
// comes from preprocessing with 8-column blocks; two consecutive 16x8 blocks are laid out like
// one 16x16 block, block indices and counts below are then in 16x8 blocks. WIDE: K or V spans
// 4 GiB or more (or a pitched layout exceeds the 24-bit multiply): row offsets in 64 bits.
// NH = 2: the D = 64 features of a row are two heads of 32 next to each other. Rows are gathered, and
// operands read, as one head's of 64; scores, softmax (m, l) and the two halves of O are each head's
// own, with the arithmetic of a D = 32 pipeline in the same order (bit-identical). Two 32-wide heads one
// by one ask for every 128-byte line twice, half of it each, and run the chain of ids, bitmaps and rows
// twice: that chain is most of a short window's time, and the vector memory path what bounds long ones
// (bf16: 100k-node community layer of 6 blocks a window, 8 x 32 111.5 -> 97.1 us a call; R-MAT 150 000
// nodes, 8 x 32 365 -> 260 us, power-law 50 000 nodes, 382 blocks, 8 x 32 1490 -> 1068 us; both with
// head groups dealt to the XCDs, which by itself made the former 295 us).
template <typename ET, int D, bool SOFTMAX, bool HEADS, bool W8, int STAGES, bool WIDE = false,
          int NH = 1>
struct PairPipeline {
  static_assert(NH == 1 || (NH == 2 && D == 64 && HEADS && !W8), "two heads of 32");
  typedef Geo<D, STAGES> G;
  typedef typename Vec<ET, 8>::type half8;
  static constexpr int T = G::T;
  static constexpr int KS = G::KS;
  static constexpr int NS = G::NS;
  static constexpr int TG = G::TG;
  static constexpr int NK = distinct_k_offsets<D>();
  static constexpr int NV = distinct_v_offsets<D>();
  static constexpr int KA = distinct_k_reads<D>();
  static constexpr int VA = distinct_v_reads<D>();
  static constexpr int NI = straddling<D>() ? gathers_of_period<D>() : 1;
  static constexpr int BPS = W8 ? 4 : 2;  // blocks of the structure per step
  static constexpr bool SPLIT_P = sizeof(ET) == 2 && !__is_same(ET, _Float16);  // bf16

  // running state
  float m[NH], l[NH];
  float4v o[T];  // NH tiles' worth of each head, one after the other

  // loop-invariant per-lane values
  half8 qf[KS];
  unsigned ring;        // LDS byte address of this wave's ring
  unsigned metaBase;    // LDS byte address of this wave's two metadata slots
  unsigned kReadAddr[KA];  // K tile: slot c, chunk 4i + g (swizzled)
  unsigned vReadAddr[VA];  // V tile: transposing read of tiles 0.., first key half
  unsigned idReadAddr[NI];  // metadata: this lane's row ids
  unsigned maskReadAddr;   // metadata: the bitmap dword with this lane's bits of block A
  int keepPos[4];          // bit position of element i in that dword
  uint32_t gatherOffK[NK], gatherOffV[NV];  // byte offset inside the row this lane fetches
  int lane, g, c;

  __device__ __forceinline__ void init(const Problem<ET>& pb, int w, unsigned ringAddr, int head) {
    lane = threadIdx.x & 63;
    g = lane >> 4;
    c = lane & 15;
    ring = ringAddr;
    metaBase = ringAddr + NS * G::STAGE;
#pragma unroll
    for (int h = 0; h < NH; h++) m[h] = l[h] = 0.0f;
#pragma unroll
    for (int j = 0; j < T; j++) o[j] = float4v{0.f, 0.f, 0.f, 0.f};
    {
      const int4v zero16 = {0, 0, 0, 0};
      const int64_t qrow = (int64_t)w * 16 + c;
      if (qrow < pb.N) {
        const half8* qp =
            reinterpret_cast<const half8*>(pb.Q + qrow * pb.pitchQ + (HEADS ? head * D : 0)) + g;
#pragma unroll
        for (int i = 0; i < KS; i++) qf[i] = qp[4 * i];
      } else {
#pragma unroll
        for (int i = 0; i < KS; i++) qf[i] = __builtin_bit_cast(half8, zero16);
      }
    }
    // gather: in instruction i this lane fetches chunk gather_pos ^ swizzle of the slot in row gather_row;
    // the chunk lands at ring + i * 1024 + lane * 16
#pragma unroll
    for (int i = 0; i < TG; i++) {
      const int s = slot_of_row<D>(gather_row<D>(i, lane)), pos = gather_pos<D>(i, lane);
      if (i < NK) gatherOffK[i] = (uint32_t)((pos ^ swz_k<D>(s)) * 16 + (HEADS ? head * D * 2 : 0));
      if (i < NV) gatherOffV[i] = (uint32_t)((pos ^ swz_v<D>(s)) * 16 + (HEADS ? head * D * 2 : 0));
    }
    // score product: lane (g, c) reads, for block b and k-step i, chunk 4i + g of slot 16b + c
#pragma unroll
    for (int i = 0; i < KA; i++)
      kReadAddr[i] = ring + lds_row_of<D>(c) * G::ROW + (((4 * i + g) ^ swz_k<D>(c)) * 16);
    // P V product: lane (g, c = 4e + x) addresses slot 16h + 4g + e, columns 16j + 4x .. +3:
    // chunk 2j + x/2 (swizzled), byte (x % 2) * 8 inside it. h = 1 is a fixed distance away.
    {
      const int e = c >> 2, x = c & 3;
      const int s = 4 * g + e;
#pragma unroll
      for (int j = 0; j < VA; j++)
        vReadAddr[j] = ring + G::TILE + lds_row_of<D>(s) * G::ROW +
                       (((2 * j + (x >> 1)) ^ swz_v<D>(s)) * 16) + (x & 1) * 8;
    }
    // metadata slot: ids of step q at q * 128, bitmaps at 512 + q * 64
#pragma unroll
    for (int i = 0; i < NI; i++) idReadAddr[i] = metaBase + slot_of_row<D>(gather_row<D>(i, lane)) * 4;
    const int maskByte = ((g >> 1) * 2 + (c >> 3)) * 8 + 7 - (c & 7);
    maskReadAddr = metaBase + 512 + (maskByte >> 2) * 4;
#pragma unroll
    for (int i = 0; i < 4; i++) keepPos[i] = 8 * (maskByte & 3) + 4 * (1 - (g & 1)) + 3 - i;
  }

  // ---- loads -------------------------------------------------------------------------------
  // Metadata of steps 4k .. 4k+3 of the run [t0, t1) into metadata slot k & 1. Lanes 0..31: the
  // 128 column ids (16 bytes each), lanes 32..47: the 64 bitmap dwords. Blocks past the end of
  // the run are folded onto its last block (the loads stay in bounds; their bits are never used).
  __device__ __forceinline__ void issue_meta(const Problem<ET>& pb, int t0, int t1, int k) {
    constexpr int IDS_PER_BLOCK = W8 ? 8 : 16;      // ids of one block of the structure
    constexpr int BM_BYTES = W8 ? 16 : 32;          // bitmap bytes of one block
    const int64_t first = (int64_t)t0 + (int64_t)k * 4 * BPS;
    const char* src;
    if (lane < 32) {
      int64_t blk = first + (lane * 4) / IDS_PER_BLOCK;
      const int within = (lane * 4) % IDS_PER_BLOCK;
      if (blk >= t1) blk = t1 - 1;
      src = reinterpret_cast<const char*>(pb.sparseAToXidx) + (blk * IDS_PER_BLOCK + within) * 4;
    } else {
      const int b = (lane - 32) & 15;  // lanes 48..63 fetch nothing
      int64_t blk = first + (b * 16) / BM_BYTES;
      const int within = (b * 16) % BM_BYTES;
      if (blk >= t1) blk = t1 - 1;
      src = reinterpret_cast<const char*>(pb.bitmapBytes) + blk * BM_BYTES + within;
    }
    F3S_LDS int4v* dst =
        (F3S_LDS int4v*)(uintptr_t)(uniform((int)metaBase) + (k & 1) * G::META_SLOT);
    if (lane < 48)
      __builtin_amdgcn_global_load_lds(reinterpret_cast<const int4v*>(src), dst, 16, 0, 0);
  }

  // K and V rows of step p into ring stage STAGE_IDX = p % NS, row ids from metadata. The step's
  // position in its metadata slot is the compile-time Q4 plus the run-time q (one of them 0).
  template <int STAGE_IDX, int Q4>
  __device__ __forceinline__ void issue_gather(const Problem<ET>& pb, int metaSlot, int q) {
    int rows[TG];
    const unsigned at = (unsigned)(metaSlot * G::META_SLOT + q * 128);
    if constexpr (straddling<D>()) {
      // slot i of this lane, and the ones as many rows further as a period has
      constexpr int P = rows_of_period<D>(), HALVES = 32 / P / 2;
      int2v r[NI][HALVES];
#pragma unroll
      for (int i = 0; i < NI; i++) {
        r[i][0] = lds_read2_b32<Q4 * 32, Q4 * 32 + P>(idReadAddr[i] + at);
        if constexpr (HALVES == 2)
          r[i][1] = lds_read2_b32<Q4 * 32 + 2 * P, Q4 * 32 + 3 * P>(idReadAddr[i] + at);
      }
      lds_wait();
#pragma unroll
      for (int i = 0; i < TG; i++) rows[i] = r[i % NI][i / NI / 2][i / NI % 2];
    } else if constexpr (D == 32) {
      const int2v r = lds_read2_b32<Q4 * 32, Q4 * 32 + 2>(idReadAddr[0] + at);
      lds_wait();
      rows[0] = r[0];
      rows[1] = r[1];
    } else {
      // groups of four consecutive dwords; group q of four slots starts 64 / CPR * 4 slots after group q - 1
      const unsigned ida = idReadAddr[0] + at;
      constexpr int RPI = 64 / G::CPR;
      int4v r[TG / 4];
      r[0] = lds_read_b128<Q4 * 128>(ida);
      if constexpr (TG >= 8) r[1] = lds_read_b128<Q4 * 128 + 1 * RPI * 16>(ida);
      if constexpr (TG >= 16) {
        r[2] = lds_read_b128<Q4 * 128 + 2 * RPI * 16>(ida);
        r[3] = lds_read_b128<Q4 * 128 + 3 * RPI * 16>(ida);
      }
      lds_wait();
#pragma unroll
      for (int q = 0; q < TG / 4; q++)
#pragma unroll
        for (int i = 0; i < 4; i++) rows[4 * q + i] = r[q][i];
    }
    const char* Kb = reinterpret_cast<const char*>(pb.K);
    const char* Vb = reinterpret_cast<const char*>(pb.V);
    const uint32_t rowBytes = HEADS ? (uint32_t)pb.pitchIn * 2u : (uint32_t)G::ROW;
    const int ringU = uniform((int)ring);
#pragma unroll
    for (int i = 0; i < TG; i++) {
      pin(rows[i]);
#ifdef F3S_PROBE_ROWMASK
      rows[i] &= F3S_PROBE_ROWMASK;
#endif
    }
    // one gather instruction: 64 lanes x 16 bytes of K (V) rows into 1 KiB of the stage
    auto gather = [&](const char* src, int ldsOffset) {
      F3S_LDS int4v* dst = (F3S_LDS int4v*)(uintptr_t)(ringU + ldsOffset);
      __builtin_amdgcn_global_load_lds(reinterpret_cast<const int4v*>(src), dst, 16, 0, 0);
    };
    if constexpr (WIDE) {
      // the reference indexes rows with int64_t (src/F3S_kernel.cu:1422-1423)
#pragma unroll
      for (int i = 0; i < TG; i++)
        gather(Kb + ((uint64_t)(uint32_t)rows[i] * rowBytes + gatherOffK[i % NK]),
               STAGE_IDX * G::STAGE + i * 1024);
#pragma unroll
      for (int i = 0; i < TG; i++)
        gather(Vb + ((uint64_t)(uint32_t)rows[i] * rowBytes + gatherOffV[i % NV]),
               STAGE_IDX * G::STAGE + G::TILE + i * 1024);
    } else {
#pragma unroll
      for (int i = 0; i < TG; i++) {
        const uint32_t ro = HEADS ? __umul24((uint32_t)rows[i], rowBytes)
                                  : (uint32_t)rows[i] * rowBytes;
        gather(Kb + (ro + gatherOffK[i % NK]), STAGE_IDX * G::STAGE + i * 1024);
      }
#pragma unroll
      for (int i = 0; i < TG; i++) {
        const uint32_t ro = HEADS ? __umul24((uint32_t)rows[i], rowBytes)
                                  : (uint32_t)rows[i] * rowBytes;
        gather(Vb + (ro + gatherOffV[i % NV]), STAGE_IDX * G::STAGE + G::TILE + i * 1024);
      }
    }
  }

  // ---- one step ------------------------------------------------------------------------------
  struct Operands {
    int4v k[2][KS];
    short4v v[T][2];
    int2v words;
  };

  template <int STAGE_IDX, int Q4>
  __device__ __forceinline__ void read_operands(int metaSlot, int q, Operands& op) {
    constexpr int SO = STAGE_IDX * G::STAGE;
    read_k_step<SO, 0>(op);
    read_v_tile<SO, 0>(op);
    op.words = lds_read2_b32<Q4 * 16, Q4 * 16 + 8>(
        maskReadAddr + (unsigned)(metaSlot * G::META_SLOT + q * 64));
  }
  template <int SO, int I>
  __device__ __forceinline__ void read_k_step(Operands& op) {
    constexpr int OFF = SO + I / KA * KA * 64;
    op.k[0][I] = lds_read_b128<OFF>(kReadAddr[I % KA]);
    op.k[1][I] = lds_read_b128<OFF + half_distance()>(kReadAddr[I % KA]);
    if constexpr (I + 1 < KS) read_k_step<SO, I + 1>(op);
  }
  template <int SO, int J>
  __device__ __forceinline__ void read_v_tile(Operands& op) {
    constexpr int OFF = SO + J / VA * VA * 32;
    op.v[J][0] = lds_read_tr16_b64<OFF>(vReadAddr[J % VA]);
    op.v[J][1] = lds_read_tr16_b64<OFF + half_distance()>(vReadAddr[J % VA]);
    if constexpr (J + 1 < T) read_v_tile<SO, J + 1>(op);
  }
  // LDS distance between the rows of slot s and slot s + 16 of a tile
  static __device__ __forceinline__ constexpr int half_distance() {
    return (lds_row_of<D>(16) - lds_row_of<D>(0)) * G::ROW;
  }

  __device__ __forceinline__ void consume(Operands& op) {
#pragma unroll
    for (int b = 0; b < 2; b++)
#pragma unroll
      for (int i = 0; i < KS; i++) pin(op.k[b][i]);
#pragma unroll
    for (int j = 0; j < T; j++) {
      pin(op.v[j][0]);
      pin(op.v[j][1]);
    }
    pin(op.words);
  }

  // nValid: blocks of the structure that exist in this step (1..BPS); only the last step of a
  // run can have fewer than BPS.
  __device__ __forceinline__ void compute(const Problem<ET>& pb, Operands& op, int tFirst,
                                          int nValid) {
#pragma unroll
    for (int b = 0; b < 2; b++)
#pragma unroll
      for (int i = 0; i < KS; i++) pin(op.k[b][i]);
    float4v sA[NH], sB[NH];
#pragma unroll
    for (int h = 0; h < NH; h++) sA[h] = sB[h] = float4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < KS; i++) {
      constexpr int KH = KS / NH;  // k-steps of a head
      sA[i / KH] = mfma_16x16x32<ET>(__builtin_bit_cast(half8, op.k[0][i]), qf[i], sA[i / KH]);
      sB[i / KH] = mfma_16x16x32<ET>(__builtin_bit_cast(half8, op.k[1][i]), qf[i], sB[i / KH]);
    }
    pin(op.words);
    int wordA = op.words[0], wordB = op.words[1];
    if constexpr (W8) {
      // this lane's slots 4g..4g+3 belong to 16x8 block g/2 (A) resp. 2 + g/2 (B) of the step
      if ((g >> 1) >= nValid) wordA = 0;
      if (2 + (g >> 1) >= nValid) wordB = 0;
    } else {
      if (nValid < 2) wordB = 0;
    }
    int keep[8];
#pragma unroll
    for (int i = 0; i < 4; i++) {
      keep[i] = __builtin_amdgcn_sbfe(wordA, keepPos[i], 1);  // 0 or -1
      keep[4 + i] = __builtin_amdgcn_sbfe(wordB, keepPos[i], 1);
    }
#pragma unroll
    for (int j = 0; j < T; j++) {
      pin(op.v[j][0]);
      pin(op.v[j][1]);
    }
#pragma unroll
    for (int h = 0; h < NH; h++) one_head(pb, op, sA[h], sB[h], keep, h, tFirst, nValid);
  }

  // softmax and second product of head h
  __device__ __forceinline__ void one_head(const Problem<ET>& pb, Operands& op, const float4v& sA,
                                           const float4v& sB, const int (&keep)[8], int h, int tFirst,
                                           int nValid) {
    constexpr int TH = T / NH;  // output tiles of a head
    float s[8];
#pragma unroll
    for (int i = 0; i < 4; i++) {
      s[i] = sA[i];
      s[4 + i] = sB[i];
    }
    if constexpr (W8) {
      if (pb.sddmm) {
        // lane (g, c): row c, columns 4(g&1)..+3 of block tFirst + g/2 (A) and + 2 (B)
        float* dst = pb.sddmm + ((size_t)(tFirst + (g >> 1)) * 16 + c) * 8 + 4 * (g & 1);
        float4 a, b;
        a.x = __int_as_float(__float_as_int(s[0]) & keep[0]);
        a.y = __int_as_float(__float_as_int(s[1]) & keep[1]);
        a.z = __int_as_float(__float_as_int(s[2]) & keep[2]);
        a.w = __int_as_float(__float_as_int(s[3]) & keep[3]);
        b.x = __int_as_float(__float_as_int(s[4]) & keep[4]);
        b.y = __int_as_float(__float_as_int(s[5]) & keep[5]);
        b.z = __int_as_float(__float_as_int(s[6]) & keep[6]);
        b.w = __int_as_float(__float_as_int(s[7]) & keep[7]);
        if ((g >> 1) < nValid) store_out(dst, out_vec{a.x,a.y,a.z,a.w});
        if (2 + (g >> 1) < nValid) store_out(dst + 256, out_vec{b.x,b.y,b.z,b.w});
      }
    }
    float e[8];
    if constexpr (SOFTMAX) {
      // fast path: exponentials against the current maximum, masked ones cleared afterwards
      const float negM = -m[h];
      float sum = 0.0f;
#pragma unroll
      for (int i = 0; i < 8; i++) {
        const float ev = fast_exp2(fmaf(s[i], pb.scaleLog2, negM));
        e[i] = __int_as_float(__float_as_int(ev) & keep[i]);
        sum += e[i];
      }
      float zmin = fminf(fminf(fabsf(s[0]), fabsf(s[1])), fabsf(s[2]));
      zmin = fminf(fminf(zmin, fabsf(s[3])), fabsf(s[4]));
      zmin = fminf(fminf(zmin, fabsf(s[5])), fabsf(s[6]));
      zmin = fminf(zmin, fabsf(s[7]));
      // some lane saw a score far above its row's maximum (or a non-finite sum), or a score
      // that is exactly zero (masked or not): redo the step the careful way
      if (__builtin_amdgcn_ballot_w64(!(sum <= kLazyLimit) || zmin == 0.0f) != 0ull) {
        float sc[8];
        float mx = m[h];
#pragma unroll
        for (int i = 0; i < 8; i++) {
          sc[i] = __int_as_float(__float_as_int(s[i]) & keep[i]) * pb.scaleLog2;
          mx = fmaxf(mx, sc[i]);
        }
        mx = row_max4(mx);
        const float alpha = fast_exp2(m[h] - mx);
        m[h] = mx;
        sum = 0.0f;
#pragma unroll
        for (int i = 0; i < 8; i++) {
          e[i] = (sc[i] == 0.0f) ? 0.0f : fast_exp2(sc[i] - mx);
          sum += e[i];
        }
        l[h] *= alpha;
#pragma unroll
        for (int j = 0; j < TH; j++) o[h * TH + j] *= alpha;
      }
      l[h] += sum;
    } else {
#pragma unroll
      for (int i = 0; i < 8; i++) e[i] = __int_as_float(__float_as_int(s[i]) & keep[i]);
    }
    half8 pf;
#pragma unroll
    for (int i = 0; i < 8; i++) pf[i] = (ET)e[i];
    if constexpr (SPLIT_P) {
      half8 pt;
#pragma unroll
      for (int i = 0; i < 8; i++) pt[i] = (ET)(e[i] - (float)pf[i]);
#pragma unroll
      for (int j = h * TH; j < (h + 1) * TH; j++) {
        const half8 va = __builtin_bit_cast(
            half8, __builtin_shufflevector(op.v[j][0], op.v[j][1], 0, 1, 2, 3, 4, 5, 6, 7));
        o[j] = mfma_16x16x32<ET>(va, pf, o[j]);
        o[j] = mfma_16x16x32<ET>(va, pt, o[j]);
      }
    } else {
#pragma unroll
      for (int j = h * TH; j < (h + 1) * TH; j++) {
        const half8 va = __builtin_bit_cast(
            half8, __builtin_shufflevector(op.v[j][0], op.v[j][1], 0, 1, 2, 3, 4, 5, 6, 7));
        o[j] = mfma_16x16x32<ET>(va, pf, o[j]);
      }
    }
  }

  // ---- the loop over the run [t0, t1) of blocks of the structure ------------------------------
  // Ring discipline per step p (stage p % NS): wait until the step's K and V rows have landed
  // (vector loads complete in issue order), read all of its operands into registers, then reuse
  // the stage at once for step p + NS; the metadata of four steps at a time is requested at the
  // first of the four preceding steps.
  __device__ __forceinline__ void run(const Problem<ET>& pb, int t0, int t1) {
    const int nSteps = (t1 - t0 + BPS - 1) / BPS;
    if (nSteps <= 0) return;
    // prologue: metadata of the first four steps, then the first NS gathers
    issue_meta(pb, t0, t1, 0);
    vm_wait<0>();
    issue_gather<0, 0>(pb, 0, 0);
    if constexpr (NS == 2) {
      if (nSteps > 1) issue_gather<1, 1>(pb, 0, 0);
    }
    int p = 0;
    bool metaIssued = false;  // the last first-of-four step requested the next four's metadata
    // One step. NS == 2: STAGE_IDX = p % NS and Q4 = p % 4 are compile-time, the loop is unrolled
    // by four. NS == 1: Q4 is 0 and the position in the metadata slot a run-time offset (two
    // scalar instructions), so that the loop is one step long: unrolled by four, its four exits
    // cost the kernels around it 40 to 70 vector registers.
#define F3S_PIPE_STEP(STAGE_IDX, Q4)                                                           \
  {                                                                                            \
    constexpr int GQ4 = NS == 2 ? (Q4 + NS) % 4 : 0;                                           \
    const int q = NS == 2 ? Q4 : p & 3;                                                        \
    /* loads issued after this step's gather: the later stages' gathers and, if one of those  \
       steps opened a group of four, its metadata load */                                     \
    if constexpr (NS == 2) {                                                                   \
      if (p + 1 < nSteps) {                                                                    \
        if (Q4 == 1 && metaIssued) vm_wait<2 * TG + 1>(); else vm_wait<2 * TG>();              \
      } else {                                                                                 \
        vm_wait<0>();                                                                          \
      }                                                                                        \
    } else {                                                                                   \
      vm_wait<0>();                                                                            \
    }                                                                                          \
    Operands op;                                                                               \
    F3S_ABL_READ((read_operands<STAGE_IDX, Q4>((p >> 2) & 1, NS == 2 ? 0 : q, op)));           \
    lds_wait();                                                                                \
    __builtin_amdgcn_sched_barrier(0);                                                         \
    if (q == 0) {                                                                              \
      metaIssued = (p >> 2) + 1 <= (nSteps - 1) >> 2;                                          \
      if (metaIssued) issue_meta(pb, t0, t1, (p >> 2) + 1);                                    \
    }                                                                                          \
    if (p + NS < nSteps)                                                                       \
      F3S_ABL_GATHER((issue_gather<STAGE_IDX, GQ4>(pb, ((p + NS) >> 2) & 1,                    \
                                                   NS == 2 ? 0 : (p + NS) & 3)));              \
    __builtin_amdgcn_sched_barrier(0);                                                         \
    {                                                                                          \
      const int tFirst = t0 + p * BPS;                                                         \
      const int left = t1 - tFirst;                                                            \
      F3S_ABL_COMPUTE(compute(pb, op, tFirst, left < BPS ? left : BPS));                       \
    }                                                                                          \
    p++;                                                                                       \
    if (p >= nSteps) break;                                                                    \
  }
    while (true) {
      F3S_PIPE_STEP(0, 0)
      if constexpr (NS == 2) {
        F3S_PIPE_STEP(1, 1)
        F3S_PIPE_STEP(0, 2)
        F3S_PIPE_STEP(1, 3)
      }
    }
#undef F3S_PIPE_STEP
  }
};

// ---- epilogue of workgroups whose waves share a window. Every thread of the workgroup calls these three; the
// buffers lie at the start of smem, where the rings were.

// The waves' partial (m, l, O) into smem: m and l [NH][NWAVES][16], O [NWAVES][16][D + 4].
template <int D, int NWAVES, bool SOFTMAX, int NH, typename PipeT>
__device__ __forceinline__ void put_partials(const PipeT& pp, unsigned char* smem, int wave) {
  int lane = threadIdx.x & 63;
  pin(lane);  // nothing below is computed in front of the caller's loop and kept in registers
  const int g = lane >> 4, c = lane & 15;
  __syncthreads();
  float* sM = reinterpret_cast<float*>(smem);
  float* sL = sM + NH * NWAVES * 16;
  float* sO = sL + NH * NWAVES * 16;
#pragma unroll
  for (int h = 0; h < NH; h++) {
    float l = pp.l[h];
    if constexpr (SOFTMAX) l = row_sum4(l);
    if (g == 0) {
      sM[(h * NWAVES + wave) * 16 + c] = pp.m[h];
      sL[(h * NWAVES + wave) * 16 + c] = l;
    }
  }
#pragma unroll
  for (int j = 0; j < D / 16; j++)
    *reinterpret_cast<float4v*>(&sO[(wave * 16 + c) * (D + 4) + 16 * j + 4 * g]) = pp.o[j];
  __syncthreads();
}

// The window's rows (16 bytes of a row per element, dealt to the threads) from the partials of four
// waves, first .. first + 3: log-sum-exp, not yet divided by l.
template <int D, int NWAVES, bool SOFTMAX, int NH>
struct MergedRows {
  static constexpr int VEC_PER_ROW = D / 4, THREADS = NWAVES * 64;
  static constexpr int N = (16 * VEC_PER_ROW + THREADS - 1) / THREADS;  // elements of a thread
  float4v acc[N];
  float m[N], l[N];
  __device__ __forceinline__ static bool has(int tid, int i) {
    return 16 * VEC_PER_ROW % THREADS == 0 || i * THREADS + tid < 16 * VEC_PER_ROW;
  }
  __device__ __forceinline__ void merge(const unsigned char* smem, int first) {
    int tid = threadIdx.x;
    pin(tid);
    const float* sM = reinterpret_cast<const float*>(smem);
    const float* sL = sM + NH * NWAVES * 16;
    const float* sO = sL + NH * NWAVES * 16;
#pragma unroll
    for (int i = 0; i < N; i++) {
      if (!has(tid, i)) continue;
      const int q = (i * THREADS + tid) / VEC_PER_ROW, cv = (i * THREADS + tid) % VEC_PER_ROW;
      const int h = NH > 1 ? cv / (VEC_PER_ROW / NH) : 0;
      const float* mOf = sM + (h * NWAVES + first) * 16 + q;
      const float* lOf = sL + (h * NWAVES + first) * 16 + q;
      const float* oOf = sO + (first * 16 + q) * (D + 4) + cv * 4;
      acc[i] = float4v{0.f, 0.f, 0.f, 0.f};
      m[i] = mOf[0];
      l[i] = 0.0f;
      if constexpr (SOFTMAX) {
#pragma unroll
        for (int v = 1; v < 4; v++) m[i] = fmaxf(m[i], mOf[v * 16]);
      }
#pragma unroll
      for (int v = 0; v < 4; v++) {
        const float4v o = *reinterpret_cast<const float4v*>(oOf + v * 16 * (D + 4));
        if constexpr (SOFTMAX) {
          const float f = fast_exp2(mOf[v * 16] - m[i]);
          l[i] = fmaf(f, lOf[v * 16], l[i]);
#pragma unroll
          for (int e = 0; e < 4; e++) acc[i][e] = fmaf(f, o[e], acc[i][e]);
        } else {
          acc[i] += o;
        }
      }
    }
  }
  __device__ __forceinline__ void add(const MergedRows& b) {
#pragma unroll
    for (int i = 0; i < N; i++) {
      if constexpr (SOFTMAX) {
        const float both = fmaxf(m[i], b.m[i]);
        const float fa = fast_exp2(m[i] - both), fb = fast_exp2(b.m[i] - both);
        m[i] = both;
        l[i] = fmaf(fb, b.l[i], fa * l[i]);
#pragma unroll
        for (int e = 0; e < 4; e++) acc[i][e] = fmaf(fb, b.acc[i][e], fa * acc[i][e]);
      } else {
        acc[i] += b.acc[i];
      }
    }
  }
  // out points at the first column, rows are pitchOut floats apart
  __device__ __forceinline__ void store(int w, int rows, float* __restrict__ out, int pitchOut) const {
    int tid = threadIdx.x;
    pin(tid);
#pragma unroll
    for (int i = 0; i < N; i++) {
      if (!has(tid, i)) continue;
      const int q = (i * THREADS + tid) / VEC_PER_ROW, cv = (i * THREADS + tid) % VEC_PER_ROW;
      const int64_t row = (int64_t)w * 16 + q;
      if (row >= rows) continue;
      float4v r = acc[i];
      if constexpr (SOFTMAX) {
        const float inv = (l[i] == 0.0f) ? 0.0f : 1.0f / l[i];
        r *= inv;
      }
      store_out(out + row * pitchOut + cv * 4, out_vec{r[0], r[1], r[2], r[3]});
    }
  }
};

}  // namespace pipe
}  // namespace f3s
