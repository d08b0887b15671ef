// Launchers of every attention entry point of the MI355X Fused3S library (gfx950): argument
// rules, the choice of schedule (workgroup per window, wave per short window, column-sliced
// units), and the hand-off to the kernels with 64-bit row offsets for K / V of 4 GiB and more.
// The kernel with one workgroup per window is f3s_window_kernel.h; this translation unit builds
// it with 32-bit row offsets.
#include <stdlib.h>
#include <string.h>

#include "f3s_common.h"
#include "f3s_window_kernel.h"

namespace f3s {

using pipe::kLog2e;
using window::HeadLayout;


// Whether a call goes to f3s_attention_mixed.hip. F3S_SHORT_WINDOWS=0 in the environment turns it off.
bool short_windows(const int32_t* windowOrder, int nRW, int64_t nTcb16, int d, int nHeads, bool w8) {
  const char* e = getenv("F3S_SHORT_WINDOWS");  // read per call, like every other switch
  if (e && strcmp(e, "0") == 0) return false;
  return mixed_windows_pay(windowOrder != nullptr, nRW, nTcb16, d, nHeads, w8);
}

// The column-sliced schedule (f3s_attention_units.hip: (window, column slice) units, every XCD
// on one slice at a time so that its K/V rows stay in that XCD's L2, plus a merge kernel) pays off
// on graphs with long windows: on the 233k-node benchmark graph (450 TC blocks per window) it
// takes 1.54 ms at d = 64 against 2.48 ms for the workgroup-per-window kernel, with 7.1 GB
// instead of 17.7 GB of traffic beyond L2.
// Short windows would be cut into units of one or two blocks; they keep the window kernel.
// Calls on small structures of narrow rows are over before their slices pay. What decides is how skewed the
// graph is, which neither the number of nodes nor of blocks says: the lines are for power-law and R-MAT graphs,
// whose hot rows stay in the L2s by themselves. Window against sliced, us; nodes, blocks a window:
// - one head, d = 64, 450 000 blocks. Below: power-law 35 000, 191 81 against 93; 50 000, 118 85 92; 70 000, 93
//   102 115; 100 000, 68 123 155; R-MAT 60 000, 94 111 155. Beyond, power-law graphs still lose by their
//   slices, but less and less (50 000, 148 101 107; 178 117 120; 203 131 130; 100 000, 103 182 188; 122 218 204),
//   and uniform graphs of more rows than an L2 has room for gain more than that, as they do below
//   (36 000, 193 89 99; 42 000, 147 97 95; 50 000, 129 122 102; 50 000, 148 132 112; 100 000, 91 255 202).
// - one head, d = 32, 260 000: power-law 35 000, 116 44 57; 50 000, 78 46 51; 50 000, 100 56 60; 70 000, 79 68
//   69; 100 000, 68 98 87; R-MAT 60 000, 78 71 78; 101 105 89; uniform 36 000, 99 41 47; 50 000, 71 56 49.
// - two and four heads of 64, 250 000 (bf16): power-law 35 000, 73 75 96 and 148 160; 103 95 106 and 204 205;
//   133 120 129 and 263 249; 50 000, 87 126 134 and 271 264; 70 000, 77 170 182 and 367 352; R-MAT 40 000, 105
//   107 183 and 218 255; uniform 36 000, 99 129 108 and 290 220.
// - pairs of 32-wide heads (bf16), 600 000 for one pair or two: power-law 50 000, 100 76 95 and 148 172; 178 133
//   149 and 263 278; 100 000, 94 165 200 and 336 358; 122 218 253 and 449 439 (fp16: 50 000, 178 123 126 and 246
//   231); R-MAT 120 000, 98 180 331 and 333 515; uniform 36 000, 147 87 101 and 173 171; 50 000, 129 134 121 and
//   267 216. 400 000 for four and eight: power-law 35 000, 133 272 291 and 629 611; 50 000, 100 320 335 and 736
//   719; 135 431 425 and 970 917; 178 563 537 and 1267 1150 (fp16, four pairs: 135 421 382; 178 552 478);
//   100 000, 68 524 574 and 1171 1287; 94 721 704 and 1590 1614; R-MAT 60 000, 123 414 474 and 948 955.
// Eight heads of 64 gain by their slices from the fewest blocks on (35 000, 73 348 347; 103 486 457; 50 000, 87
// 631 593; R-MAT 40 000, 105 505 493), and so do numbers of heads that leave an XCD several of them to gather
// (three to sixteen heads of 64, 35 000, 103: 3 212 177, 5 452 314, 6 433 334, 16 1081 829; six of 32, 50 000,
// 100 325 299; 135 459 370).
bool windows_suffice(int64_t nTcb, int d, int nHeads) {
  if (getenv("F3S_SCHEDULE") || getenv("F3S_SLICE_PHASES")) return false;  // asked for
  if (d > 64) return false;
  if (nHeads <= 1) return nTcb < (d <= 32 ? 260000 : 450000);
  if (d == 32 && !heads_in_pairs(d, nHeads)) return false;
  const int units = d == 32 ? nHeads / 2 : nHeads;
  if (units > head_groups(64, units)) return false;  // several to an XCD
  if (d == 32) return nTcb < (units <= 2 ? 600000 : 400000);
  return units <= 4 && nTcb < 250000;
}

// Whether a call that is given a workspace uses it, that is, takes the column-sliced schedule: the
// launchers below and the queries that callers allocate by ask this one function. nHeads = 0: the
// single-head layout; ldIn: row pitch of Q / K / V in elements.
// F3S_SCHEDULE=window / =sliced in the environment overrides the choice.
int attention_uses_workspace(int N, int64_t nTcb, int nHeads, int d, int dtype, int64_t ldIn) {
  const char* e = getenv("F3S_SCHEDULE");  // read per call
  const int forced = (e && strcmp(e, "sliced") == 0) ? 1 : (e && strcmp(e, "window") == 0) ? -1 : 0;
  if ((dtype != 0 && dtype != 1) || !head_dim_supported(d) || N <= 0) return 0;
  if (gather_needs_wide_offsets(N, ldIn * 2, nHeads > 0)) return 0;  // launch_window_wide's
  if (forced) return forced > 0;
  const int64_t nRW = ((int64_t)N + kWinRows - 1) / kWinRows;
  return nRW >= 2048 && nTcb >= 64 * nRW && !windows_suffice(nTcb, d, nHeads);
}

int launch_attention(const int32_t* rowWindowOffset, const int32_t* windowOrder,
                     const int32_t* sparseAToXidx, const uint64_t* bitmap, int N, int64_t nTcb,
                     int d, int dtype, const void* Q, const void* K, const void* V,
                     float scalingFactor, int applySoftmax, float* out,
                     unsigned long long* cuTimer, void* workspace, size_t wsBytes, int prepared,
                     hipStream_t stream) {
  if (dtype != 0 && dtype != 1)
    return fail(-3, "f3s_attention_fwd: dtype %d not supported (0 = fp16, 1 = bf16)", dtype);
  if (scalingFactor == 0.0f) return fail(-2, "f3s_attention_fwd: scalingFactor must be non-zero");
  if (!head_dim_supported(d))
    return fail(-2, "f3s_attention_fwd: head dim %d unsupported (a multiple of 32 up to 256)", d);
  // the reference divides unmasked scores by scalingFactor (src/F3S_kernel.cu:1666-1667);
  // exponentials are taken in base 2, so log2(e) is folded into the same multiplier
  const float scaleLog2 = applySoftmax ? kLog2e / scalingFactor : 1.0f;
  // K / V of 4 GiB and more: every window goes to the window kernel built with 64-bit row
  // offsets (the other schedules exist with 32-bit offsets only)
  if (gather_needs_wide_offsets(N, (int64_t)d * 2, false))
    return launch_window_wide(rowWindowOffset, windowOrder, sparseAToXidx, bitmap, N, d, dtype, Q,
                              K, V, scaleLog2, applySoftmax, out, cuTimer, 0, d, d, nTcb, stream);
  if (workspace && !cuTimer && attention_uses_workspace(N, nTcb, 0, d, dtype, d))
    return launch_attention_sliced(rowWindowOffset, windowOrder, sparseAToXidx, bitmap, N, d, dtype,
                                   Q, K, V, scaleLog2, applySoftmax, out, workspace, wsBytes,
                                   nTcb, 0, d, d, prepared ? 2 : 0, stream);
  const int nRWi = (N + kWinRows - 1) / kWinRows;
  // the timed form is the window kernel's, and from 16 blocks a window on so is the one that draws windows from a cursor
  const bool cursor = window::window_cursor_requested() && nTcb >= 16 * (int64_t)nRWi;
  if (!cuTimer && !cursor && short_windows(windowOrder, nRWi, nTcb, d, 0, false))
    return launch_attention_mixed(rowWindowOffset, windowOrder, sparseAToXidx, bitmap, N, d, dtype, Q, K, V,
                                  scaleLog2, applySoftmax, out, 0, d, d, nTcb, stream);
  const HeadLayout single = {0, d, d, nTcb};
  return dtype == 0 ? window::dispatch_d<_Float16, false>(rowWindowOffset, windowOrder, sparseAToXidx, bitmap, N,
                                           d, Q, K, V, scaleLog2, applySoftmax, out, cuTimer,
                                           single, stream)
                    : window::dispatch_d<__bf16, false>(rowWindowOffset, windowOrder, sparseAToXidx, bitmap, N, d,
                                         Q, K, V, scaleLog2, applySoftmax, out, cuTimer, single,
                                         stream);
}

// Builds the column-sliced schedule's index (slice boundaries) in `workspace` and marks it as
// belonging to these arrays, so that attention calls with the same arrays skip that step.
// nHeads = 0: the single-head layout.
int launch_attention_prepare(const int32_t* rowWindowOffset, const int32_t* sparseAToXidx, int N,
                             int64_t nTcb, int d, int nHeads, void* workspace, size_t wsBytes,
                             hipStream_t stream) {
  if (!head_dim_supported(d))
    return fail(-2, "f3s_attention_prepare: head dim %d unsupported (a multiple of 32 up to 256)",
                d);
  if (nHeads < 0 || nHeads > 1024)
    return fail(-2, "f3s_attention_prepare: nHeads %d out of range (0..1024)", nHeads);
  return launch_attention_sliced(rowWindowOffset, nullptr, sparseAToXidx, nullptr, N, d, 0,
                                 nullptr, nullptr, nullptr, 1.0f, 1, nullptr, workspace, wsBytes,
                                 nTcb, nHeads, nHeads * d, nHeads * d, 1, stream);
}

int launch_attention_tcb8(const int32_t* rowWindowOffset, const int32_t* windowOrder,
                          const int32_t* sparseAToXidx, const uint64_t* bitmap, int N, int d,
                          const void* Q, const void* K, const void* V, int applySoftmax,
                          float* out, float* sddmm, int64_t nTcb8, hipStream_t stream) {
  // this path has no score scaling (src/F3S_kernel.cu:709-735)
  const float scaleLog2 = applySoftmax ? kLog2e : 1.0f;
  if (gather_needs_wide_offsets(N, (int64_t)d * 2, false))
    return launch_tcb8_wide(rowWindowOffset, windowOrder, sparseAToXidx, bitmap, N, d, Q, K, V,
                            scaleLog2, applySoftmax, out, sddmm, nTcb8, stream);
  // (at d = 32 the window kernel is the faster one: R-MAT, 150 000 nodes, 15 blocks of 16 a window: 72 against 81 us)
  if (d > 32 && short_windows(windowOrder, (N + kWinRows - 1) / kWinRows, nTcb8 / 2, d, 0, true))
    return launch_tcb8_mixed(rowWindowOffset, windowOrder, sparseAToXidx, bitmap, N, d, Q, K, V, scaleLog2,
                             applySoftmax, out, sddmm, nTcb8, stream);
#define F3S_DISPATCH(DD)                                                                      \
  if (d == DD)                                                                                \
    return applySoftmax                                                                       \
               ? window::launch_tcb8<DD, true, false>(rowWindowOffset, windowOrder,           \
                                                      sparseAToXidx, bitmap, N, Q, K, V,      \
                                                      scaleLog2, out, sddmm, nTcb8, stream)   \
               : window::launch_tcb8<DD, false, false>(rowWindowOffset, windowOrder,          \
                                                       sparseAToXidx, bitmap, N, Q, K, V,     \
                                                       scaleLog2, out, sddmm, nTcb8, stream);
  F3S_FOR_EACH_HEAD_DIM(F3S_DISPATCH)
#undef F3S_DISPATCH
  return fail(-2, "f3s_attention_fwd_tcb8: head dim %d unsupported (a multiple of 32 up to 256)",
              d);
}

int launch_attention_heads(const int32_t* rowWindowOffset, const int32_t* windowOrder,
                           const int32_t* sparseAToXidx, const uint64_t* bitmap, int N,
                           int64_t nTcb, int nHeads, int d, int dtype, const void* Q, const void* K,
                           const void* V, int64_t ldIn, float scalingFactor, int applySoftmax,
                           float* out, int64_t ldOut, void* workspace, size_t wsBytes,
                           int prepared, hipStream_t stream) {
  if (dtype != 0 && dtype != 1)
    return fail(-3, "f3s_attention_fwd_heads: dtype %d not supported (0 = fp16, 1 = bf16)", dtype);
  if (scalingFactor == 0.0f)
    return fail(-2, "f3s_attention_fwd_heads: scalingFactor must be non-zero");
  if (nHeads < 1 || nHeads > 1024)
    return fail(-2, "f3s_attention_fwd_heads: nHeads %d out of range (1..1024)", nHeads);
  if (ldIn < (int64_t)nHeads * d || ldOut < (int64_t)nHeads * d)
    return fail(-2, "f3s_attention_fwd_heads: row pitches must be at least nHeads*d");
  if (ldIn % 8 != 0 || ldOut % 4 != 0)
    return fail(-2, "f3s_attention_fwd_heads: rows must stay 16-byte aligned (ldIn %% 8 == 0, "
                    "ldOut %% 4 == 0)");
  if (!head_dim_supported(d))
    return fail(-2, "f3s_attention_fwd_heads: head dim %d unsupported (a multiple of 32 up to 256)",
                d);
  if (ldIn >= ((int64_t)1 << 31) || ldOut >= ((int64_t)1 << 31))
    return fail(-2, "f3s_attention_fwd_heads: row pitches must be below 2^31 elements");
  const int64_t nRW = ((int64_t)N + kWinRows - 1) / kWinRows;
  if (nRW * nHeads >= ((int64_t)1 << 31))
    return fail(-2, "f3s_attention_fwd_heads: too many (window, head) workgroups");
  const float scaleLog2 = applySoftmax ? kLog2e / scalingFactor : 1.0f;
  if (gather_needs_wide_offsets(N, ldIn * 2, true))
    return launch_window_wide(rowWindowOffset, windowOrder, sparseAToXidx, bitmap, N, d, dtype, Q,
                              K, V, scaleLog2, applySoftmax, out, nullptr, nHeads, (int)ldIn,
                              (int)ldOut, nTcb, stream);
  if (workspace && attention_uses_workspace(N, nTcb, nHeads, d, dtype, ldIn))
    return launch_attention_sliced(rowWindowOffset, windowOrder, sparseAToXidx, bitmap, N, d, dtype,
                                   Q, K, V, scaleLog2, applySoftmax, out, workspace, wsBytes,
                                   nTcb, nHeads, (int)ldIn, (int)ldOut, prepared ? 2 : 0, stream);
  if (short_windows(windowOrder, (int)nRW, nTcb, d, nHeads, false))
    return launch_attention_mixed(rowWindowOffset, windowOrder, sparseAToXidx, bitmap, N, d, dtype, Q, K, V,
                                  scaleLog2, applySoftmax, out, nHeads, (int)ldIn, (int)ldOut, nTcb,
                                  stream);
  const HeadLayout hl = {nHeads, (int)ldIn, (int)ldOut, nTcb};
  return dtype == 0 ? window::dispatch_d<_Float16, false>(rowWindowOffset, windowOrder, sparseAToXidx, bitmap, N,
                                           d, Q, K, V, scaleLog2, applySoftmax, out, nullptr, hl,
                                           stream)
                    : window::dispatch_d<__bf16, false>(rowWindowOffset, windowOrder, sparseAToXidx, bitmap, N, d,
                                         Q, K, V, scaleLog2, applySoftmax, out, nullptr, hl,
                                         stream);
}

}  // namespace f3s
