"""Preprocessing at the window sizes where its kernels change hands or fill up: groups of 64 edges,
the most a wave takes, the sort kernels' capacities, and columns that spread evenly, crowd into a few
bins, repeat or descend. Bit-exact against the oracle, through the one call and through count + fill."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

KEYS = ["rowWindowOffset", "sortedRowWindows", "tcblockRowid", "tcblocktileId", "tcblockOffset",
        "sparseAToXidx", "blockPartition", "edgeToColumn", "edgeToRow"]


def window_rows(rng, n, N, columns):
    """16 rows with n edges in all (some rows empty), columns per `columns`."""
    share = rng.random(16) * (rng.random(16) > 0.2)
    share[rng.integers(16)] += 0.5
    cuts = np.sort(rng.choice(16, size=n, p=share / share.sum()))
    rows = []
    for r in range(16):
        k = int((cuts == r).sum())
        if columns == "crowded":
            lo = N // 3
            pool = np.concatenate([np.arange(lo, min(N, lo + max(300, 2 * n // 8))),
                                   rng.integers(0, N, 20)])
            cols = rng.choice(np.unique(pool), size=min(k, 200), replace=False)
            cols = np.concatenate([cols, rng.choice(N, size=k - len(cols), replace=False)])
        else:
            cols = rng.choice(N, size=k, replace=k > N)
        cols = np.unique(cols) if columns != "rough" else cols
        if columns == "rough" and k > 2:
            cols[k // 2] = cols[0]  # unsorted, with a repeated column
        rows.append(cols.astype(np.int32))
    return rows


def build(rng, sizes, N, columns):
    rows = [r for n in sizes for r in window_rows(rng, n, N, columns)]
    rows += [np.zeros(0, np.int32)] * (N - len(rows))
    rowPtr = np.zeros(N + 1, np.int32)
    rowPtr[1:] = np.cumsum([len(r) for r in rows])
    return rowPtr, np.concatenate(rows).astype(np.int32)


SIZES = [0, 1, 2, 63, 64, 65, 255, 256, 257, 700, 958, 959, 960, 961, 962, 1023, 1024, 1025, 1100,
         2048, 4095, 4096, 4097, 5000]


@pytest.mark.parametrize("W", [16, 8])
@pytest.mark.parametrize("columns", ["even", "crowded", "rough"])
# 1000: fewer columns than bins; 40 000: one bitset pass; 400 003: sort kernels for the long windows
@pytest.mark.parametrize("N", [1000, 40_000, 400_003])
def test_window_sizes(oracle_mod, N, columns, W):
    from fused3s_amd import capi
    print("case window sizes N=%d %s W=%d" % (N, columns, W), flush=True)
    rng = np.random.default_rng(N + W)
    sizes = SIZES + ([16_384, 16_385, 20_000] if N > 1000 else [])
    rowPtr, colIdx = build(rng, sizes, N, columns)
    want = oracle_mod.preprocess(rowPtr, colIdx, N, 16, W)
    rp, ci = torch.as_tensor(rowPtr).cuda(), torch.as_tensor(colIdx).cuda()
    for two_phase in (False, True):
        got = capi.preprocess(rp, ci, N, 16, W, two_phase=two_phase)
        assert got["blockCount"] == want["blockCount"]
        for k in KEYS:
            assert np.array_equal(got[k].cpu().numpy(), want[k]), (k, two_phase)
        bm = got["tcbBitMap"].cpu().view(torch.int64).numpy().view(np.uint64)
        assert np.array_equal(bm, want["tcbBitMap"]), two_phase


# Windows on both sides of 2048 (each workgroup adds up the counts in front of it, or a scan is
# launched) and of 16 384 (one launch per phase, or one per kind of window), counts that tie, counts
# beyond the last bin of the window order, and graphs without edges
@pytest.mark.parametrize("nRW,edges,wide", [(1, 0, 0), (8, 5, 0), (9, 20, 1), (2047, 3, 1),
                                            (2048, 2, 2), (2049, 2, 2), (16_384, 1, 2),
                                            (16_385, 1, 2)])
@pytest.mark.parametrize("W", [16, 8])
def test_window_counts(oracle_mod, nRW, edges, wide, W):
    from fused3s_amd import capi
    print("case window counts nRW=%d edges=%d wide=%d W=%d" % (nRW, edges, wide, W), flush=True)
    rng = np.random.default_rng(nRW + W)
    N = 16 * nRW - 5
    degree = rng.integers(0, edges + 1, N) if edges else np.zeros(N, np.int64)
    for k in range(wide):  # 40 000 edges: more than 4095 blocks of 8 columns
        degree[16 * int(rng.integers(nRW - 1))] = min(N, 40_000)
    rowPtr = np.zeros(N + 1, np.int32)
    rowPtr[1:] = np.cumsum(degree)
    colIdx = np.concatenate([np.sort(rng.choice(N, size=int(k), replace=False)) if k > 100 else
                             np.sort(rng.integers(0, N, int(k))) for k in degree]).astype(np.int32)
    want = oracle_mod.preprocess(rowPtr, colIdx, N, 16, W)
    rp, ci = torch.as_tensor(rowPtr).cuda(), torch.as_tensor(colIdx).cuda()
    for two_phase in (False, True):
        got = capi.preprocess(rp, ci, N, 16, W, two_phase=two_phase)
        assert got["blockCount"] == want["blockCount"]
        for k in KEYS:
            assert np.array_equal(got[k].cpu().numpy(), want[k]), (k, two_phase)
        bm = got["tcbBitMap"].cpu().view(torch.int64).numpy().view(np.uint64)
        assert np.array_equal(bm, want["tcbBitMap"]), two_phase


# A window whose columns crowd into few of its bins is binned again around its middle edge, and sorted where
# that crowds as well. Communities at both ends of the columns and in the middle, two far apart, one column
# in many edges, bins filled to the limit of 24 and beyond; the last column of 2^22 is a word of ones
@pytest.mark.parametrize("N", [900, 15_000, 400_003, 1 << 22])
def test_crowded_windows(oracle_mod, N):
    from fused3s_amd import capi
    print("case crowded windows N=%d" % N, flush=True)
    rng = np.random.default_rng(N)

    def around(at, n, width):
        at = min(max(0, at), N - width)
        return at + rng.integers(0, width, n)

    bits = max(1, (N - 1).bit_length() - 10)
    windows = []
    for n in (25, 64, 65, 128, 129, 250, 256, 257, 500, 704, 705, 960):
        width = min(N, 200 + n // 4)
        for at in (0, N // 2, N - width):
            windows.append(around(at, n, width))                                  # one community
            windows.append(np.where(rng.random(n) < 0.15, rng.integers(0, N, n), around(at, n, width)))
        windows.append(np.where(rng.random(n) < 0.5, around(0, n, width), around(N - width, n, width)))
        windows.append(np.full(n, N - 1))                                         # sorted after both attempts
        windows.append(np.where(rng.random(n) < 0.3, N - 1, rng.integers(0, N, n)))
        for k in (23, 24, 25):                                                    # bins of just that many edges
            lo = (N // 3 >> bits) << bits
            spread = rng.integers(0, N, n)
            spread[:min(n, k)] = lo + np.arange(min(n, k)) % (1 << bits)
            windows.append(spread)
    degree = np.zeros(N, np.int64)
    columns = []
    for w, cols in enumerate(windows[:(N + 15) // 16]):
        rows = np.sort(rng.integers(0, 16, len(cols)))
        rows = np.minimum(rows, N - 1 - 16 * w)
        order = np.lexsort((cols, rows)) if w % 4 else np.argsort(rows, kind="stable")
        degree[16 * w:16 * w + 16] += np.bincount(rows, minlength=16)[:min(16, N - 16 * w)]
        columns.append(cols[order])
    rowPtr = np.zeros(N + 1, np.int32)
    rowPtr[1:] = np.cumsum(degree)
    colIdx = np.concatenate(columns).astype(np.int32)
    want = oracle_mod.preprocess(rowPtr, colIdx, N, 16, 16)
    got = capi.preprocess(torch.as_tensor(rowPtr).cuda(), torch.as_tensor(colIdx).cuda(), N, 16, 16)
    for k in KEYS:
        assert np.array_equal(got[k].cpu().numpy(), want[k]), k


# One launch ranks the short and the long windows of up to 16 384: workgroups of eight waves from 8000
# windows or 1.25M edges on, of at most 480 edges a window, of four otherwise; the long ones are filled 528
# blocks of 16 columns or 640 of 8 at a time
@pytest.mark.parametrize("nRW,edges", [(7999, 60), (8000, 60), (2600, 479), (2606, 480), (2600, 482), (16_384, 20)])
@pytest.mark.parametrize("W", [16, 8])
def test_waves_of_the_one_launch(oracle_mod, nRW, edges, W):
    from fused3s_amd import capi
    print("case one launch nRW=%d edges=%d W=%d" % (nRW, edges, W), flush=True)
    rng = np.random.default_rng(nRW + edges)
    N, E = 16 * nRW - 5, nRW * edges
    wide = {16: 528 * 16, 48: 528 * 16 + 1, 4000: 640 * 8, 4032: 640 * 8 + 1, N - 1: 961, 8000: 3039}
    degree = np.bincount(rng.integers(5000, N - 400, E - sum(wide.values())), minlength=N)
    for r, n in wide.items():
        degree[r] += n  # long windows among the short ones
    rowPtr = np.zeros(N + 1, np.int32)
    rowPtr[1:] = np.cumsum(degree)
    row = np.repeat(np.arange(N), degree)
    colIdx = rng.integers(0, N, E)
    colIdx = colIdx[np.lexsort((colIdx, row))].astype(np.int32)
    assert rowPtr[-1] == E
    for r in wide:
        colIdx[rowPtr[r]:rowPtr[r + 1]] = np.sort(rng.choice(N, degree[r], replace=False))
    want = oracle_mod.preprocess(rowPtr, colIdx, N, 16, W)
    got = capi.preprocess(torch.as_tensor(rowPtr).cuda(), torch.as_tensor(colIdx).cuda(), N, 16, W)
    for k in KEYS:
        assert np.array_equal(got[k].cpu().numpy(), want[k]), k


# Above 393 216 nodes a workgroup ranks the windows of 961 to 2048 and of up to 16 384 edges: 256 and 1024
# edges at a time, bins of 32 edges and more by a radix sort. The last column of a power of two has a bit
# more than the others
@pytest.mark.parametrize("N", [1 << 19, (1 << 19) - 1, 500_000])
def test_windows_of_a_workgroup(oracle_mod, N):
    from fused3s_amd import capi
    print("case windows of a workgroup N=%d" % N, flush=True)
    rng = np.random.default_rng(N)
    windows = []
    for n in (961, 1023, 1024, 1025, 1536, 2048, 4095, 4096, 4097, 5000, 16_383, 16_384, 16_385):
        even = rng.integers(0, N, n)
        even[:2] = [0, N - 1]
        windows.append(even)
        windows.append(np.where(rng.random(n) < 0.2, rng.integers(0, N, n), N // 2 + rng.integers(0, 300, n)))
        windows.append(np.where(rng.random(n) < 16 / n, N - 1, even))
        for k in (31, 32, 33):
            spread = even.copy()
            spread[2:2 + k] = 0 if k == 33 else N - 1
            windows.append(spread)
    degree = np.zeros(N, np.int64)
    columns = []
    for w, cols in enumerate(windows):
        rows = np.sort(rng.integers(0, 16, len(cols)))
        degree[16 * w:16 * w + 16] = np.bincount(rows, minlength=16)
        columns.append(cols[np.lexsort((cols, rows))] if w % 4 else cols)
    rowPtr = np.zeros(N + 1, np.int32)
    rowPtr[1:] = np.cumsum(degree)
    colIdx = np.concatenate(columns).astype(np.int32)
    want = oracle_mod.preprocess(rowPtr, colIdx, N, 16, 16)
    got = capi.preprocess(torch.as_tensor(rowPtr).cuda(), torch.as_tensor(colIdx).cuda(), N, 16, 16)
    for k in KEYS:
        assert np.array_equal(got[k].cpu().numpy(), want[k]), k


# A window's own sixteen columns (the diagonal of an adjacency matrix) get bins of their own where the bins have
# room for that: the most columns for which they do, one more, and powers of two on either side; windows of a wave
# (ten bits of bins), of 256 threads and of 1024 (eleven and thirteen) with all, some and none of their own columns,
# own columns in every row, and neighbours on both sides of them; the last window, whose columns are the last ones
@pytest.mark.parametrize("W", [16, 8])
@pytest.mark.parametrize("N", [1024, 1025, (1 << 15) - 17 * 32 - 1, (1 << 15) - 17 * 32, 1 << 15,
                               (1 << 19) - 17 * 256 - 2, (1 << 19) - 17 * 256 - 1, (1 << 19) - 17 * 512])
def test_own_columns(oracle_mod, N, W):
    from fused3s_amd import capi
    print("case own columns N=%d W=%d" % (N, W), flush=True)
    rng = np.random.default_rng(N + W)
    nRW = (N + 15) // 16
    rows = [np.zeros(0, np.int32)] * N
    sizes = [40, 400, 900] + ([1500, 2047, 2049, 3000, 5000] if N > 393_216 else [])
    picked = np.concatenate([[0, nRW - 1], rng.choice(np.arange(1, nRW - 1), 3 * len(sizes) - 2, replace=False)])
    for k, w in enumerate(picked):
        own = np.arange(16 * w, min(16 * w + 16, N))
        for r in own:
            cols = rng.choice(N, size=min(sizes[k % len(sizes)] // 16, N // 2), replace=False)
            near = np.clip(16 * w + rng.integers(-40, 56, 6), 0, N - 1)
            extra = {0: [r], 1: own, 2: near}[k % 3]
            rows[r] = np.unique(np.concatenate([cols, extra])).astype(np.int32)
    rowPtr = np.zeros(N + 1, np.int32)
    rowPtr[1:] = np.cumsum([len(r) for r in rows])
    colIdx = np.concatenate(rows).astype(np.int32)
    want = oracle_mod.preprocess(rowPtr, colIdx, N, 16, W)
    rp, ci = torch.as_tensor(rowPtr).cuda(), torch.as_tensor(colIdx).cuda()
    got = capi.preprocess(rp, ci, N, W=W)
    for key in KEYS:
        assert np.array_equal(got[key].cpu().numpy(), want[key]), key
    assert np.array_equal(got["tcbBitMap"].cpu().view(torch.int64).numpy().view(np.uint64), want["tcbBitMap"])


# Columns that crowd into few bins are binned again, by what they are, around the window's middle edge: communities
# around the window's own columns, below, above, and across the ends of the range, narrower and wider than the
# 512 columns (or four bins) that half of the bins then cover, alone and with edges elsewhere
@pytest.mark.parametrize("N", [1025, 100_000, (1 << 17) - 17 * 128 - 1, (1 << 17) - 17 * 128, 500_000])
def test_communities_around_own_columns(oracle_mod, N):
    from fused3s_amd import capi
    print("case communities N=%d" % N, flush=True)
    rng = np.random.default_rng(N)
    nRW = (N + 15) // 16
    rows = [np.zeros(0, np.int32)] * N
    kinds = [(reach, shift, size) for reach in (40, 120, 300, 700, 3000) for shift in (-1, 0, 1) for size in (150, 500, 940)]
    picked = np.unique(np.concatenate([[0, 1, nRW - 2, nRW - 1],
                                       rng.choice(nRW, min(nRW - 4, len(kinds) + 10), replace=False)]))
    for k, w in enumerate(rng.permutation(picked)):
        reach, shift, size = kinds[k % len(kinds)]
        own = np.arange(16 * w, min(16 * w + 16, N))
        near = np.arange(max(16 * w + shift * reach - reach, 0), min(16 * w + 16 + shift * reach + reach, N))
        if len(near) == 0:
            near = own
        for r in own:
            cols = rng.choice(near, size=min(size // 16 - 1, len(near)), replace=False)
            far = rng.integers(0, N, k % 2)
            rows[r] = np.unique(np.concatenate([cols, far, [r]])).astype(np.int32)
    rowPtr = np.zeros(N + 1, np.int32)
    rowPtr[1:] = np.cumsum([len(r) for r in rows])
    colIdx = np.concatenate(rows).astype(np.int32)
    want = oracle_mod.preprocess(rowPtr, colIdx, N)
    got = capi.preprocess(torch.as_tensor(rowPtr).cuda(), torch.as_tensor(colIdx).cuda(), N)
    for key in KEYS:
        assert np.array_equal(got[key].cpu().numpy(), want[key]), key
    assert np.array_equal(got["tcbBitMap"].cpu().view(torch.int64).numpy().view(np.uint64), want["tcbBitMap"])


def split_columns(rng, cols, lengths):
    """16 ascending rows of the given lengths over `cols`, which together name every one of them."""
    cols = np.sort(cols)
    rows = [np.sort(rng.choice(cols, size=min(k, len(cols)), replace=False)) for k in lengths]
    at = int(np.argmax(lengths))
    missing = np.setdiff1d(cols, np.concatenate(rows))
    rows[at] = np.union1d(rows[at], missing)
    return [r.astype(np.int32) for r in rows]


# Graphs of long windows keep a window's ids in LDS beside its bitmaps where both fit (up to 940 blocks of
# 16 columns at this N), as 16-bit halves whose upper ones change at multiples of 65 536, and count with
# 16-bit prefixes up to 65 535 distinct columns: windows on both sides of each, rows that start at every
# place of a group of four edges, several of them in one group, and a window of repeated columns.
@pytest.mark.parametrize("W", [16, 8])
def test_long_windows_ids_and_prefixes(oracle_mod, W):
    from fused3s_amd import capi
    print("case long windows, ids and prefixes W=%d" % W, flush=True)
    rng = np.random.default_rng(41 + W)
    N = 131_200
    even = lambda n: rng.choice(N, size=n, replace=False)
    ends = np.concatenate([np.arange(101), np.arange(N - 99, N)])
    about = np.concatenate([np.arange(65_530, 65_541), np.arange(131_069, 131_076)])
    windows = [split_columns(rng, even(n), [n // 8] * 16) for n in (15_039, 15_040, 15_041)]
    windows += [split_columns(rng, even(n), [n // 2] * 16) for n in (65_535, 65_536, 65_537)]
    windows += [split_columns(rng, ends, [k % 4 for k in range(15)] + [150])]
    windows += [split_columns(rng, about, [1, 0, 2, 1, 1, 1, 3, 0, 0, 1, 5, 2, 2, 1, 1, 18])]
    windows += [split_columns(rng, even(40), [1] * 16), split_columns(rng, even(3), [0] * 15 + [3])]
    rough = split_columns(rng, even(9_000), [1_000] * 16)
    rough[7][500] = rough[7][2]
    windows += [rough]
    nRW = (N + 15) // 16
    while sum(len(r) for rows in windows for r in rows) < 2048 * nRW:  # every second column, 16 rows
        windows += [[np.flatnonzero(rng.random(N) < 0.5).astype(np.int32) for _ in range(16)]]
    rows = [r for w in windows for r in w]
    rowPtr = np.zeros(N + 1, np.int32)
    rowPtr[1:len(rows) + 1] = np.cumsum([len(r) for r in rows])
    rowPtr[len(rows) + 1:] = rowPtr[len(rows)]
    colIdx = np.concatenate(rows).astype(np.int32)
    want = oracle_mod.preprocess(rowPtr, colIdx, N, 16, W)
    assert list(want["blockPartition"][:6]) == [-(-n // W) for n in (15_039, 15_040, 15_041, 65_535,
                                                                    65_536, 65_537)]
    got = capi.preprocess(torch.as_tensor(rowPtr).cuda(), torch.as_tensor(colIdx).cuda(), N, 16, W)
    for k in KEYS:
        assert np.array_equal(got[k].cpu().numpy(), want[k]), k
    assert np.array_equal(got["tcbBitMap"].cpu().view(torch.int64).numpy().view(np.uint64),
                          want["tcbBitMap"])


# Above 16 384 windows the order of the one call comes from rows of a histogram, one per 1024 windows (up to
# 524 288 of them), whose last bin is 1023 blocks and more; long windows go through lists, mid and large
# ones (one bitset pass: all of them large): windows on both sides of each, ties across rows
@pytest.mark.parametrize("nRW", [16_385, 17_407, 17_408, 17_409, 18_432, 24_576, 24_577, 40_000,
                                 524_288, 524_289])
def test_order_beside_the_fill(oracle_mod, nRW):
    from fused3s_amd import capi
    print("case order beside the fill nRW=%d" % nRW, flush=True)
    rng = np.random.default_rng(nRW)
    N, W = 16 * nRW - 3, 8
    degree = np.zeros(N, np.int64)
    degree[rng.choice(N, 50_000, replace=False)] = rng.integers(1, 40, 50_000)
    wide = np.array([1022, 1023, 1024, 1024, 2045, 2046, 2047, 120, 121, 512, 513]) * 8
    at = np.concatenate([[0, 1023, 1024, nRW - 2], rng.choice(nRW - 2, len(wide) - 4, replace=False)])
    for w, n in zip(at, wide):
        degree[16 * w:16 * w + 16] = 0
        degree[16 * w] = n
    rowPtr = np.zeros(N + 1, np.int32)
    rowPtr[1:] = np.cumsum(degree)
    colIdx = rng.integers(0, N, int(rowPtr[-1])).astype(np.int32)
    for w, n in zip(at, wide):
        if degree[16 * w] == n:
            colIdx[rowPtr[16 * w]:rowPtr[16 * w + 1]] = np.sort(rng.choice(N, int(n), replace=False))
    want = oracle_mod.preprocess(rowPtr, colIdx, N, 16, W)
    rp, ci = torch.as_tensor(rowPtr).cuda(), torch.as_tensor(colIdx).cuda()
    for two_phase in (False, True):
        got = capi.preprocess(rp, ci, N, 16, W, two_phase=two_phase)
        for k in KEYS:
            assert np.array_equal(got[k].cpu().numpy(), want[k]), (k, two_phase)


# The order's histogram has 4096 bins: windows of 4095 blocks and more take further rounds. Counts at
# the rounds' edges, ties of more than a wave, rounds that no window falls into, and one window that
# spans every node
@pytest.mark.parametrize("W,counts", [
    (8, [4093, 4094, 4095, 4096, 8189, 8190, 8191, 12_284, 12_285, 16_375, 0, 1]),
    (8, [16_375]),
    (8, [4095] * 70 + [4094, 4100]),
    (16, [4094, 4095, 4096, 8186]),
])
def test_window_order_of_wide_windows(oracle_mod, W, counts):
    from fused3s_amd import capi
    print("case wide windows W=%d counts=%s" % (W, counts[:12]), flush=True)
    N = 131_000
    rng = np.random.default_rng(len(counts) + W)
    rows = [np.sort(rng.choice(N, size=3, replace=False)).astype(np.int32) for _ in range(N)]
    at = rng.choice(N // 16, size=len(counts), replace=False)
    if len(counts) > 64:
        at = np.arange(100, 100 + len(counts))
    for w, blocks in zip(at, counts):
        cols = np.sort(rng.choice(N, size=blocks * W, replace=False)).astype(np.int32)
        for r in range(16):
            rows[16 * w + r] = cols[r::16]
    rowPtr = np.zeros(N + 1, np.int32)
    rowPtr[1:] = np.cumsum([len(r) for r in rows])
    colIdx = np.concatenate(rows)
    want = oracle_mod.preprocess(rowPtr, colIdx, N, 16, W)
    assert sorted(counts) == sorted(want["blockPartition"][at])
    rp, ci = torch.as_tensor(rowPtr).cuda(), torch.as_tensor(colIdx).cuda()
    for two_phase in (False, True):
        got = capi.preprocess(rp, ci, N, 16, W, two_phase=two_phase)
        for k in KEYS:
            assert np.array_equal(got[k].cpu().numpy(), want[k]), (k, two_phase)


@pytest.mark.parametrize("nRW", [1, 511, 512, 513, 2048, 4097, 16_384])
def test_window_order_alone(nRW):
    """Long windows first, equal counts by window; from 512 blocks on, 64 bins an octave."""
    from fused3s_amd import capi
    print("case window order nRW=%d" % nRW, flush=True)
    rng = np.random.default_rng(nRW)
    count = rng.integers(0, 40, nRW)
    far = rng.random(nRW) < 0.1
    count[far] = rng.choice([511, 512, 513, 1023, 1024, 5000, 100_000], size=int(far.sum()))
    rwo = torch.zeros(nRW + 1, dtype=torch.int32, device="cuda")
    rwo[1:] = torch.as_tensor(np.cumsum(count), device="cuda")
    order = torch.full((nRW,), -1, dtype=torch.int32, device="cuda")
    rc = capi.lib().f3s_window_order(capi._ptr(rwo), nRW, capi._ptr(order), capi._stream())
    assert rc == 0, capi.lib().f3s_last_error()
    bucket = np.where(count < 512, count, 0)
    for octave in range(9, 17):
        inside = (count >> octave) == 1
        bucket[inside] = 512 + (octave - 9) * 64 + ((count[inside] >> (octave - 6)) & 63)
    np.testing.assert_array_equal(order.cpu().numpy(), np.argsort(-bucket, kind="stable"))


@pytest.mark.parametrize("nRW", [1, 65, 513, 2049, 16_384])
def test_window_order_of_descending_offsets(nRW):
    """Offsets that did not come from preprocessing: a window whose range is negative counts as empty,
    and the order is still a permutation of all windows."""
    from fused3s_amd import capi
    print("case descending offsets nRW=%d" % nRW, flush=True)
    rng = np.random.default_rng(nRW)
    offsets = rng.integers(-2**31, 2**31, nRW + 1) if nRW == 65 else rng.integers(0, 500, nRW + 1)
    rwo = torch.as_tensor(offsets.astype(np.int32)).cuda()
    order = torch.full((nRW,), -1, dtype=torch.int32, device="cuda")
    rc = capi.lib().f3s_window_order(capi._ptr(rwo), nRW, capi._ptr(order), capi._stream())
    assert rc == 0, capi.lib().f3s_last_error()
    got = order.cpu().numpy()
    np.testing.assert_array_equal(np.sort(got), np.arange(nRW))
    if nRW != 65:
        count = np.maximum(np.diff(offsets), 0)
        np.testing.assert_array_equal(got, np.argsort(-count, kind="stable"))


def test_call_without_order_on_descending_offsets(oracle_mod):
    """A call that makes its own order (1040 windows of 33 blocks, d = 256) writes zeros to the rows of a
    window whose offsets descend, as the call with a given order does."""
    from fused3s_amd import F3S
    print("case own order, descending offsets", flush=True)
    nRW, blocks, d = 1040, 33, 256
    N = 16 * nRW
    rng = np.random.default_rng(3)
    atox = np.sort(rng.integers(0, N, (nRW, blocks * 16)), axis=1).astype(np.int32)
    bitmap = rng.integers(0, 2**63, nRW * blocks * 4, dtype=np.uint64)
    rwo = np.arange(nRW + 1) * blocks
    broken = rwo.copy()
    broken[500] = 0  # window 499 descends, window 500 spans the first 501 windows' blocks
    Q, K, V = [torch.rand((N, d), dtype=torch.float32).half().cuda() for _ in range(3)]
    dev = lambda a: torch.as_tensor(a).cuda()
    at, bm = dev(atox.reshape(-1)), dev(bitmap.view(np.int64)).view(torch.uint64)
    out = []
    for offsets in (rwo, broken):
        spoiled = torch.full((N, d), float("nan"), device="cuda")
        del spoiled  # the memory the call's result is likely to get
        out.append(F3S.f3s_1tb1rw(dev(offsets.astype(np.int32)), at, bm, N, Q, K, V, 8, True,
                                  False)[1].cpu().numpy())
    assert not out[1][499 * 16:500 * 16].any()
    keep = np.ones(N, bool)
    keep[499 * 16:501 * 16] = False
    assert np.isfinite(out[1]).all() and np.array_equal(out[0][keep], out[1][keep])


def test_threads_and_streams(oracle_mod):
    """Eight host threads preprocess graphs of their own on streams of their own at the same time: each
    gets its own total and, for a graph with a column that does not exist, its own error."""
    import threading

    from fused3s_amd import capi
    print("case threads", flush=True)
    graphs = []
    for k in range(8):
        rng = np.random.default_rng(k)
        N = 500 + 700 * k
        rowPtr, colIdx = build(rng, [int(n) for n in rng.integers(0, 300, N // 16)], N, "even")
        if k == 5:
            colIdx[len(colIdx) // 2] = N
        want = None if k == 5 else oracle_mod.preprocess(rowPtr, colIdx, N, 16, 16)
        graphs.append((N, torch.as_tensor(rowPtr).cuda(), torch.as_tensor(colIdx).cuda(), want))
    torch.cuda.synchronize()
    wrong = []

    def work(k):
        N, rp, ci, want = graphs[k]
        with torch.cuda.stream(torch.cuda.Stream()):
            for turn in range(10):
                try:
                    got = capi.preprocess(rp, ci, N, two_phase=bool(turn % 2))
                except RuntimeError as e:
                    if want is not None or "column index" not in str(e):
                        wrong.append((k, turn, str(e)))
                    continue
                torch.cuda.current_stream().synchronize()
                if want is None or got["blockCount"] != want["blockCount"] or not np.array_equal(
                        got["sparseAToXidx"].cpu().numpy(), want["sparseAToXidx"]):
                    wrong.append((k, turn))

    threads = [threading.Thread(target=work, args=(k,)) for k in range(8)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong, wrong
