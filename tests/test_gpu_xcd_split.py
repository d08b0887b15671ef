"""How units are dealt to the XCDs: head groups, slice groups, phases and window groups of the
column-sliced schedule, and the chunks of the launches with waves for short windows, at head counts and window
counts that do not divide evenly. Every (window, head) has to be computed exactly once."""
import numpy as np
import pytest
import torch

from conftest import random_csr

pytestmark = pytest.mark.gpu


def on_gpu(oracle_mod, rowPtr, colIdx, N):
    pre = oracle_mod.preprocess(rowPtr, colIdx, N)
    t = lambda k: torch.as_tensor(pre[k].astype(np.int32)).cuda()
    bm = torch.as_tensor(pre["tcbBitMap"].view(np.int64)).cuda().view(torch.uint64)
    return pre, (t("rowWindowOffset"), t("sortedRowWindows"), t("sparseAToXidx"), bm)


def check(oracle_mod, pre, N, heads, d, Q, K, V, got):
    got = got.cpu().numpy().reshape(N, heads, d)
    for h in range(heads):
        want = oracle_mod.attention_ref(pre["rowWindowOffset"], pre["sparseAToXidx"],
                                        pre["tcbBitMap"], N, Q[:, h].contiguous().cpu().numpy(),
                                        K[:, h].contiguous().cpu().numpy(),
                                        V[:, h].contiguous().cpu().numpy(), float(np.sqrt(d)))
        assert np.abs(got[:, h] - want).max() < 2e-2, h
        assert np.abs(got[:, h] - want).mean() < 1e-3 * np.abs(want).mean(), h


# (1, 64): window groups; (3, 32), (6, 64): heads that split once or not at all; (4, 64): head and
# slice groups; (8, 64), (8, 128): one head per XCD and two phases
@pytest.mark.parametrize("heads,d", [(1, 64), (3, 32), (6, 64), (4, 64), (8, 64), (8, 128)])
@pytest.mark.parametrize("N", [17, 1003])
def test_sliced(oracle_mod, monkeypatch, N, heads, d):
    from fused3s_amd import capi
    print("case sliced split N=%d heads=%d d=%d" % (N, heads, d), flush=True)
    rng = np.random.default_rng(heads * d)
    rowPtr, colIdx = random_csr(rng, N, 30, hub=37, empty_frac=0.05)
    pre, (rwo, order, atox, bm) = on_gpu(oracle_mod, rowPtr, colIdx, N)
    g = torch.Generator().manual_seed(d)
    Q, K, V = [torch.randn((N, heads, d), generator=g).half().cuda() for _ in range(3)]
    monkeypatch.setenv("F3S_SCHEDULE", "sliced")
    ws = capi.attention_workspace(N, d, "cuda", heads=heads)
    ws.fill_(0xFF)
    got = capi.attention_heads(rwo, order, atox, bm, N, Q, K, V, float(np.sqrt(d)), workspace=ws)
    check(oracle_mod, pre, N, heads, d, Q, K, V, got)


# K + V of a group of heads that would take 18 and 17 slices of 8 MiB: 16 wider ones are used. Columns at
# every slice edge, and a window that names all slices
@pytest.mark.parametrize("persistent", ["0", "1"])
@pytest.mark.parametrize("heads,d,N", [(0, 256, 140_003), (2, 128, 270_011)])
def test_sixteen_slices(oracle_mod, monkeypatch, heads, d, N, persistent):
    from fused3s_amd import capi
    print("case sixteen slices heads=%d d=%d persistent=%s" % (heads, d, persistent), flush=True)
    nRW, width = (N + 15) // 16, (N + 15) // 16  # slices of N / 16 columns, rounded up
    rng = np.random.default_rng(d)
    edge = np.concatenate([np.arange(1, 16) * width + k for k in (-1, 0, 1)])
    deg = rng.integers(0, 3, N)
    deg[5] = 4000
    deg[100:100 + len(edge)] = 1
    rowPtr = np.zeros(N + 1, np.int32)
    rowPtr[1:] = np.cumsum(deg)
    colIdx = rng.integers(0, N, int(rowPtr[-1])).astype(np.int32)
    colIdx[rowPtr[5]:rowPtr[6]] = np.sort(rng.choice(N, size=4000, replace=False))
    colIdx[rowPtr[100]:rowPtr[100 + len(edge)]] = edge
    pre, (rwo, order, atox, bm) = on_gpu(oracle_mod, rowPtr, colIdx, N)
    g = torch.Generator().manual_seed(d)
    Q, K, V = [torch.randn((N, max(heads, 1), d), generator=g).half().cuda() for _ in range(3)]
    monkeypatch.setenv("F3S_SCHEDULE", "sliced")
    monkeypatch.setenv("F3S_SLICED_PERSISTENT", persistent)
    monkeypatch.delenv("F3S_SLICE_PHASES", raising=False)
    ws = capi.attention_workspace(N, d, "cuda", heads=heads)
    per_slice = nRW * max(heads, 1) * (16 * d + 32) * 4  # bytes of partial results
    assert 16 <= ws.numel() / per_slice < 17
    ws.fill_(0xFF)
    if heads:
        got = capi.attention_heads(rwo, order, atox, bm, N, Q, K, V, float(np.sqrt(d)), workspace=ws)
    else:
        got = capi.attention(rwo, order, atox, bm, N, *[t[:, 0].contiguous() for t in (Q, K, V)],
                             float(np.sqrt(d)), workspace=ws)
    check(oracle_mod, pre, N, max(heads, 1), d, Q, K, V, got)


# The resident form deals the same slices in as few phases as they divide into: 3 (three phases as in
# launch order), 4 (one phase; with four heads in two), 5 and 6 slices
@pytest.mark.parametrize("heads,d,N", [(0, 64, 70_001), (0, 128, 60_013), (4, 64, 100_003),
                                       (0, 128, 81_003), (2, 64, 180_001)])
def test_resident_deals_the_same_slices(oracle_mod, monkeypatch, heads, d, N):
    from fused3s_amd import capi
    print("case resident deal heads=%d d=%d N=%d" % (heads, d, N), flush=True)
    rng = np.random.default_rng(N)
    deg = rng.poisson(1.0, N)
    deg[::5003] = 900
    rowPtr = np.zeros(N + 1, np.int32)
    rowPtr[1:] = np.cumsum(deg)
    colIdx = rng.integers(0, N, int(rowPtr[-1])).astype(np.int32)
    pre, (rwo, order, atox, bm) = on_gpu(oracle_mod, rowPtr, colIdx, N)
    g = torch.Generator().manual_seed(N)
    Q, K, V = [torch.randn((N, max(heads, 1), d), generator=g).half().cuda() for _ in range(3)]
    monkeypatch.setenv("F3S_SCHEDULE", "sliced")
    ws = capi.attention_workspace(N, d, "cuda", heads=heads)
    got = []
    for persistent in ("0", "1"):
        monkeypatch.setenv("F3S_SLICED_PERSISTENT", persistent)
        ws.fill_(0xFF)
        if heads:
            got.append(capi.attention_heads(rwo, order, atox, bm, N, Q, K, V, float(np.sqrt(d)),
                                            workspace=ws))
        else:
            got.append(capi.attention(rwo, order, atox, bm, N,
                                      *[t[:, 0].contiguous() for t in (Q, K, V)],
                                      float(np.sqrt(d)), workspace=ws))
    assert torch.equal(got[0], got[1])
    check(oracle_mod, pre, N, max(heads, 1), d, Q, K, V, got[1])


# The number of slices follows from the blocks per window: of 2 048 windows, the first `long` name
# `blocks` blocks each (2.5, 4.5 and 8 slices' worth on average at d = 128; K + V of 17 and 134 MB bound
# it, one or four slices at a time). A prepared workspace of one structure serves a call on another, whose
# slices are other ones.
@pytest.mark.parametrize("heads,d,N", [(0, 128, 32_771), (0, 256, 131_101), (2, 32, 32_771),
                                       (4, 128, 65_551)])
def test_slices_by_blocks_per_window(oracle_mod, monkeypatch, heads, d, N):
    from fused3s_amd import capi
    print("case slices by blocks heads=%d d=%d N=%d" % (heads, d, N), flush=True)
    monkeypatch.setenv("F3S_SCHEDULE", "sliced")
    monkeypatch.delenv("F3S_SLICE_PHASES", raising=False)
    g = torch.Generator().manual_seed(N)
    Q, K, V = [torch.randn((N, max(heads, 1), d), generator=g).half().cuda() for _ in range(3)]
    ws = capi.attention_workspace(N, d, "cuda", heads=heads)
    structures = []
    for per_window in (3, 90, 300):  # blocks of 16 distinct columns
        rng = np.random.default_rng(per_window)
        long = min((N + 15) // 16 - 2, 40)
        rowPtr = np.zeros(N + 1, np.int32)
        deg = np.zeros(N, np.int64)
        deg[:16 * long:16] = min(N, 16 * per_window * ((N + 15) // 16) // long)
        deg[N // 2:] = 1
        rowPtr[1:] = np.cumsum(deg)
        cols = [np.sort(rng.choice(N, size=k, replace=False)) for k in deg[:16 * long:16]]
        colIdx = np.concatenate(cols + [rng.integers(0, N, int(deg[N // 2:].sum()))])
        structures.append(on_gpu(oracle_mod, rowPtr, colIdx.astype(np.int32), N))
    for prepared_for, (pre, (rwo, order, atox, bm)) in zip((0, 0, 2), structures):
        ws.fill_(0xFF)
        base = structures[prepared_for][1]
        capi.attention_prepare(base[0], base[2], N, d, ws, heads=heads)
        if heads:
            got = capi.attention_heads(rwo, order, atox, bm, N, Q, K, V, float(np.sqrt(d)),
                                       workspace=ws, prepared=True)
        else:
            got = capi.attention(rwo, order, atox, bm, N, *[t[:, 0].contiguous() for t in (Q, K, V)],
                                 float(np.sqrt(d)), workspace=ws, prepared=True)
        check(oracle_mod, pre, N, max(heads, 1), d, Q, K, V, got)


# Single-head calls at d <= 64 on structures of fewer blocks than 260 000 (d = 32) or 450 000 (d = 64) leave
# their workspace alone, those of more use it
@pytest.mark.parametrize("d,blocks", [(32, 259_000), (32, 261_000), (64, 449_000), (64, 451_000),
                                      (96, 200_000)])
def test_small_single_head_calls_leave_the_workspace(oracle_mod, monkeypatch, d, blocks):
    from fused3s_amd import capi
    print("case small single head d=%d blocks=%d" % (d, blocks), flush=True)
    monkeypatch.delenv("F3S_SCHEDULE", raising=False)
    monkeypatch.delenv("F3S_SLICE_PHASES", raising=False)
    N = 16 * 2048 - 3
    rng = np.random.default_rng(blocks)
    long = 300
    deg = np.ones(N, np.int64)
    deg[:16 * long:16] = min(N, 16 * blocks // long)
    rowPtr = np.zeros(N + 1, np.int32)
    rowPtr[1:] = np.cumsum(deg)
    colIdx = np.concatenate([np.sort(rng.choice(N, size=k, replace=False)) if k > 1 else
                             rng.integers(0, N, 1) for k in deg]).astype(np.int32)
    pre, (rwo, order, atox, bm) = on_gpu(oracle_mod, rowPtr, colIdx, N)
    limit = {32: 260_000, 64: 450_000}.get(d, 0)
    assert pre["blockCount"] >= 64 * 2048
    g = torch.Generator().manual_seed(d)
    Q, K, V = [torch.randn((N, 1, d), generator=g).half().cuda() for _ in range(3)]
    assert (capi.attention_workspace(N, d, "cuda", nTCB=atox.numel() // 16) is None) == (
        pre["blockCount"] < limit)
    ws = capi.attention_workspace(N, d, "cuda")
    ws.fill_(0xFF)
    got = capi.attention(rwo, order, atox, bm, N, *[t[:, 0].contiguous() for t in (Q, K, V)],
                         float(np.sqrt(d)), workspace=ws)
    assert bool((ws == 0xFF).all()) == (pre["blockCount"] < limit)
    check(oracle_mod, pre, N, 1, d, Q, K, V, got)


# The window kernel deals the XCDs groups of heads: every (window, head) exactly once, for head counts that
# split into one to eight groups or not at all, and one window more or less than a share of them
@pytest.mark.parametrize("heads,d", [(2, 32), (3, 32), (4, 32), (6, 32), (16, 32), (5, 64), (12, 64),
                                     (16, 64), (4, 96), (7, 128)])
@pytest.mark.parametrize("N", [16, 16 * 7 + 1, 16 * 9])
def test_window_kernel_head_groups(oracle_mod, monkeypatch, heads, d, N):
    from fused3s_amd import capi
    print("case window head groups heads=%d d=%d N=%d" % (heads, d, N), flush=True)
    monkeypatch.setenv("F3S_SCHEDULE", "window")
    rng = np.random.default_rng(heads + N)
    pre, (rwo, order, atox, bm) = on_gpu(oracle_mod, *random_csr(rng, N, 9, empty_frac=0.1), N)
    g = torch.Generator().manual_seed(d)
    Q, K, V = [torch.randn((N, heads, d), generator=g).half().cuda() for _ in range(3)]
    out = torch.full((N, heads * d), float("nan"), device="cuda")
    for od in (order, None):
        got = capi.attention_heads(rwo, od, atox, bm, N, Q, K, V, float(np.sqrt(d)), out=out.clone())
        check(oracle_mod, pre, N, heads, d, Q, K, V, got)


# 32-wide heads two at a time: bit-identical to head by head through every schedule (windows, with and
# without natural order; short windows with long ones beside them, too few of them for pairs at two and four
# heads; column slices in both forms), on rows of a pitch that shifts the pairs off the 128-byte lines, scores
# far above the running maximum in one head of a pair only, and scores that are exactly 0
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("heads", [2, 4, 6, 16])
@pytest.mark.parametrize("kind", ["window", "short", "sliced", "resident"])
def test_pairs_of_heads_are_bit_identical(oracle_mod, monkeypatch, kind, heads, dtype):
    from fused3s_amd import capi
    print("case pairs of heads %s heads=%d %s" % (kind, heads, dtype), flush=True)
    rng = np.random.default_rng(heads)
    d, N = 32, 16 * (1100 if kind == "short" else 300 if kind != "window" else
                     2000 if heads == 2 else 1000) + 5
    deg = rng.poisson(2.0 if kind == "short" else 60.0, N)
    deg[::1999] = 900
    rows = [np.unique(rng.integers(0, N, k)) for k in deg]
    rowPtr = np.zeros(N + 1, np.int32)
    rowPtr[1:] = np.cumsum([len(r) for r in rows])
    pre, (rwo, order, atox, bm) = on_gpu(oracle_mod, rowPtr, np.concatenate(rows).astype(np.int32), N)
    # enough for the window kernel to take pairs
    assert kind != "window" or pre["blockCount"] * (heads // 2) >= (100_000 if heads == 2 else 50_000)
    monkeypatch.setenv("F3S_SCHEDULE", "window" if kind in ("window", "short") else "sliced")
    monkeypatch.setenv("F3S_SLICED_PERSISTENT", "1" if kind == "resident" else "0")
    g = torch.Generator().manual_seed(heads)
    store = torch.randn((3, N, heads * d + 8), generator=g)
    store[0, ::7, d:2 * d] *= 40.0  # scores of head 1 far above the others'
    store[0, 3::11, :d] = 0.0
    store = store.to(dtype).cuda()
    Q, K, V = [store[k, :, :heads * d].unflatten(1, (heads, d)) for k in range(3)]
    monkeypatch.setenv("F3S_SLICE_PHASES", "1")  # as many slices for one head as for all
    scratch = lambda n: None if kind in ("window", "short") else capi.attention_workspace(
        N, d, "cuda", heads=n)
    for od in (order, None) if kind == "window" else (order,):
        got = capi.attention_heads(rwo, od, atox, bm, N, Q, K, V, float(np.sqrt(d)),
                                   workspace=scratch(heads))
        one = [capi.attention_heads(rwo, od, atox, bm, N, *[t[:, h:h + 1] for t in (Q, K, V)],
                                    float(np.sqrt(d)), workspace=scratch(1)) for h in range(heads)]
        assert torch.isfinite(got).all()
        assert torch.equal(got, torch.cat(one, dim=1))


# Wave-per-window launches take 32-wide heads in pairs from 50 000 blocks times pairs on, one or two pairs of
# fewer blocks head by head: both sides of the line, bit-identical to head by head, a few long windows beside
@pytest.mark.parametrize("missing", [1, 0])
@pytest.mark.parametrize("heads,blocks", [(2, 50_000), (4, 25_000)])
def test_pairs_of_heads_in_short_windows(oracle_mod, heads, blocks, missing):
    from fused3s_amd import capi
    print("case short pairs heads=%d blocks=%d" % (heads, blocks - missing), flush=True)
    nRW, d = blocks // 14, 32
    N = 16 * nRW - 3
    rng = np.random.default_rng(blocks + missing)
    counts = np.full(nRW, 14)
    counts[::701] = 41
    over = int(counts.sum()) - (blocks - missing)
    counts[np.setdiff1d(np.arange(nRW), np.arange(0, nRW, 701))[:over]] -= 1
    rwo = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    assert rwo[-1] == blocks - missing < 16 * nRW
    step = N // (41 * 16)
    atox = np.concatenate([np.arange(16 * c) * step for c in counts])
    atox = (atox + rng.integers(0, step, len(atox))).astype(np.int32)
    bitmap = rng.integers(0, 2**63, len(atox) // 4, dtype=np.uint64)
    bitmap &= rng.integers(0, 2**63, len(bitmap), dtype=np.uint64)
    order = np.argsort(-counts, kind="stable").astype(np.int32)
    pre = dict(rowWindowOffset=rwo, sparseAToXidx=atox, tcbBitMap=bitmap)
    dev = lambda a: torch.as_tensor(a).cuda()
    args = dev(rwo), dev(order), dev(atox), dev(bitmap.view(np.int64)).view(torch.uint64), N
    g = torch.Generator().manual_seed(heads)
    Q, K, V = [torch.randn((N, heads, d), generator=g).half().cuda() for _ in range(3)]
    got = capi.attention_heads(*args, Q, K, V, float(np.sqrt(d)))
    one = [capi.attention_heads(*args, *[t[:, h:h + 1] for t in (Q, K, V)], float(np.sqrt(d)))
           for h in range(heads)]
    assert torch.equal(got, torch.cat(one, dim=1))
    check(oracle_mod, pre, N, heads, d, Q, K, V, got)


# The build with 64-bit row offsets takes 32-wide heads in pairs as well: rows of Q, K and V in one array of
# more than 4 GiB, bit-identical to head by head, on both sides of the lines (one pair 100 000 blocks, four
# pairs 12 500)
@pytest.mark.parametrize("heads,deg", [(2, 60), (8, 8), (8, 3)])
def test_pairs_of_heads_beyond_4_gib(oracle_mod, heads, deg):
    from fused3s_amd import capi
    print("case wide pairs heads=%d deg=%d" % (heads, deg), flush=True)
    N, d, pitch = 33_003, 32, (1 << 16) + 8
    assert capi.lib().f3s_attention_uses_wide_offsets(N, pitch * 2, 1) == 1
    rng = np.random.default_rng(deg)
    pre, (rwo, order, atox, bm) = on_gpu(oracle_mod, *random_csr(rng, N, deg, hub=1999), N)
    assert (pre["blockCount"] * (heads // 2) >= (100_000 if heads == 2 else 50_000)) == (deg != 3)
    g = torch.Generator().manual_seed(heads)
    store = torch.empty((N, pitch), dtype=torch.float16, device="cuda")
    Q, K, V = [store[:, at:at + heads * d].unflatten(1, (heads, d)) for at in (8, 1024, pitch - heads * d)]
    for t in (Q, K, V):
        t.copy_(torch.randn((N, heads, d), generator=g).half())
    scale = float(np.sqrt(d))
    got = capi.attention_heads(rwo, order, atox, bm, N, Q, K, V, scale)
    one = [capi.attention_heads(rwo, order, atox, bm, N, *[t[:, h:h + 1] for t in (Q, K, V)], scale)
           for h in range(heads)]
    assert torch.equal(got, torch.cat(one, dim=1))
    check(oracle_mod, pre, N, heads, d, Q, K, V, got)


# 1025 windows: one more than a whole number of chunks for every number of head groups
@pytest.mark.parametrize("heads,d", [(1, 32), (3, 64), (4, 64), (8, 32), (2, 128)])
def test_short_windows(oracle_mod, heads, d):
    from fused3s_amd import capi
    N = 16 * 1024 + 3
    print("case short split heads=%d d=%d" % (heads, d), flush=True)
    rng = np.random.default_rng(heads + d)
    deg = rng.poisson(2.0, N)
    deg[::1999] = 700  # windows for the team of waves
    rowPtr = np.zeros(N + 1, np.int32)
    rowPtr[1:] = np.cumsum(deg)
    colIdx = np.concatenate([np.sort(rng.choice(N, size=k, replace=False)) for k in deg]
                            ).astype(np.int32)
    pre, (rwo, order, atox, bm) = on_gpu(oracle_mod, rowPtr, colIdx, N)
    g = torch.Generator().manual_seed(d)
    Q, K, V = [torch.randn((N, heads, d), generator=g).half().cuda() for _ in range(3)]
    got = capi.attention_heads(rwo, order, atox, bm, N, Q, K, V, float(np.sqrt(d)))
    check(oracle_mod, pre, N, heads, d, Q, K, V, got)
