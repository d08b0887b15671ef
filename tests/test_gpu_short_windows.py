"""Graphs of short windows: one launch computes the short windows by waves and the long ones by
workgroups. Checked against the reference-emulating oracle for fp16 and bf16, single head and
multi-head, with the heavy-first order, a shuffled order (where its first window is short, the short ones
are then taken in natural order) and without an order (a workgroup for every window)."""
import numpy as np
import pytest
import torch

from conftest import random_csr

pytestmark = pytest.mark.gpu
MAX_ABS = 2e-2
MEAN_REL = {torch.float16: 1e-3, torch.bfloat16: 1e-3}


def bits(t):
    t = t.contiguous().cpu()
    if t.dtype == torch.float16:
        return t.numpy()
    return t.view(torch.int16).numpy().view(np.uint16)


def sparse_graph_with_a_few_long_windows(seed, N=20000):
    """~1 edge per row (3-4 TC blocks per window) plus hub rows every 2003 rows whose windows
    have far more than 32 blocks."""
    rng = np.random.default_rng(seed)
    deg = rng.poisson(1.0, N)
    deg[::2003] = 900
    deg[1600:1616] = 0  # one empty window
    rowPtr = np.zeros(N + 1, np.int32)
    rowPtr[1:] = np.cumsum(deg)
    colIdx = np.concatenate([np.sort(rng.choice(N, size=k, replace=False)) for k in deg]
                            ).astype(np.int32)
    return rowPtr, colIdx


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("d", [32, 64, 128])
def test_split_single_head(oracle_mod, dtype, d):
    from fused3s_amd import capi
    print("case short_windows single %s d=%d" % (dtype, d), flush=True)
    N = 20000
    rowPtr, colIdx = sparse_graph_with_a_few_long_windows(d)
    pre = oracle_mod.preprocess(rowPtr, colIdx, N)
    counts = np.diff(pre["rowWindowOffset"])
    nRW = len(counts)
    # the split is taken (short on average), and there are long and empty windows
    assert nRW >= 1024 and counts.sum() < 16 * nRW and counts.max() > 32 and counts.min() == 0
    g = torch.Generator().manual_seed(d)
    Q, K, V = [torch.randn((N, d), generator=g).to(dtype) for _ in range(3)]
    scale = float(np.sqrt(d))
    want = oracle_mod.attention_ref(pre["rowWindowOffset"], pre["sparseAToXidx"], pre["tcbBitMap"],
                                    N, bits(Q), bits(K), bits(V), scale,
                                    dtype=0 if dtype == torch.float16 else 1)
    dev = "cuda"
    rwo = torch.as_tensor(pre["rowWindowOffset"].astype(np.int32)).to(dev)
    atox = torch.as_tensor(pre["sparseAToXidx"].astype(np.int32)).to(dev)
    bm = torch.as_tensor(pre["tcbBitMap"].view(np.int64)).to(dev).view(torch.uint64)
    heavy_first = torch.as_tensor(pre["sortedRowWindows"].astype(np.int32)).to(dev)
    shuffled = heavy_first[torch.randperm(nRW, generator=g).to(dev)].contiguous()
    Qd, Kd, Vd = Q.to(dev), K.to(dev), V.to(dev)
    outs = {}
    for name, order in (("heavy_first", heavy_first), ("shuffled", shuffled), ("natural", None)):
        out = torch.full((N, d), float("nan"), dtype=torch.float32, device=dev)
        capi.attention(rwo, order, atox, bm, N, Qd, Kd, Vd, scale, out=out)
        torch.cuda.synchronize()
        got = out.cpu().numpy()
        assert np.isfinite(got).all(), name  # every row written exactly by one of the kernels
        assert np.abs(got - want).max() < MAX_ABS, name
        assert np.abs(got - want).mean() / np.abs(want).mean() < MEAN_REL[dtype], name
        outs[name] = got
    # without softmax (fp16 only: the bf16 rounding of raw scores is covered elsewhere)
    if dtype == torch.float16:
        want_n = oracle_mod.attention_ref(pre["rowWindowOffset"], pre["sparseAToXidx"],
                                          pre["tcbBitMap"], N, bits(Q), bits(K), bits(V), 1.0,
                                          applySoftmax=False)
        got_n = capi.attention(rwo, heavy_first, atox, bm, N, Qd, Kd, Vd, 1.0, False).cpu().numpy()
        assert np.abs(got_n - want_n).max() < 2e-2 * max(1.0, np.abs(want_n).max())


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_split_multi_head_equals_per_head(oracle_mod, dtype):
    from fused3s_amd import capi
    print("case short_windows heads %s" % dtype, flush=True)
    N, heads, d = 20000, 3, 32
    rowPtr, colIdx = sparse_graph_with_a_few_long_windows(7)
    pre = oracle_mod.preprocess(rowPtr, colIdx, N)
    dev = "cuda"
    rwo = torch.as_tensor(pre["rowWindowOffset"].astype(np.int32)).to(dev)
    atox = torch.as_tensor(pre["sparseAToXidx"].astype(np.int32)).to(dev)
    bm = torch.as_tensor(pre["tcbBitMap"].view(np.int64)).to(dev).view(torch.uint64)
    order = torch.as_tensor(pre["sortedRowWindows"].astype(np.int32)).to(dev)
    g = torch.Generator().manual_seed(1)
    Q, K, V = [(torch.randn((N, heads, d), generator=g) * d ** -0.25).to(dtype).to(dev)
               for _ in range(3)]
    scale = float(np.sqrt(d))
    out = torch.full((N, heads * d), float("nan"), dtype=torch.float32, device=dev)
    capi.attention_heads(rwo, order, atox, bm, N, Q, K, V, scale, out=out)
    torch.cuda.synchronize()
    assert bool(torch.isfinite(out).all())
    for h in range(heads):
        qh, kh, vh = (x[:, h].contiguous() for x in (Q, K, V))
        single = capi.attention(rwo, order, atox, bm, N, qh, kh, vh, scale)
        assert torch.equal(out[:, h * d:(h + 1) * d], single), "head %d" % h
        want = oracle_mod.attention_ref(pre["rowWindowOffset"], pre["sparseAToXidx"],
                                        pre["tcbBitMap"], N, bits(qh), bits(kh), bits(vh), scale,
                                        dtype=0 if dtype == torch.float16 else 1)
        got = single.cpu().numpy()
        assert np.abs(got - want).max() < MAX_ABS
        assert np.abs(got - want).mean() / np.abs(want).mean() < MEAN_REL[dtype]


def test_many_long_units_per_workgroup(oracle_mod):
    """More long (window, pair of heads) units than the long-window launch has workgroups (512): its
    workgroups find several units each and compute them one after the other. 40 000 rows, one
    edge per row on average, 310 windows whose rows name 40 columns each; eight heads."""
    from fused3s_amd import capi
    print("case short_windows many long units", flush=True)
    N, heads, d = 40000, 8, 32
    rng = np.random.default_rng(11)
    deg = rng.poisson(1.0, N)
    for w in range(0, N // 16, 8)[:310]:
        deg[16 * w:16 * w + 16] = 40
    rowPtr = np.zeros(N + 1, np.int32)
    rowPtr[1:] = np.cumsum(deg)
    colIdx = np.concatenate([np.sort(rng.choice(N, size=k, replace=False)) for k in deg]
                            ).astype(np.int32)
    pre = oracle_mod.preprocess(rowPtr, colIdx, N)
    counts = np.diff(pre["rowWindowOffset"])
    nRW = len(counts)
    assert nRW >= 1024 and counts.sum() < 16 * nRW        # the split is taken
    assert (counts > 32).sum() * heads > 2 * 1024          # two long units per workgroup and more
    dev = "cuda"
    rwo = torch.as_tensor(pre["rowWindowOffset"].astype(np.int32)).to(dev)
    atox = torch.as_tensor(pre["sparseAToXidx"].astype(np.int32)).to(dev)
    bm = torch.as_tensor(pre["tcbBitMap"].view(np.int64)).to(dev).view(torch.uint64)
    heavy_first = torch.as_tensor(pre["sortedRowWindows"].astype(np.int32)).to(dev)
    g = torch.Generator().manual_seed(3)
    shuffled = heavy_first[torch.randperm(nRW, generator=g).to(dev)].contiguous()
    Q, K, V = [(torch.randn((N, heads, d), generator=g) * d ** -0.25).to(torch.bfloat16).to(dev)
               for _ in range(3)]
    scale = float(np.sqrt(d))
    want = [oracle_mod.attention_ref(pre["rowWindowOffset"], pre["sparseAToXidx"],
                                     pre["tcbBitMap"], N, bits(Q[:, h]), bits(K[:, h]),
                                     bits(V[:, h]), scale, dtype=1) for h in range(heads)]
    for name, order in (("heavy_first", heavy_first), ("shuffled", shuffled)):
        out = torch.full((N, heads * d), float("nan"), dtype=torch.float32, device=dev)
        capi.attention_heads(rwo, order, atox, bm, N, Q, K, V, scale, out=out)
        torch.cuda.synchronize()
        got = out.cpu().numpy()
        assert np.isfinite(got).all(), name  # every row written by exactly one of the kernels
        for h in range(heads):
            gh = got[:, h * d:(h + 1) * d]
            assert np.abs(gh - want[h]).max() < MAX_ABS, (name, h)
            assert np.abs(gh - want[h]).mean() / np.abs(want[h]).mean() < MEAN_REL[torch.bfloat16]
    # single head through the same launch shape
    q1, k1, v1 = (x[:, 0].contiguous() for x in (Q, K, V))
    out1 = torch.full((N, d), float("nan"), dtype=torch.float32, device=dev)
    capi.attention(rwo, heavy_first, atox, bm, N, q1, k1, v1, scale, out=out1)
    torch.cuda.synchronize()
    assert np.abs(out1.cpu().numpy() - want[0]).max() < MAX_ABS


# A wave per window and a workgroup per long one, at the edges of what decides between them: windows all alike (the
# waves then go by window number), one window just long or just not (32 blocks, or 9/4 of the mean), means on both
# sides of 16 and 32 blocks (of those above 16 the fewest windows are a workgroup's each up to d = 128 with less than
# three heads); four and eight waves to a workgroup, all of a head dimension's forms; 1 024 windows,
# the fewest, and a last one of a single row. Every row is compared with the oracle (fp32 sums of 16-bit
# probabilities), in heavy-first and in shuffled order.
def _structure(rng, nRW, counts):
    N = 16 * nRW - 15
    rwo = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    most = int(counts.max()) * 16
    step = N // most
    atox = np.concatenate([np.arange(16 * c) * step for c in counts])
    atox = (atox + rng.integers(0, step, len(atox))).astype(np.int32)
    bitmap = rng.integers(0, 2**63, len(atox) // 4, dtype=np.uint64)
    bitmap &= rng.integers(0, 2**63, len(bitmap), dtype=np.uint64)
    return N, dict(rowWindowOffset=rwo, sparseAToXidx=atox, tcbBitMap=bitmap)


@pytest.mark.parametrize("heads,d,dtype", [
    (1, 32, torch.float16), (1, 64, torch.bfloat16), (4, 64, torch.float16), (2, 32, torch.bfloat16),
    (8, 32, torch.float16), (1, 96, torch.float16), (3, 128, torch.bfloat16), (1, 192, torch.float16)])
@pytest.mark.parametrize("kind", ["alike", "one_not_long", "one_long", "many_long", "mean_30"])
def test_waves_and_teams(oracle_mod, kind, heads, d, dtype):
    from fused3s_amd import capi
    print("case waves and teams %s %dx%d %s" % (kind, heads, d, dtype), flush=True)
    rng = np.random.default_rng(heads * d)
    nRW = 1024 + (7 if heads == 1 else 0)
    counts = rng.integers(0, 6, nRW)
    if kind == "one_not_long":
        counts[700] = 32
    elif kind == "one_long":
        counts[700] = 33
    elif kind == "many_long":
        counts[::9] = 34 + np.arange(len(counts[::9])) % 9
    elif kind == "mean_30":
        counts[:] = 28 + counts % 4
        counts[11::50] = 69  # 9/4 of the mean and a block more
    N, pre = _structure(rng, nRW, counts)
    dev = lambda a: torch.as_tensor(a).cuda()
    rwo, atox, bm = dev(pre["rowWindowOffset"]), dev(pre["sparseAToXidx"]), dev(
        pre["tcbBitMap"].view(np.int64)).view(torch.uint64)
    heavy = np.argsort(-counts, kind="stable").astype(np.int32)
    g = torch.Generator().manual_seed(d)
    Q, K, V = [(torch.randn((N, heads, d), generator=g) * d ** -0.25).to(dtype).cuda() for _ in range(3)]
    scale = float(np.sqrt(d))
    outs = []
    for order in (heavy, rng.permutation(heavy)):
        out = torch.full((N, heads * d), float("nan"), device="cuda")
        capi.attention_heads(rwo, dev(order), atox, bm, N, Q, K, V, scale, out=out)
        outs.append(out.cpu().numpy())
    for h in range(heads):
        want = oracle_mod.attention_ref(pre["rowWindowOffset"], pre["sparseAToXidx"], pre["tcbBitMap"], N,
                                        bits(Q[:, h]), bits(K[:, h]), bits(V[:, h]), scale,
                                        dtype=0 if dtype == torch.float16 else 1)
        for got in outs:
            gh = got[:, h * d:(h + 1) * d]
            assert np.isfinite(gh).all()
            assert np.abs(gh - want).max() < MAX_ABS
            assert np.abs(gh - want).mean() / np.abs(want).mean() < MEAN_REL[dtype]


@pytest.mark.parametrize("d,nRW", [(64, 5632), (64, 1030), (128, 2816), (128, 1030), (160, 1030)])
@pytest.mark.parametrize("longest", [9, 65])
def test_waves_and_teams_of_narrow_blocks(oracle_mod, longest, d, nRW):
    """16x8 blocks with their scores: odd block counts, so that windows and their shared runs end inside a
    step; `longest` 9: windows all alike, 65: one window of one block more than a wave takes. Up to d = 128
    1030 windows are a workgroup's each."""
    from fused3s_amd import capi
    print("case waves and teams 16x8 longest=%d d=%d windows=%d" % (longest, d, nRW), flush=True)
    rng = np.random.default_rng(d + longest)
    counts = rng.integers(0, 10, nRW)
    counts[5::400] = longest
    N = 16 * nRW - 3
    rwo = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    step = N // (8 * 65)
    atox = np.concatenate([np.arange(8 * c) * step for c in counts])
    atox = (atox + rng.integers(0, step, len(atox))).astype(np.int32)
    bitmap = rng.integers(0, 2**63, len(atox) // 4, dtype=np.uint64)
    bitmap &= rng.integers(0, 2**63, len(bitmap), dtype=np.uint64)
    g = torch.Generator().manual_seed(d)
    Q, K, V = [(torch.randn((N, d), generator=g) * d ** -0.5).half() for _ in range(3)]
    want, scores = oracle_mod.attention_tcb8(rwo, atox, bitmap, N, Q.numpy(), K.numpy(), V.numpy(),
                                             save_sddmm=True)
    order = np.argsort(-counts, kind="stable").astype(np.int32)
    got, got_scores = capi.attention_tcb8(
        torch.as_tensor(rwo).cuda(), torch.as_tensor(order).cuda(), torch.as_tensor(atox).cuda(),
        torch.as_tensor(bitmap.view(np.int64)).cuda().view(torch.uint64), N, Q.cuda(), K.cuda(), V.cuda(),
        save_sddmm=True)
    got, got_scores = got.cpu().numpy(), got_scores.cpu().numpy()
    assert np.isfinite(got).all()
    assert np.abs(got - want).max() < MAX_ABS
    assert np.abs(got_scores.reshape(-1) - np.asarray(scores).reshape(-1)).max() < 2e-2


# Offsets that do not belong to the structure: a window whose end lies so far in front of its begin that the
# difference of the two does not fit 32 bits is empty, and so is the one that begins there
@pytest.mark.parametrize("heads", [1, 4])
def test_ends_far_in_front_of_begins(heads):
    from fused3s_amd import capi
    print("case ends far in front of begins heads=%d" % heads, flush=True)
    rng = np.random.default_rng(heads)
    nRW, d = 1030, 64
    counts = rng.integers(1, 6, nRW)
    counts[::90] = 40
    N, pre = _structure(rng, nRW, counts)
    dev = lambda a: torch.as_tensor(a).cuda()
    atox, bm = dev(pre["sparseAToXidx"]), dev(pre["tcbBitMap"].view(np.int64)).view(torch.uint64)
    order = dev(np.argsort(-counts, kind="stable").astype(np.int32))
    g = torch.Generator().manual_seed(heads)
    Q, K, V = [torch.randn((N, heads, d), generator=g).half().cuda() for _ in range(3)]
    whole = capi.attention_heads(dev(pre["rowWindowOffset"]), order, atox, bm, N, Q, K, V, 8.0)
    rwo = pre["rowWindowOffset"].copy()
    bad = [89, 200, 359, 1000]  # 89 and 359 in front of long windows
    rwo[np.array(bad) + 1] = [-2**31, -2**31 + 7, -2**31 + 1, -2**31 + 1000]
    got = capi.attention_heads(dev(rwo), order, atox, bm, N, Q, K, V, 8.0)
    torch.cuda.synchronize()
    rows = torch.zeros(16 * nRW, dtype=torch.bool, device="cuda")
    for w in bad:
        rows[16 * w:16 * w + 32] = True
    rows = rows[:N]
    assert not got[rows].any()
    assert torch.equal(got[~rows], whole[~rows])


# A long window is a workgroup's whatever the order: its rows come out as in heavy-first order, bit for bit, where
# the order begins with a short window, where it begins with a long one and has others at its very end, and where
# it is natural; above d = 128 and for pairs of heads a workgroup has four runs, else eight, in one turn or two
@pytest.mark.parametrize("heads,d", [(1, 32), (1, 64), (4, 64), (2, 128), (8, 32), (1, 160), (3, 224)])
def test_long_windows_of_any_order(heads, d):
    from fused3s_amd import capi
    print("case long windows of any order %dx%d" % (heads, d), flush=True)
    rng = np.random.default_rng(heads * d)
    nRW = 1100
    counts = rng.integers(0, 6, nRW)
    counts[np.concatenate([[7, 8], np.arange(20, nRW, 83), [nRW - 1]])] = 34 + rng.integers(0, 40)
    N, pre = _structure(rng, nRW, counts)
    dev = lambda a: torch.as_tensor(a).cuda()
    args = dev(pre["rowWindowOffset"]), dev(pre["sparseAToXidx"]), dev(pre["tcbBitMap"].view(np.int64)).view(torch.uint64)
    g = torch.Generator().manual_seed(d)
    Q, K, V = [torch.randn((N, heads, d), generator=g).to(torch.bfloat16).cuda() for _ in range(3)]

    def call(order):
        out = torch.full((N, heads * d), float("nan"), device="cuda")
        return capi.attention_heads(args[0], dev(order.astype(np.int32)), *args[1:], N, Q, K, V, d ** 0.5, out=out)

    heavy = np.argsort(-counts, kind="stable")
    want = call(heavy)
    assert torch.isfinite(want).all()
    longFirst = rng.permutation(heavy[1:])
    ends = np.concatenate([[heavy[0]], longFirst[counts[longFirst] <= 33], longFirst[counts[longFirst] > 33]])
    orders = [np.arange(nRW), heavy[::-1], rng.permutation(heavy), ends]
    assert [counts[o[0]] > 33 for o in orders] == [False, False, counts[orders[2][0]] > 33, True]
    assert counts[ends[counts.sum() // 33 + 1:]].max() > 33  # beyond as many positions as can be long ones
    for k, order in enumerate(orders):
        assert torch.equal(call(order), want), k


# An order that names some of the windows and is filled up with what is no window, or with one again and again: the
# other windows' rows are left as they are, also where all windows are alike
@pytest.mark.parametrize("fill", [-1, 1 << 30, "last"])
@pytest.mark.parametrize("longest", [7, 60])
def test_filled_up_orders(longest, fill):
    from fused3s_amd import capi
    print("case filled up orders longest=%d %s" % (longest, fill), flush=True)
    rng = np.random.default_rng(longest)
    nRW, heads, d = 1050, 4, 64
    counts = 4 + rng.integers(0, 3, nRW)
    counts[333::100] = longest
    N, pre = _structure(rng, nRW, counts)
    dev = lambda a: torch.as_tensor(a).cuda()
    args = dev(pre["rowWindowOffset"]), dev(pre["sparseAToXidx"]), dev(pre["tcbBitMap"].view(np.int64)).view(torch.uint64)
    g = torch.Generator().manual_seed(longest)
    Q, K, V = [torch.randn((N, heads, d), generator=g).half().cuda() for _ in range(3)]
    heavy = np.argsort(-counts, kind="stable").astype(np.int32)
    whole = capi.attention_heads(args[0], dev(heavy), *args[1:], N, Q, K, V, 8.0)
    some = heavy[rng.random(nRW) < 0.4]
    order = np.full(nRW, some[-1] if fill == "last" else fill, np.int32)
    order[:len(some)] = some
    named = np.zeros(nRW, bool)
    named[some] = True
    rows = torch.as_tensor(np.repeat(named, 16)[:N]).cuda()
    out = torch.full((N, heads * d), float("nan"), device="cuda")
    capi.attention_heads(args[0], dev(order), *args[1:], N, Q, K, V, 8.0, out=out)
    assert torch.equal(out[rows], whole[rows])
    assert torch.isnan(out[~rows]).all()


# From 16 blocks a window on, and with 16x8 blocks, what takes a call depends on windows times heads: one window fewer
# than the line and the call is the workgroup-per-window kernel's, bit for bit; at the line it is not, and its rows
# are the same to the rounding of 16-bit probabilities. One pair of 32-wide heads and single ones have no such line.
@pytest.mark.parametrize("heads,d,W,line", [
    (1, 64, 16, 5632), (2, 64, 16, 2816), (3, 64, 16, 1366), (1, 96, 16, 2816), (1, 128, 16, 2816), (2, 128, 16, 1408),
    (4, 32, 16, 2816), (6, 32, 16, 1366), (2, 32, 16, None), (1, 32, 16, None), (1, 256, 16, 1200), (1, 64, 8, 5632),
    (1, 96, 8, 2816), (1, 128, 8, 2816)])
def test_line_in_windows_and_heads(monkeypatch, heads, d, W, line):
    from fused3s_amd import capi
    print("case line in windows and heads %dx%d W=%d" % (heads, d, W), flush=True)
    for nRW, mixed in [(6000, False)] if line is None else [(line - 1, False), (line, True)]:
        rng = np.random.default_rng(nRW)
        counts = 16 + rng.integers(0, 3, nRW)
        counts[5::97] = 70 + rng.integers(0, 9)
        rwo = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
        N = 16 * nRW - 3
        step = N // (W * int(counts.max()))
        atox = np.concatenate([np.arange(W * c) * step for c in counts])
        atox = (atox + rng.integers(0, step, len(atox))).astype(np.int32)
        bitmap = rng.integers(0, 2**63, len(atox) // 4, dtype=np.uint64)
        bitmap &= rng.integers(0, 2**63, len(bitmap), dtype=np.uint64)
        dev = lambda a: torch.as_tensor(a).cuda()
        args = [dev(rwo), dev(np.argsort(-counts, kind="stable").astype(np.int32)), dev(atox),
                dev(bitmap.view(np.int64)).view(torch.uint64), N]
        g = torch.Generator().manual_seed(d)
        args += [(torch.randn((N, heads, d), generator=g) * d ** -0.25).half().cuda() for _ in range(3)]
        if W == 8:
            args[5:] = [t[:, 0].contiguous() for t in args[5:]]
        call = capi.attention_tcb8 if W == 8 else capi.attention_heads
        got = call(*args)
        monkeypatch.setenv("F3S_SHORT_WINDOWS", "0")
        want = call(*args)
        monkeypatch.delenv("F3S_SHORT_WINDOWS")
        assert torch.equal(got, want) != mixed, nRW
        assert (got - want).abs().max().item() < MAX_ABS
        assert ((got - want).abs().mean() / want.abs().mean()).item() < MEAN_REL[torch.float16]


# F3S_WINDOW_PERSISTENT=1 asks for the cursor form of the workgroup-per-window kernel, also where an ordered call of
# 16 blocks a window and more would go to the kernel for short windows
@pytest.mark.parametrize("d,nRW", [(64, 5700), (160, 1100)])
def test_cursor_form_is_asked_for(monkeypatch, d, nRW):
    from fused3s_amd import capi
    print("case cursor form d=%d" % d, flush=True)
    rng = np.random.default_rng(d)
    counts = 16 + rng.integers(0, 5, nRW)
    counts[11::300] = 65
    N, pre = _structure(rng, nRW, counts)
    dev = lambda a: torch.as_tensor(a).cuda()
    args = [dev(pre["rowWindowOffset"]), dev(np.argsort(-counts, kind="stable").astype(np.int32)),
            dev(pre["sparseAToXidx"]), dev(pre["tcbBitMap"].view(np.int64)).view(torch.uint64), N]
    g = torch.Generator().manual_seed(d)
    args += [torch.randn((N, d), generator=g).half().cuda() for _ in range(3)]
    plain = capi.attention(*args, 8.0)
    monkeypatch.setenv("F3S_WINDOW_PERSISTENT", "1")
    cursor = capi.attention(*args, 8.0)
    monkeypatch.setenv("F3S_WINDOW_PERSISTENT", "0")
    monkeypatch.setenv("F3S_SHORT_WINDOWS", "0")
    windows = capi.attention(*args, 8.0)
    assert torch.equal(cursor, windows) and not torch.equal(plain, windows)


# Calls without an order above d = 128 on more windows than an order is made for: the workgroups look for long windows
# in natural order. The rows are those of a call in heavy-first order.
@pytest.mark.parametrize("heads,d", [(1, 160), (2, 256)])
def test_many_windows_without_an_order(heads, d):
    from fused3s_amd import capi
    print("case many windows without an order %dx%d" % (heads, d), flush=True)
    rng = np.random.default_rng(d)
    nRW = 16_385
    counts = rng.integers(0, 5, nRW)
    counts[np.array([0, 3, 7000, 7001, nRW - 1])] = [33, 40, 64, 34, 51]
    N, pre = _structure(rng, nRW, counts)
    dev = lambda a: torch.as_tensor(a).cuda()
    rwo, atox, bm = dev(pre["rowWindowOffset"]), dev(pre["sparseAToXidx"]), dev(
        pre["tcbBitMap"].view(np.int64)).view(torch.uint64)
    order = dev(np.argsort(-counts, kind="stable").astype(np.int32))
    g = torch.Generator(device="cuda").manual_seed(d)
    Q, K, V = [torch.randn((N, heads, d), generator=g, device="cuda").bfloat16() for _ in range(3)]
    outs = []
    for o in (None, order):
        out = torch.full((N, heads * d), float("nan"), device="cuda")
        outs.append(capi.attention_heads(rwo, o, atox, bm, N, Q, K, V, d ** 0.5, out=out))
    assert torch.isfinite(outs[0]).all() and torch.equal(*outs)
    if heads == 1:
        assert torch.equal(capi.attention(rwo, None, atox, bm, N, *[t[:, 0].contiguous() for t in (Q, K, V)], d ** 0.5),
                           outs[0])


# The forms of a single head of 96 and 128: eight waves to a workgroup, and four that take the same eight runs in two
# turns, from 500 000 blocks on or with three heads. A head's rows are the same in all of them; those of the
# window kernel differ by the rounding of 16-bit probabilities.
@pytest.mark.parametrize("W", [16, 8])
@pytest.mark.parametrize("d,nRW,mean", [(96, 2900, 17), (128, 2900, 17), (96, 17_000, 30), (128, 17_000, 30)])
def test_eight_and_four_waves_of_single_heads(monkeypatch, d, nRW, mean, W):
    from fused3s_amd import capi
    print("case eight and four waves W=%d d=%d windows=%d" % (W, d, nRW), flush=True)
    rng = np.random.default_rng(d + W)
    counts = mean * (16 // W) - 1 + rng.integers(0, 3, nRW)
    counts[::nRW // 17] = 140 + rng.integers(0, 60)
    assert (counts.sum() * W // 16 >= 500_000) == (nRW > 10_000)
    rwo = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    N = 16 * nRW - 9
    step = N // (W * int(counts.max()))
    atox = (np.arange(rwo[-1] * W) - np.repeat(rwo[:-1] * W, counts * W)) * step + rng.integers(0, step, rwo[-1] * W)
    bits = [rng.integers(0, 2**63, len(atox) // 4) for _ in range(2)]
    dev = lambda a: torch.as_tensor(a).cuda()
    args = [dev(rwo), dev(np.argsort(-counts, kind="stable").astype(np.int32)), dev(atox.astype(np.int32)),
            dev(bits[0] & bits[1]).view(torch.uint64), N]
    g = torch.Generator(device="cuda").manual_seed(d)
    Q, K, V = [(torch.randn((N, 3, d), generator=g, device="cuda") * d ** -0.25).half() for _ in range(3)]
    one = [t[:, 1].contiguous() for t in (Q, K, V)]
    call = capi.attention if W == 16 else capi.attention_tcb8
    got = call(*args, *one)
    monkeypatch.setenv("F3S_SHORT_WINDOWS", "0")
    want = call(*args, *one)
    monkeypatch.delenv("F3S_SHORT_WINDOWS")
    assert not torch.equal(got, want) and (got - want).abs().max().item() < MAX_ABS
    assert ((got - want).abs().mean() / want.abs().mean()).item() < MEAN_REL[torch.float16]
    if W == 16:
        assert torch.equal(capi.attention_heads(*args, Q, K, V)[:, d:2 * d], got)
