"""Where the workgroup-per-window kernel changes between one ring stage and two at d = 32: graphs of one
TC block fewer than 96 a window and head on average, and of exactly 96, through every entry that runs it;
and long windows of 20 MB of K + V, of one block fewer than 160 a window and of exactly 160."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
N_WINDOWS = 110
N = 16 * N_WINDOWS - 3


def graph(rng, sizes, missing):
    """Windows of sizes[0] and sizes[1] blocks in turn, the last block ragged, `missing` blocks fewer."""
    blocks = np.tile(sizes, N_WINDOWS // 2)
    blocks[7] -= missing
    rows = []
    for b in blocks:
        cols = np.sort(rng.choice(N, size=min(N, int(b) * 16 - 5), replace=False))
        owner = rng.integers(0, 13, len(cols))  # the last window has 13 rows
        rows += [cols[owner == r] for r in range(16)]
    rows = rows[:N]
    rowPtr = np.zeros(N + 1, np.int32)
    rowPtr[1:] = np.cumsum([len(r) for r in rows])
    return rowPtr, np.concatenate(rows).astype(np.int32), int(blocks.sum())


@pytest.mark.parametrize("softmax", [True, False])
@pytest.mark.parametrize("missing", [1, 0])
def test_both_sides_of_the_line(oracle_mod, tmp_path, monkeypatch, missing, softmax):
    from fused3s_amd import F3S, capi
    print("case window team missing=%d softmax=%d" % (missing, softmax), flush=True)
    rng = np.random.default_rng(missing)
    rowPtr, colIdx, total = graph(rng, [110, 82], missing)
    heads, d = 3, 32
    g = torch.Generator().manual_seed(missing)
    # without softmax a row sums about 120 products: features that keep it near 1
    Q, K, V = [(torch.rand((N, heads, d), generator=g) * (1.0 if softmax else 0.1)).half()
               for _ in range(3)]

    def reference(call, pre, h):
        return call(pre["rowWindowOffset"], pre["sparseAToXidx"], pre["tcbBitMap"], N,
                    *[t[:, h].contiguous().numpy() for t in (Q, K, V)], applySoftmax=softmax)

    def close(got, want, what):
        got = got.cpu().numpy()
        assert np.abs(got - want).max() < 2e-2, what
        assert np.abs(got - want).mean() < 1e-3 * np.abs(want).mean(), what

    dev = lambda a: torch.as_tensor(a.astype(np.int32)).cuda()
    words = lambda a: torch.as_tensor(a.view(np.int64)).cuda().view(torch.uint64)
    pre = oracle_mod.preprocess(rowPtr, colIdx, N)
    assert pre["blockCount"] == total == 96 * N_WINDOWS - missing
    rwo, order, atox = [dev(pre[k]) for k in ("rowWindowOffset", "sortedRowWindows", "sparseAToXidx")]
    bm = words(pre["tcbBitMap"])
    one = [t[:, 0].contiguous().cuda() for t in (Q, K, V)]
    want = reference(oracle_mod.attention_ref, pre, 0)
    for o in (order, None):
        close(capi.attention(rwo, o, atox, bm, N, *one, applySoftmax=softmax), want, "one head")
    if softmax:
        monkeypatch.chdir(tmp_path)  # the timed call leaves a file
        close(F3S.f3s_1tb1rw(rwo, atox, bm, N, *one, 8, True, True)[1], want, "timed")
    pre8 = oracle_mod.preprocess(rowPtr, colIdx, N, 16, 8)
    got, scores = capi.attention_tcb8(dev(pre8["rowWindowOffset"]), dev(pre8["sortedRowWindows"]),
                                      dev(pre8["sparseAToXidx"]), words(pre8["tcbBitMap"]), N, *one,
                                      applySoftmax=softmax, save_sddmm=True)
    close(got, reference(oracle_mod.attention_tcb8, pre8, 0), "16x8")
    assert torch.isfinite(scores).all()
    rowPtr, colIdx, total = graph(rng, [50, 14], missing)  # 32 blocks, three heads
    pre = oracle_mod.preprocess(rowPtr, colIdx, N)
    assert 3 * total == 96 * N_WINDOWS - 3 * missing == 3 * pre["blockCount"]
    rwo, order, atox = [dev(pre[k]) for k in ("rowWindowOffset", "sortedRowWindows", "sparseAToXidx")]
    got = capi.attention_heads(rwo, order, atox, words(pre["tcbBitMap"]), N, Q.cuda(), K.cuda(),
                               V.cuda(), applySoftmax=softmax)
    for h in range(heads):
        close(got[:, h * d:(h + 1) * d], reference(oracle_mod.attention_ref, pre, h), "head %d" % h)


# eight heads are computed in pairs, five (K + V of exactly 20 MiB) one by one
@pytest.mark.parametrize("heads", [8, 5])
@pytest.mark.parametrize("missing", [1, 0])
def test_long_windows_of_many_heads(oracle_mod, missing, heads):
    from fused3s_amd import capi
    print("case window team, long windows missing=%d heads=%d" % (missing, heads), flush=True)
    nRW, blocks, d = 2048, 160, 32
    N = 16 * nRW
    rng = np.random.default_rng(missing)
    atox = np.sort(np.argpartition(rng.random((nRW, 4096)), blocks * 16, axis=1)[:, :blocks * 16])
    atox = (atox * 8 + rng.integers(0, 8, atox.shape)).astype(np.int32).reshape(-1)
    bitmap = rng.integers(0, 2**63, nRW * blocks * 4, dtype=np.uint64)
    bitmap &= rng.integers(0, 2**63, len(bitmap), dtype=np.uint64)
    rwo = (np.arange(nRW + 1) * blocks).astype(np.int32)
    rwo[-1] -= missing
    atox, bitmap = atox[:rwo[-1] * 16], bitmap[:rwo[-1] * 4]
    g = torch.Generator().manual_seed(missing)
    Q, K, V = [torch.randn((N, heads, d), generator=g).half() for _ in range(3)]
    dev = lambda a: torch.as_tensor(a).cuda()
    got = capi.attention_heads(dev(rwo), None, dev(atox), dev(bitmap.view(np.int64)).view(torch.uint64),
                               N, Q.cuda(), K.cuda(), V.cuda(), float(np.sqrt(d))).cpu().numpy()
    for h in (0, heads - 1):
        want = oracle_mod.attention_ref(rwo, atox, bitmap, N, *[t[:, h].contiguous().numpy()
                                                                for t in (Q, K, V)], float(np.sqrt(d)))
        assert np.abs(got[:, h * d:(h + 1) * d] - want).max() < 2e-2, h
        assert np.abs(got[:, h * d:(h + 1) * d] - want).mean() < 1e-3 * np.abs(want).mean(), h
