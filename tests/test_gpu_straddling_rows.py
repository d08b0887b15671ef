"""Head dimensions whose rows begin in one gather instruction and end in the next (96, 160, 192, 224),
with 128 beside them: every element of every row has to arrive at its place in the tile.

Small whole numbers, no softmax: scores of at most 2 d = 448 are exact in 16 bits, sums of at most
700 * 448 * 2 < 2^24 exact in 32, so the results equal those of 64-bit arithmetic bit for bit, whatever
the order of the sums."""
import numpy as np
import pytest
import torch

from conftest import random_csr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("schedule", ["window", "sliced", "resident", "heads", "tcb8"])
@pytest.mark.parametrize("d", [96, 128, 160, 192, 224])
def test_rows_arrive_whole(oracle_mod, monkeypatch, d, schedule):
    from fused3s_amd import capi
    print("case straddling d=%d %s" % (d, schedule), flush=True)
    N = 700  # windows of 1 to about 40 blocks, odd and even, the last of 12 rows
    rng = np.random.default_rng(d)
    rowPtr, colIdx = random_csr(rng, N, 12, hub=501, empty_frac=0.1)
    heads = 2 if schedule == "heads" else 1
    dtype = torch.bfloat16 if schedule in ("heads", "sliced") else torch.float16
    Q = rng.integers(-1, 2, (N, heads, d))
    K, V = rng.integers(-2, 3, (2, N, heads, d))
    A = np.zeros((N, N))
    for r in range(N):
        A[r, colIdx[rowPtr[r]:rowPtr[r + 1]]] = 1
    want = np.stack([(A * (Q[:, h] @ K[:, h].T)) @ V[:, h] for h in range(heads)], 1).reshape(N, heads * d)
    pre = oracle_mod.preprocess(rowPtr, colIdx, N, 16, 8 if schedule == "tcb8" else 16)
    rwo, atox = (torch.as_tensor(pre[k].astype(np.int32)).cuda() for k in ("rowWindowOffset", "sparseAToXidx"))
    bm = torch.as_tensor(pre["tcbBitMap"].view(np.int64)).cuda().view(torch.uint64)
    q, k, v = (torch.as_tensor(t).to(dtype).cuda() for t in (Q, K, V))
    if schedule == "heads":
        got = capi.attention_heads(rwo, None, atox, bm, N, q, k, v, 1.0, False)
    elif schedule == "tcb8":
        got = capi.attention_tcb8(rwo, None, atox, bm, N, q[:, 0].contiguous(), k[:, 0].contiguous(),
                                  v[:, 0].contiguous(), False)
        got = got[0] if isinstance(got, (tuple, list)) else got
    else:
        ws = None
        if schedule != "window":
            monkeypatch.setenv("F3S_SCHEDULE", "sliced")
            monkeypatch.setenv("F3S_SLICED_PERSISTENT", "1" if schedule == "resident" else "0")
            ws = capi.attention_workspace(N, d, "cuda", nTCB=int(pre["blockCount"]), dtype=dtype)
        got = capi.attention(rwo, None, atox, bm, N, q[:, 0].contiguous(), k[:, 0].contiguous(),
                             v[:, 0].contiguous(), 1.0, False, workspace=ws)
    torch.cuda.synchronize()
    assert np.array_equal(got.cpu().numpy().astype(np.float64).reshape(want.shape), want)
