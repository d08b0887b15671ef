"""The work that users of fused3s_amd have it do, as cases that can be timed.

Two things are asked of the framework: the TC-block structure of a graph (once per graph) and
attention over that structure (once per layer and step). A case is one call of either, through
the `F3S` operator module or, where a serving program keeps its own workspace, through
fused3s_amd.capi. Graphs are the synthetic families of fused3s_amd.synth at the sizes of its
configurations, of the tests, and between them.

  op      structure   F3S.preprocess_gpu
          attend      F3S.f3s_1tb1rw* on one head (`call` says which one)
          blocks8     F3S.f3s_1tb1tcb on 16x8 blocks
          layer       multi-head attention, F3S.f3s_multihead_scaleQK (`api` = "module") or
                      capi.attention_heads on a prepared workspace (`api` = "capi")
  graph   gnm, rmat, chunglu, sbm with N nodes and about E directed edges
"""
import math

import torch

from fused3s_amd import F3S, capi, synth

DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16}
SBM_CLUSTER = 200  # nodes per community of the sbm graphs
SBM_P_OUT = 1e-5


def listed():
    return [
        # a citation-sized graph, as in examples, tests and small-graph inference: latency of a call
        dict(name="structure_tiny", op="structure", graph="gnm", N=2708, E=23864, W=16),
        dict(name="attend_tiny", op="attend", call="scaleQK", graph="gnm", N=2708, E=23864, d=64,
             dtype="fp16"),
        # a mid-sized skewed graph: the ordinary case of both calls
        dict(name="structure_medium", op="structure", graph="rmat", N=169343, E=2795000, W=16),
        dict(name="attend_medium", op="attend", call="scaleQK", graph="rmat", N=169343, E=2795000,
             d=64, dtype="fp16"),
        # the 16x8 operator with its score output, which the accuracy harness compares (d = 128)
        dict(name="blocks8_scores", op="blocks8", graph="rmat", N=65521, E=1310000, d=128,
             dtype="fp16", sddmm=True),
        # a graph-transformer layer on a community graph: short windows, many heads
        dict(name="layer_communities", op="layer", api="module", graph="sbm", N=100000, E=591712,
             heads=8, d=32, dtype="bf16"),
        # ragged sizes in natural window order without softmax, a head dimension between powers of two
        dict(name="attend_ragged", op="attend", call="natural_no_softmax", graph="chunglu",
             N=50021, E=4100000, d=96, dtype="bf16"),
        # a layer on a graph of long windows in a serving loop that keeps its workspace
        dict(name="layer_long", op="layer", api="capi", graph="chunglu", N=60013, E=18000000,
             heads=4, d=64, dtype="bf16"),
        # the dense power-law graph of the headline benchmark
        dict(name="structure_large", op="structure", graph="chunglu", N=232965, E=114600000, W=16),
        dict(name="attend_large", op="attend", call="scaleQK", graph="chunglu", N=232965,
             E=114600000, d=64, dtype="fp16"),
        # a very large sparse graph: the most nodes, K and V far beyond the caches
        dict(name="structure_huge", op="structure", graph="rmat_flat", N=2449029, E=61430000, W=16),
        dict(name="attend_huge", op="attend", call="scaleQK", graph="rmat_flat", N=2449029,
             E=61430000, d=128, dtype="fp16"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_graph(rng, kinds):
    kind = rng.choice(kinds)
    if kind == "gnm":  # small and uniform
        N = _log_int(rng, 700, 30000)
        return dict(graph=kind, N=N, E=N + 2 * int(N * rng.uniform(2, 10)))
    if kind in ("rmat", "rmat_flat"):  # skewed, few edges per row
        N = _log_int(rng, 20000, 2000000)
        return dict(graph=kind, N=N, E=int(N * rng.uniform(9, 28)))
    if kind == "chunglu":  # long rows
        N = _log_int(rng, 12000, 200000)
        return dict(graph=kind, N=N, E=N * _log_int(rng, 50, 480))
    N = _log_int(rng, 15000, 200000)  # sbm: communities
    N -= N % SBM_CLUSTER
    p_in = rng.uniform(0.02, 0.2)
    return dict(graph="sbm", N=N, E=int(N * (1 + 0.93 * SBM_CLUSTER * p_in + N * SBM_P_OUT)))


def draw(rng):
    op = rng.choice(["structure", "structure", "attend", "attend", "attend", "layer", "layer",
                     "blocks8"])
    if op == "structure":
        case = _draw_graph(rng, ["gnm", "rmat", "rmat_flat", "chunglu", "sbm"])
        return dict(op=op, W=rng.choice([16, 16, 16, 8]), **case)
    if op == "blocks8":
        case = _draw_graph(rng, ["gnm", "rmat"])
        N = min(case["N"], 150000)
        case.update(N=N, E=case["E"] * N // case["N"])
        return dict(op=op, d=rng.choice([32, 64, 64, 128, 128]), dtype="fp16",
                    sddmm=rng.choice([True, False]), **case)
    if op == "layer":
        case = _draw_graph(rng, ["gnm", "rmat", "chunglu", "sbm", "sbm"])
        heads, d = rng.choice([(2, 64), (4, 32), (4, 64), (8, 32), (8, 64), (4, 128)])
        extra = dict(op=op, api=rng.choice(["module", "capi"]), heads=heads)
    else:
        case = _draw_graph(rng, ["gnm", "rmat", "rmat", "rmat_flat", "chunglu", "chunglu"])
        heads, d = 1, rng.choice([32, 64, 64, 64, 96, 128, 128, 128, 160, 192, 224, 256])
        extra = dict(op=op, call=rng.choice(["scaleQK", "scaleQK", "scaleQK", "permuteV",
                                             "scheduled", "natural", "natural_no_softmax"]))
    # no more than the largest listed case: neither in rows nor in edges times width
    shrink = min(1.0, 2449029 * 128 / (case["N"] * heads * d), 61430000 * 128 / (case["E"] * heads * d))
    if shrink < 1.0:
        N = int(case["N"] * shrink)
        if case["graph"] == "sbm":
            N -= N % SBM_CLUSTER
        case.update(N=N, E=int(case["E"] * N / case["N"]))
    return dict(extra, d=d, dtype=rng.choice(["fp16", "bf16"]), **case)


# ---------------------------------------------------------------------------------- preparation
def _base_graph(case):
    N, E, dev = case["N"], case["E"], "cuda"
    if case["graph"] == "gnm":
        return synth.gnm_graph(N, (E - N) // 2, 0, dev)
    if case["graph"] == "rmat":
        return synth.rmat_graph(N, E, 0.57, 0.19, 0.19, 0, dev)
    if case["graph"] == "rmat_flat":
        return synth.rmat_graph(N, E, 0.45, 0.22, 0.22, 0, dev)
    if case["graph"] == "chunglu":
        return synth.chung_lu_graph(N, E, 2.1, min(26000, N // 8), 0, dev)
    # the density inside the communities follows from the edge count (pairs drawn twice collapse)
    return synth.sbm_graph(N, N // SBM_CLUSTER, _sbm_p_in(case), SBM_P_OUT, 0, dev)


def _graph(case, seed):
    """The case's graph with its nodes renamed by the seed: groups of 16 nodes (one row window) move
    as a whole and are shuffled inside, so that every seed has another CSR with as many edges and
    TC blocks. Communities stay neighbours: their windows are rotated, the others permuted."""
    rowPtr, colIdx = _base_graph(case)
    N, dev = case["N"], colIdx.device
    gen = torch.Generator(device=dev).manual_seed(seed)
    full = N // 16
    if case["graph"] == "sbm":
        turn = torch.randint(1, max(2, full), (1,), generator=gen, device=dev)
        window = (torch.arange(full, device=dev) + turn) % max(1, full)
    else:
        window = torch.randperm(full, generator=gen, device=dev)
    inside = torch.rand((full, 16), generator=gen, device=dev).argsort(dim=1)
    name = torch.arange(N, device=dev)
    name[:16 * full] = (window[:, None] * 16 + inside).flatten()
    rows = torch.repeat_interleave(name, (rowPtr[1:] - rowPtr[:-1]).long())
    key = torch.sort(rows * N + name[colIdx.long()]).values
    rows = torch.div(key, N, rounding_mode="floor")
    colIdx = (key - rows * N).to(torch.int32)
    rowPtr = torch.zeros(N + 1, dtype=torch.int64, device=dev)
    rowPtr[1:] = torch.cumsum(torch.bincount(rows, minlength=N), 0)
    return rowPtr.to(torch.int32), colIdx


def _sbm_p_in(case):
    return min(0.5, (case["E"] / case["N"] - 1 - case["N"] * SBM_P_OUT) / (0.93 * SBM_CLUSTER))


def _edge_buffers(rowPtr, colIdx):
    dev, nRW, E = colIdx.device, (rowPtr.numel() + 14) // 16, colIdx.numel()
    return [torch.zeros(n, dtype=torch.int32, device=dev) for n in (nRW, E, E)]


def prepare(case, seed):
    rowPtr, colIdx = _graph(case, seed)
    N = case["N"]
    state = dict(case=case, N=N, rowPtr=rowPtr, colIdx=colIdx)
    if case["op"] == "structure":
        state["buffers"] = _edge_buffers(rowPtr, colIdx)
        return state
    W = 8 if case["op"] == "blocks8" else 16
    rwo, order, _, _, _, atox, bitmap, _ = F3S.preprocess_gpu(
        colIdx, rowPtr, N, 16, W, *_edge_buffers(rowPtr, colIdx))
    state.update(rwo=rwo, order=order, atox=atox, bitmap=bitmap)
    d, heads, dtype = case["d"], case.get("heads", 1), DTYPES[case["dtype"]]
    shape = (N, heads, d) if case["op"] == "layer" else (N, d)
    gen = torch.Generator(device="cuda").manual_seed(seed)
    scaled = case["op"] == "layer" or case.get("call") == "scaleQK"
    for name in "QKV":
        if scaled:  # normalised features, scores divided by sqrt(d)
            x = torch.randn(shape, generator=gen, device="cuda") * (d ** -0.5 if heads > 1 else 1.0)
        else:  # the unscaled calls are used on features in [0, 1)
            x = torch.rand(shape, generator=gen, device="cuda")
        state[name] = x.to(dtype)
    if case.get("api") == "capi":
        ws = capi.attention_workspace(N, d, "cuda", nTCB=atox.numel() // 16, dtype=dtype,
                                      heads=heads)
        if ws is not None:
            capi.attention_prepare(rwo, atox, N, d, ws, heads=heads)
        state["workspace"] = ws
    return state


# ------------------------------------------------------------------------------------- one pass
def run(state):
    case, N = state["case"], state["N"]
    if case["op"] == "structure":
        made = F3S.preprocess_gpu(state["colIdx"], state["rowPtr"], N, 16, case["W"],
                                  *state["buffers"])
        rwo, order, rowid, tile, toff, atox, bitmap, blocks = made
        return [rwo, order, rowid, tile, toff, atox, bitmap.view(torch.int64), blocks,
                *state["buffers"]]
    rwo, order, atox, bitmap = state["rwo"], state["order"], state["atox"], state["bitmap"]
    Q, K, V = state["Q"], state["K"], state["V"]
    if case["op"] == "blocks8":
        _, out, scores = F3S.f3s_1tb1tcb(rwo, atox, bitmap, N, Q, K, V, True, case["sddmm"])
        return [out, scores] if case["sddmm"] else out
    scale = math.sqrt(case["d"])
    if case["op"] == "layer":
        if case["api"] == "module":
            return F3S.f3s_multihead_scaleQK(rwo, order, atox, bitmap, N, Q, K, V, scale)[1]
        ws = state["workspace"]
        return capi.attention_heads(rwo, order, atox, bitmap, N, Q, K, V, scale, workspace=ws,
                                    prepared=ws is not None)
    call = case["call"]
    if call == "scaleQK":
        return F3S.f3s_1tb1rw_scheduled_permuteV_scaleQK(rwo, order, atox, bitmap, N, Q, K, V,
                                                         scale, 8)[1]
    if call == "permuteV":
        return F3S.f3s_1tb1rw_scheduled_permuteV(rwo, order, atox, bitmap, N, Q, K, V, 8)[1]
    if call == "scheduled":
        return F3S.f3s_1tb1rw_scheduled(rwo, order, atox, bitmap, N, Q, K, V, 8, False)[1]
    return F3S.f3s_1tb1rw(rwo, atox, bitmap, N, Q, K, V, 8, call == "natural", False)[1]


# ------------------------------------------------------------------------------- work, tolerance
def _blocks(case, W):
    """TC blocks of the graph, near enough: a window's distinct columns over W, the last one half
    full. The skewed families repeat few columns inside a window, the communities many."""
    N, E = case["N"], case["E"]
    nRW = (N + 15) // 16
    columns = E
    if case["graph"] == "sbm":
        columns = nRW * (SBM_CLUSTER * (1 - (1 - _sbm_p_in(case)) ** 16) +
                         N * (1 - (1 - SBM_P_OUT) ** 16))
    return columns / W + nRW / 2


def work(case):
    N, E = case["N"], case["E"]
    nRW = (N + 15) // 16
    W = 8 if case["op"] == "blocks8" else case.get("W", 16)
    blocks = _blocks(case, W)
    per_block = 4 * W + 2 * W  # column ids and bitmap
    if case["op"] == "structure":
        # row pointers and columns in; rank and row of every edge, tile ids, window arrays and the
        # per-block arrays out
        return {"bytes": 4 * (N + 1) + 4 * E + 9 * E + 12 * nRW + (per_block + 8) * blocks,
                "flops": 0}
    D = case["d"] * case.get("heads", 1)
    size = 3 * 2 * N * D + 4 * N * D + per_block * blocks + 8 * nRW
    if case.get("sddmm"):
        size += 4 * 16 * W * blocks
    return {"bytes": size, "flops": 4 * D * E}


def tolerance(case):
    if case["op"] == "structure":
        return "exact"
    # fp32 sums of products whose probabilities are rounded to 16 bits (fp16, or a bf16 pair)
    return {"rel": 1e-3, "max": 2e-2}
