"""The work that users of this engine have it do, as measurable cases.

Every case is a dict of plain values; `kind` names the call:

  static    one static solve of an uploaded graph: "host" arrays (the drop-in's form) or "device" pointers
  dynamic   one dynamic solve (ND, DT, DF, DF-P) of an updated graph from the previous ranks
  update    a batch applied to the resident graph in place, then a DF-P solve; then the inverse batch likewise
  stream    the same two batches through a streaming session
  ppr       batched personalized PageRank: `columns` seed sets of 1 .. 1000 vertices
  weighted  weighted PageRank and its gradient through torch.autograd (forward and backward)

Graphs are directed RMAT (a/b/c/d = .57/.19/.19/.05, duplicates removed, a self-loop per vertex) over n vertices with
`factor` sampled edges per vertex, or the road-like 2D grid (4-neighbour edges kept with probability 0.62, symmetrized,
self-loops). `blocking`, `layout` and `window` are the launch plan a tuned program keeps for its graph (0: the default
row plan): what the autotuner chooses on graphs of that size.
"""
from __future__ import annotations

import math
import sys
from pathlib import Path

import numpy as np
import torch

sys.path.insert(0, str(Path(__file__).resolve().parent.parent / "pagerank-cuda-dynamic_amd"))

from pagerank_amd import (DYNAMIC_FRONTIER, DYNAMIC_TRAVERSAL, NAIVE_DYNAMIC, PRUNE_DYNAMIC_FRONTIER, STATIC, Batch,  # noqa: E402
                          Context, DeviceGraph, HostGraph, PagerankOptions, Stream, Tuning, pagerankStaticHip,
                          ppr_batched, solve, solve_device)

METHODS = {"nd": NAIVE_DYNAMIC, "dt": DYNAMIC_TRAVERSAL, "df": DYNAMIC_FRONTIER, "dfp": PRUNE_DYNAMIC_FRONTIER}
DAMPING, TOLERANCE, FLAG_TOLERANCE, MOST = 0.85, 1e-10, 1e-6, 500
DEV = "cuda"


def listed():
    return [
        # The smallest call a program makes: a graph of a thousand vertices, through host arrays.
        dict(name="static-n1k", kind="static", n=1024, factor=16.0, blocking=0, form="host"),
        # The configuration of the reference's CPU path: RMAT scale 16, through host arrays, untuned.
        dict(name="static-n64k", kind="static", n=65536, factor=16.0, blocking=0, form="host"),
        # A mid-sized graph of an odd size with the default plan.
        dict(name="static-n300k", kind="static", n=300007, factor=20.0, blocking=0, form="host"),
        # A tuned static solve with its arrays resident on the device: about a million vertices.
        dict(name="static-n1m", kind="static", n=1048576, factor=16.0, blocking=2048, form="device"),
        # The same on RMAT scale 24, the largest listed: 280M edges.
        dict(name="static-n16m", kind="static", n=16777216, factor=16.0, blocking=8192, form="device"),
        # A road-like graph: the 6000 x 4000 grid in its own order through the banded plan.
        dict(name="static-grid", kind="static", rows=6000, cols=4000, blocking=0, layout=1, window=1, form="device"),
        # A dynamic solve of a small graph without tuning: one batch of 1e-3 |E|.
        dict(name="df-n64k", kind="dynamic", method="df", n=65536, factor=16.0, blocking=0, fraction=1e-3),
        # A program that follows a large graph: batches of 1e-5 |E| applied in place, DF-P after each.
        dict(name="update-dfp-n1m5", kind="update", n=1500000, factor=16.0, blocking=2048, fraction=1e-5),
        # The same as a streaming session, with batches of 1e-4 |E|.
        dict(name="stream-dfp-n500k", kind="stream", n=500009, factor=16.0, blocking=2048, fraction=1e-4),
        # A full batch of personalized columns.
        dict(name="ppr64-n1m", kind="ppr", n=1048576, factor=16.0, columns=64),
        # A handful of personalized columns on a graph of an odd size.
        dict(name="ppr5-n100k", kind="ppr", n=100003, factor=12.0, columns=5),
        # A training step through the ranks: forward and gradients of all edge weights and the teleport vector.
        dict(name="weighted-n1m", kind="weighted", n=1048576, factor=16.0, blocking=2048),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _plan(edges):
    """The blocking of the launch plan a program keeps at this many edges: rows below 2^20 edges, then the blocked
    plan with blocks that grow with the graph."""
    return 0 if edges < 1 << 20 else 2048 if edges < 40e6 else 4096 if edges < 150e6 else 8192


def draw(rng):
    kind = rng.choice(["static", "static", "static", "grid", "dynamic", "dynamic", "update", "stream", "ppr", "ppr",
                       "weighted", "weighted"])
    factor = round(rng.uniform(6.0, 24.0), 1)
    if kind == "grid":
        return dict(kind="static", rows=_log(rng, 100, 5000), cols=_log(rng, 100, 4400), blocking=0, layout=1, window=1,
                    form=rng.choice(["host", "device"]))
    if kind == "static":
        n = _log(rng, 700, 8e6)
        tuned = rng.random() < 0.7
        return dict(kind=kind, n=n, factor=factor, blocking=_plan(n * factor) if tuned else 0,
                    form="host" if n < 500000 and rng.random() < 0.7 else "device")
    if kind == "dynamic":
        n = _log(rng, 1000, 1.5e6)
        return dict(kind=kind, method=rng.choice(["nd", "dt", "df", "dfp"]), n=n, factor=factor,
                    blocking=_plan(n * factor) if rng.random() < 0.7 else 0, fraction=rng.choice([1e-4, 1e-3]))
    if kind in ("update", "stream"):
        n = _log(rng, 20000, 1.5e6)
        return dict(kind=kind, n=n, factor=factor, blocking=max(2048, _plan(n * factor)),
                    fraction=rng.choice([1e-5, 1e-4, 1e-3]))
    if kind == "ppr":
        columns = rng.randint(1, 64)
        return dict(kind=kind, n=_log(rng, 2000, 1e6), factor=factor, columns=columns)
    n = _log(rng, 1000, 2e6)
    return dict(kind=kind, n=n, factor=factor, blocking=_plan(n * factor))


# ---- graphs ----


def _generator(seed, what):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed * 16 + what)
    return g


def _rmat_keys(n, factor, seed):
    """Sorted keys source * n + target of the graph's edges."""
    g = _generator(seed, 0)
    m, levels = int(n * factor), max(1, (n - 1).bit_length())
    src = torch.zeros(m, dtype=torch.int64, device=DEV)
    dst = torch.zeros(m, dtype=torch.int64, device=DEV)
    for _ in range(levels):
        u = torch.rand(m, generator=g, device=DEV)
        src.mul_(2).add_(u >= 0.76)
        dst.mul_(2).add_(((u >= 0.57) & (u < 0.76)) | (u >= 0.95))
    if n & (n - 1):
        keep = (src < n) & (dst < n)
        src, dst = src[keep], dst[keep]
    loops = torch.arange(n, device=DEV) * (n + 1)
    return torch.unique(torch.cat([src.mul_(n).add_(dst), loops]))


def _grid_keys(rows, cols, seed):
    g = _generator(seed, 0)
    n = rows * cols
    at = torch.arange(n, device=DEV).view(rows, cols)
    right = torch.rand(rows, cols - 1, generator=g, device=DEV) < 0.62
    down = torch.rand(rows - 1, cols, generator=g, device=DEV) < 0.62
    u = torch.cat([at[:, :-1][right], at[:-1][down]])
    v = torch.cat([at[:, 1:][right], at[1:][down]])
    return torch.sort(torch.cat([u * n + v, v * n + u, at.view(-1) * (n + 1)]))[0]


def _keys(case, seed):
    if case["kind"] == "weighted":  # a training program keeps its graph: the seed makes the weights and the loss
        seed = 1
    if "rows" in case:
        return case["rows"] * case["cols"], _grid_keys(case["rows"], case["cols"], seed)
    return case["n"], _rmat_keys(case["n"], case["factor"], seed)


def _offsets(of, n):
    off = torch.zeros(n + 1, dtype=torch.int64, device=DEV)
    torch.cumsum(torch.bincount(of, minlength=n), 0, out=off[1:])
    return off


def _u32(t):
    return t.to(torch.int32).cpu().numpy().view(np.uint32)


def _host_graph(n, keys):
    src, dst = keys // n, keys % n
    out_off = _offsets(src, n)
    back, eid = torch.sort(dst * n + src)
    return HostGraph(arrays=dict(out_off=_u32(out_off), out_edg=_u32(dst), outdeg=_u32(out_off.diff()),
                                 in_off=_u32(_offsets(back // n, n)), in_edg=_u32(back % n), in_eid=_u32(eid)))


def _batch_keys(n, keys, fraction, seed):
    """Sorted keys of a batch: 80% insertions of uniform absent pairs, 20% deletions of uniform edges that are no
    self-loops."""
    g = _generator(seed, 1)
    size = max(5, int(fraction * len(keys)))
    pick = keys[torch.randint(len(keys), (size // 5 + 1,), generator=g, device=DEV)]
    dels = torch.unique(pick[pick // n != pick % n])
    ins = torch.unique(torch.randint(n * n, (size - size // 5,), generator=g, device=DEV))
    at = torch.searchsorted(keys, ins).clamp_(max=len(keys) - 1)
    return dels, ins[keys[at] != ins]


def _batch(n, dels, ins):
    return Batch(_u32(dels // n), _u32(dels % n), _u32(ins // n), _u32(ins % n))


def _apply(keys, dels, ins):
    gone = torch.zeros(len(keys), dtype=torch.bool, device=DEV)
    gone[torch.searchsorted(keys, dels)] = True
    return torch.sort(torch.cat([keys[~gone], ins]))[0]


def _seed_sets(case, seed):
    r = np.random.RandomState(seed % (1 << 32))
    return [r.choice(case["n"], size=r.randint(1, min(1000, case["n"]) + 1), replace=False).astype(np.uint32)
            for _ in range(case["columns"])]


def _weighted_inputs(n, m, seed):
    """Edge weights in U(0.5, 1.5), a uniform teleport vector, and the gradient of L = sum c_v r_v^2 with c ~ N(0, 1)
    as a function of r."""
    g = _generator(seed, 2)
    w = torch.rand(m, generator=g, device=DEV) + 0.5
    s = torch.full((n,), 1.0 / n, dtype=torch.float64, device=DEV)
    c = torch.randn(n, generator=g, device=DEV, dtype=torch.float64)
    return w, s, c


# ---- what is measured ----


def prepare(case, seed):
    n, keys = _keys(case, seed)
    kind, ctx = case["kind"], Context(0)
    ctx.set_tuning(Tuning(blocking=case.get("blocking", 0), layout=case.get("layout", 0), window=case.get("window", 0)))
    o = PagerankOptions()
    state = dict(kind=kind, form=case.get("form"), ctx=ctx, options=o, method=METHODS.get(case.get("method")))
    ranks = lambda: torch.empty(n, dtype=torch.float64, device=DEV)  # noqa: E731
    if kind in ("dynamic", "update", "stream"):
        dels, ins = _batch_keys(n, keys, case["fraction"], seed)
        state["batch"] = _batch(n, dels, ins)
    if kind == "dynamic":  # the previous ranks come from a solve of the graph before the batch
        x = ctx.upload(_host_graph(n, keys))
        state["q"] = pagerankStaticHip(x, o).ranks
        x.close()
        keys = _apply(keys, dels, ins)
    state["graph"] = graph = DeviceGraph(ctx, _host_graph(n, keys), with_out=kind not in ("static", "ppr"))
    if kind == "static" and case["form"] == "device":
        state["ranks"] = ranks()
    elif kind == "update":
        state["q"], state["ranks"] = ranks(), [ranks(), ranks()]
        solve_device(graph, STATIC, o, None, state["q"].data_ptr())
        state["batches"] = [state["batch"], _batch(n, ins, dels)]
        state["sources"] = [[torch.from_numpy(a.view(np.int32)).to(DEV) for a in (b.del_u, b.del_v, b.ins_u)]
                            for b in state["batches"]]
    elif kind == "stream":
        state["batches"] = [state["batch"], _batch(n, ins, dels)]
        state["session"] = Stream(graph, PRUNE_DYNAMIC_FRONTIER, o, max_batch=len(dels) + len(ins))
    elif kind == "ppr":
        state["seeds"] = _seed_sets(case, seed)
    elif kind == "weighted":
        state["w"], state["s"], state["c"] = _weighted_inputs(n, len(keys), seed)
        state["w"].requires_grad_()
        state["s"].requires_grad_()
    torch.cuda.synchronize()
    return state


def run(state):
    kind, graph, o = state["kind"], state["graph"], state["options"]
    if kind == "static" and state["form"] == "host":
        r = pagerankStaticHip(graph, o)
        return dict(ranks=r.ranks, iterations=r.iterations)
    if kind == "static":
        st = solve_device(graph, STATIC, o, None, state["ranks"].data_ptr())
        return dict(ranks=state["ranks"], iterations=int(st.iterations))
    if kind == "dynamic":
        r = solve(graph, state["method"], o, state["batch"], state["q"])
        return dict(ranks=r.ranks, iterations=r.iterations)
    if kind == "update":
        q, counts = state["q"], []
        for batch, on_device, out in zip(state["batches"], state["sources"], state["ranks"]):
            graph.update(batch)
            du, dv, iu = on_device
            st = solve_device(graph, PRUNE_DYNAMIC_FRONTIER, o, q.data_ptr(), out.data_ptr(),
                              (du.data_ptr(), dv.data_ptr(), len(du), iu.data_ptr(), len(iu)))
            q = out
            counts.append(int(st.iterations))
        return dict(first=state["ranks"][0], second=state["ranks"][1], iterations=counts)
    if kind == "stream":
        a, b = (state["session"].update(batch) for batch in state["batches"])
        return dict(first=a.ranks, second=b.ranks, iterations=[a.iterations, b.iterations])
    if kind == "ppr":
        r = ppr_batched(graph, state["seeds"], o)
        return dict(ranks=r.ranks, iterations=r.iterations)
    from pagerank_amd import autograd
    r = autograd.pagerank(state["w"], state["s"], graph, o)
    gw, gs = torch.autograd.grad(r, (state["w"], state["s"]), 2 * state["c"] * r.detach())
    return dict(ranks=r.detach(), grad_weights=gw, grad_teleport=gs)


def work(case):
    """What the iterations cannot do without: each reads every edge's 4-byte neighbour id and, per vertex, an offset,
    an out-degree and the old rank, and writes the new rank. The iterations are about what these graphs take."""
    if "rows" in case:
        n, its = case["rows"] * case["cols"], 12
        m = n * (1 + 4 * 0.62)
    else:
        n = case["n"]
        m, its = n * (case["factor"] + 1), max(20, round(82 - 1.85 * (math.log2(n) - 12)))
    kind, k = case["kind"], case.get("columns", 1)
    if kind in ("dynamic", "update", "stream"):
        its = its // 3
    per = 4 * m + n * (8 + 16 * k)
    flops = 2 * k * m + 3 * k * n
    if kind == "weighted":
        per, flops, its = 8 * m + 32 * n, 3 * m + 3 * n, 2 * its
    if kind in ("update", "stream"):
        per, flops = 2 * per, 2 * flops
    return {"bytes": float(its * per), "flops": float(its * flops)}


# ---- the same in 64 bits with plain torch ----


def _matrix(n, rows, cols, values):
    """Row-sorted entries as an n x n matrix of 64-bit values."""
    return torch.sparse_csr_tensor(_offsets(rows, n), cols, values, size=(n, n), check_invariants=False)


def _csr(n, keys):
    """Sources and targets of the edges, the out-degrees, and the matrix that sums over in-neighbours."""
    src, dst = keys // n, keys % n
    back = torch.sort(dst * n + src)[0]
    sums = _matrix(n, back // n, back % n, torch.ones(len(keys), dtype=torch.float64, device=DEV))
    return src, dst, torch.bincount(src, minlength=n).double(), sums


def _exact_static(n, keys, q=None):
    _, _, deg, sums = _csr(n, keys)
    r = torch.full((n,), 1.0 / n, dtype=torch.float64, device=DEV) if q is None else q
    for it in range(1, MOST + 1):
        a = (1 - DAMPING) / n + DAMPING * (sums @ (r / deg))
        change = float((a - r).abs().max())
        r = a
        if change < TOLERANCE:
            break
    return r, it


def _exact_dynamic(method, n, keys, dels, ins, q):
    """DT, DF and DF-P on the graph `keys`, from q, for the batch that led to it."""
    if method == "nd":
        return _exact_static(n, keys, q)
    src, dst, deg, sums = _csr(n, keys)
    vaff = torch.zeros(n, dtype=torch.bool, device=DEV)
    front = torch.zeros(n, dtype=torch.bool, device=DEV)
    front[dels // n] = True
    front[ins // n] = True
    vaff[dels % n] = True
    vaff[dst[front[src]]] = True
    while method == "dt":
        before = int(vaff.sum())
        vaff[dst[vaff[src]]] = True
        if int(vaff.sum()) == before:
            break
    r = q
    for it in range(1, MOST + 1):
        c = r / deg
        s = sums @ c
        a = (1 - DAMPING) / n + DAMPING * s
        if method == "dfp":
            a = ((1 - DAMPING) / n + DAMPING * (s - c)) / (1 - DAMPING / deg)
        a = torch.where(vaff, a, r)
        change = float((a - r).abs().max())
        rel = (a - r).abs() / torch.maximum(a, r)
        r = a
        if change < TOLERANCE:
            break
        if method != "dt":
            front = vaff & (rel > FLAG_TOLERANCE)
            if method == "dfp":
                vaff &= rel > FLAG_TOLERANCE
            vaff[dst[front[src]]] = True
    return r, it


def _exact_ppr(n, keys, sets):
    _, _, deg, sums = _csr(n, keys)
    k = len(sets)
    s = torch.zeros(n, k, dtype=torch.float64, device=DEV)
    for j, v in enumerate(sets):
        s[torch.from_numpy(v.astype(np.int64)).to(DEV), j] = 1.0 / len(v)
    out = torch.empty_like(s)
    counts = np.zeros(k, dtype=np.int32)
    for j0 in range(0, k, 8):
        cols = slice(j0, min(k, j0 + 8))
        r, live = s[:, cols].clone(), torch.ones(cols.stop - j0, dtype=torch.bool, device=DEV)
        for it in range(1, MOST + 1):
            a = (1 - DAMPING) * s[:, cols] + DAMPING * (sums @ (r / deg[:, None]))
            change = (a - r).abs().amax(0)
            r = torch.where(live, a, r)
            counts[cols] = np.where(live.cpu().numpy(), it, counts[cols])
            live &= change >= TOLERANCE
            if not bool(live.any()):
                break
        out[:, cols] = r
    return out.cpu().numpy(), counts


def _exact_weighted(n, keys, seed):
    w, s, c = _weighted_inputs(n, len(keys), seed)
    src, dst = keys // n, keys % n
    w = w.double()
    out = _matrix(n, src, dst, w)
    back, eid = torch.sort(dst * n + src)
    sums = _matrix(n, back // n, back % n, w[eid])
    W = out @ torch.ones_like(s)
    r = s
    for _ in range(MOST):
        a = (1 - DAMPING) * s + DAMPING * (sums @ (r / W))
        change = float((a - r).abs().max())
        r = a
        if change < TOLERANCE:
            break
    g = 2 * c * r
    lam = g
    for _ in range(MOST):
        a = g + DAMPING / W * (out @ lam)
        change = float((a - lam).abs().max())
        lam = a
        if change < TOLERANCE:
            break
    mean = (lam - g) / DAMPING
    gw = (DAMPING * r / W)[src] * (lam[dst] - mean[src])
    return dict(ranks=r, grad_weights=gw, grad_teleport=(1 - DAMPING) * lam)


def exact(case, seed):
    n, keys = _keys(case, seed)
    kind = case["kind"]
    if kind == "static":
        r, it = _exact_static(n, keys)
        return dict(ranks=r, iterations=it)
    if kind == "ppr":
        r, counts = _exact_ppr(n, keys, _seed_sets(case, seed))
        return dict(ranks=r, iterations=counts)
    if kind == "weighted":
        return _exact_weighted(n, keys, seed)
    dels, ins = _batch_keys(n, keys, case["fraction"], seed)
    q, _ = _exact_static(n, keys)
    y = _apply(keys, dels, ins)
    if kind == "dynamic":
        r, it = _exact_dynamic(case["method"], n, y, dels, ins, q)
        return dict(ranks=r, iterations=it)
    first, a = _exact_dynamic("dfp", n, y, dels, ins, q)
    second, b = _exact_dynamic("dfp", n, keys, ins, dels, first)
    return dict(first=first, second=second, iterations=[a, b])
