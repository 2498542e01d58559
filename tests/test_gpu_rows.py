"""The row plan at the edges of its row classes and of its gather batches: rows of one lane group, one wave, one
workgroup and several chunks, with every remainder of a batch of eight gathers per lane."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

DEGREES = ([1, 2, 3, 4, 5, 7, 8, 9, 15, 16, 17, 31, 32, 33, 63, 64, 65] + [64 * k + j for k in range(2, 10) for j in (-1, 0, 1)]
           + [1023, 1024, 1025] + [256 * k + j for k in range(5, 10) for j in (-1, 0, 1)]
           + [4095, 4097, 16383, 16384, 16385, 40001])


def degree_graph(n: int, seed: int):
    """Vertex i has in-degree DEGREES[i % len] (a self-loop among them) for the first rows, 1 (its self-loop) after."""
    from pagerank_amd import HostGraph
    rng = np.random.RandomState(seed)
    src, dst = [], []
    for i, d in enumerate(DEGREES):
        u = (i + 1 + rng.randint(0, n - d) + np.arange(d - 1)) % n
        u = u[u != i]
        src.append(u)
        dst.append(np.full(len(u), i))
    return HostGraph.from_edges(n, np.concatenate(src).astype(np.uint32), np.concatenate(dst).astype(np.uint32))


@pytest.mark.parametrize("method", [0, 3, 4], ids=["static", "DF", "DFP"])
@pytest.mark.parametrize("n", [40003, 65536])
def test_row_classes(ctx, oracle_mod, n, method):
    """Every row of at most 40001 terms differs from the oracle's by rounding only: the sums of d non-negative terms
    in two orders differ by at most 2 d 2^-53 of the sum, which the iteration amplifies by 1 / (1 - 0.85): 6e-11."""
    from pagerank_amd import Batch, apply_batch, solve
    x = degree_graph(n, 7)
    q, _, _ = oracle_mod.pagerank_cuda(oracle_mod.STATIC, x)
    b = Batch.random(x, 300, 0.8, seed=3)
    y = apply_batch(x, b)
    print(f"[rows] N={y.N} M={y.M} method={method}", flush=True)
    res = solve(ctx.upload(y), method, batch=b if method else None, q=q if method else None)
    ref, it, _ = oracle_mod.pagerank_cuda(method, y, b if method else None, q if method else None)
    assert abs(res.iterations - it) <= 1
    if res.iterations == it:
        assert np.all(np.abs(res.ranks - ref) <= 6e-11 * ref)
    assert np.abs(res.ranks - ref).max() <= 1e-9


def small_graph(n: int, seed: int):
    """The first rows have the degrees of DEGREES that n allows, up to 1025 (in all 12,000 edges); the rest 1 to 3."""
    from pagerank_amd import HostGraph
    rng = np.random.RandomState(seed)
    src, dst = [rng.randint(0, n, 2 * n)], [np.arange(2 * n) % n]
    for i, d in enumerate([d for d in DEGREES if d <= min(1025, n // 2)]):
        src.append((i + 1 + rng.randint(0, n - d) + np.arange(d - 1)) % n)
        dst.append(np.full(d - 1, i))
    return HostGraph.from_edges(n, np.concatenate(src).astype(np.uint32), np.concatenate(dst).astype(np.uint32))


@pytest.mark.parametrize("method", range(5), ids=["static", "ND", "DT", "DF", "DFP"])
@pytest.mark.parametrize("n", [1, 63, 65, 1023, 1100, 2049, 2900, 3600, 5800])
def test_small_graphs(ctx, oracle_mod, n, method):
    """Sizes on both sides of what one workgroup's LDS holds. The bound is test_row_classes' with sums of at most 1,100
    terms: 1.6e-12. Then 600 iterations at tolerance 0, which take several launches."""
    from pagerank_amd import Batch, PagerankOptions, apply_batch, solve
    x = small_graph(n, n)
    q, _, _ = oracle_mod.pagerank_cuda(oracle_mod.STATIC, x)
    b = Batch.random(x, max(1, n // 100), 0.8, seed=3) if n > 1 else Batch.empty()
    y = apply_batch(x, b)
    yg = ctx.upload(y)
    args = (b if method else None, q if method else None)
    print(f"[small] N={y.N} M={y.M} method={method}", flush=True)
    for tolerance, iterations in ((1e-10, 500), (0.0, 600)):
        o = PagerankOptions(tolerance=tolerance, maxIterations=iterations)
        res = solve(yg, method, o, batch=args[0], q=args[1])
        ref, it, _ = oracle_mod.pagerank_cuda(method, y, *args, tolerance=tolerance, max_iterations=iterations)
        assert abs(res.iterations - it) <= 1 and (tolerance or res.iterations == it)
        if res.iterations == it:
            assert np.all(np.abs(res.ranks - ref) <= 1.6e-12 * ref)
        assert np.abs(res.ranks - ref).max() <= 1e-9
        again = solve(yg, method, o, batch=args[0], q=args[1])
        assert np.array_equal(again.ranks, res.ranks)


@pytest.mark.parametrize("method", [0, 1], ids=["static", "ND"])
@pytest.mark.parametrize("largest", [65535, 65536, 65539, 1 << 24, (1 << 32) - 1])
def test_small_graph_with_large_out_degrees(ctx, method, largest):
    """Without an out-CSR nothing bounds the out-degrees by the edges (an in-graph that holds part of a larger one).
    Twenty iterations against numpy in 64 bits, with test_small_graphs' bound."""
    from pagerank_amd import HostGraph, PagerankOptions, solve
    x = small_graph(900, 11)
    deg = x.outdeg.copy()
    deg[::7] = largest
    deg[3::7] = np.minimum(largest, 65534)
    y = HostGraph(arrays=dict(out_off=x.out_off, out_edg=x.out_edg, in_off=x.in_off, in_edg=x.in_edg, in_eid=x.in_eid,
                              outdeg=deg))
    q = np.random.RandomState(2).rand(y.N)
    q /= q.sum()
    print(f"[small] out-degrees up to {largest} method={method}", flush=True)
    res = solve(ctx.upload(y, with_out=False), method, PagerankOptions(tolerance=0.0, maxIterations=20),
                q=q if method else None)
    row = np.repeat(np.arange(y.N), np.diff(y.in_off.astype(np.int64)))
    r = q if method else np.full(y.N, 1.0 / y.N)
    for _ in range(20):
        r = 0.15 / y.N + 0.85 * np.bincount(row, (r / deg)[y.in_edg], y.N)
    assert res.iterations == 20
    assert np.all(np.abs(res.ranks - r) <= 1.6e-12 * r)


@pytest.mark.parametrize("method", [3, 4], ids=["DF", "DFP"])
@pytest.mark.parametrize("edges", [2, 300])
def test_extension_inside_the_update(ctx, method, edges):
    """The extension within the update (direction 1 at this size) sets the flags that push and pull set, in rows of every
    class: the ranks are the same bit for bit."""
    from pagerank_amd import Batch, apply_batch, solve
    x = degree_graph(40003, 9)
    q = solve(ctx.upload(x), 0).ranks
    b = Batch.random(x, edges, 0.8, seed=5)
    yg = ctx.upload(apply_batch(x, b))
    old = ctx.get_tuning()
    out = {}
    try:
        for d in (0, 1, 2):
            print(f"[inside] method={method} edges={edges} direction={d}", flush=True)
            t = ctx.get_tuning()
            t.extension_direction = d
            ctx.set_tuning(t)
            out[d] = solve(yg, method, batch=b, q=q)
    finally:
        ctx.set_tuning(old)
    for d in (1, 2):
        assert out[d].iterations == out[0].iterations
        assert np.array_equal(out[d].ranks, out[0].ranks), d


@pytest.mark.parametrize("method", [3, 4], ids=["DF", "DFP"])
@pytest.mark.parametrize("edges", [40, 20000])
def test_extension_directions_above_the_inside_limit(ctx, method, edges):
    """Above 2^24 edges the extension is a launch of its own, pushed, pulled, or the cheaper by the sums that the rank
    launches leave (direction 1); rows cut into chunks, which the second launch finishes, add to those sums too. All three
    set the same flags: the ranks are the same bit for bit."""
    from pagerank_amd import Batch, HostGraph, apply_batch, solve
    x = HostGraph.rmat(20, 18, seed=6)
    b = Batch.random(x, edges, 0.8, seed=2)
    y = apply_batch(x, b)
    assert y.M > 1 << 24 and np.diff(y.in_off.astype(np.int64)).max() > 16384
    q = solve(ctx.upload(x), 0).ranks
    yg = ctx.upload(y)
    old = ctx.get_tuning()
    out = {}
    try:
        for d in (0, 1, 2):
            print(f"[outside] M={y.M} method={method} edges={edges} direction={d}", flush=True)
            t = ctx.get_tuning()
            t.extension_direction = d
            ctx.set_tuning(t)
            out[d] = solve(yg, method, batch=b, q=q)
    finally:
        ctx.set_tuning(old)
    for d in (1, 2):
        assert out[d].iterations == out[0].iterations
        assert np.array_equal(out[d].ranks, out[0].ranks), d


@pytest.mark.parametrize("direction", [0, 2])
def test_hub_chunks_of_the_push_across_tunings(ctx, oracle_mod, direction):
    """A source of 6000 out-edges among the batch's: the push takes it in chunks of the cached out-degree schedule, before
    and after a tuning change that rebuilds the rank plan (the pull for comparison)."""
    from pagerank_amd import Batch, HostGraph, apply_batch, solve
    n = 9000
    rng = np.random.default_rng(4)
    src = np.concatenate([np.zeros(6000, np.uint32), rng.integers(0, n, 30000).astype(np.uint32)])
    dst = np.concatenate([np.arange(1, 6001, dtype=np.uint32), rng.integers(0, n, 30000).astype(np.uint32)])
    x = HostGraph.from_edges(n, src, dst, self_loops=True)
    b = Batch.tidy(x, [[0, 1]], [[0, 7000], [5, 8000]])
    y = apply_batch(x, b)
    print(f"[hub push] N={y.N} M={y.M} direction={direction}", flush=True)
    yg = ctx.upload(y)
    q, _, _ = oracle_mod.pagerank_cuda(oracle_mod.STATIC, x)
    ref, it, _ = oracle_mod.pagerank_cuda(3, y, b, q)
    old = ctx.get_tuning()
    try:
        for switch in (64, 128):
            t = ctx.get_tuning()
            t.extension_direction, t.switch_degree = direction, switch
            ctx.set_tuning(t)
            res = solve(yg, 3, batch=b, q=q)
            assert abs(res.iterations - it) <= 1
            assert np.abs(res.ranks - ref).max() <= 1e-9
    finally:
        ctx.set_tuning(old)


@pytest.mark.parametrize("method", [0, 3], ids=["static", "DF"])
def test_rows_without_in_edges_beyond_one_workgroup(ctx, oracle_mod, method):
    """More vertices than one workgroup's LDS holds, most of them without in-edges, one row in chunks of 64 edges. (Not
    DF-P: its closed form takes every vertex to have a self-loop, and without one the oracle too diverges to NaN.)"""
    from pagerank_amd import Batch, HostGraph, Tuning, apply_batch, solve
    n = 9000
    u = np.arange(n, dtype=np.uint32)
    src = np.concatenate([u[1:], [0], u[:100]])
    dst = np.concatenate([np.zeros(n - 1, np.uint32), [1], (u[:100] * 7 + 3) % 50])
    x = HostGraph.from_edges(n, src, dst, self_loops=False)
    b = Batch.tidy(x, np.zeros((0, 2)), [[3, 60], [200, 61]])
    y = apply_batch(x, b)
    q, _, _ = oracle_mod.pagerank_cuda(oracle_mod.STATIC, x)
    args = (b, q) if method else (None, None)
    old = ctx.get_tuning()
    print(f"[no-in-edges] N={y.N} M={y.M} method={method}", flush=True)
    try:
        ctx.set_tuning(Tuning(64, 64, old.low_width, old.check_interval, 0))
        res = solve(ctx.upload(y), method, batch=args[0], q=args[1])
    finally:
        ctx.set_tuning(old)
    ref, it, _ = oracle_mod.pagerank_cuda(method, y, *args)
    assert abs(res.iterations - it) <= 1
    assert np.abs(res.ranks - ref).max() <= 1e-9
    if not method:
        assert np.all(res.ranks[np.diff(y.in_off.astype(np.int64)) == 0] == (1 - 0.85) / n)


@pytest.mark.parametrize("method", [3, 4], ids=["DF", "DFP"])
def test_push_of_every_out_degree(ctx, method):
    """Sources of every class and remainder of the push (lane groups, waves, chunks; eight loads in flight a lane) in the
    frontier: pushed and pulled, the same flags, hence the same bits."""
    from pagerank_amd import Batch, HostGraph, apply_batch, solve
    t = degree_graph(40003, 17)
    dst = np.repeat(np.arange(t.N, dtype=np.uint32), np.diff(t.out_off.astype(np.int64)))
    x = HostGraph.from_edges(t.N, t.out_edg.astype(np.uint32), dst)  # transposed: DEGREES are out-degrees
    q = solve(ctx.upload(x), 0).ranks
    k = np.arange(len(DEGREES))
    b = Batch.tidy(x, np.zeros((0, 2)), np.stack([k, 30000 + k], axis=1))
    yg = ctx.upload(apply_batch(x, b))
    old = ctx.get_tuning()
    out = {}
    try:
        for d in (0, 2):
            print(f"[push] method={method} direction={d}", flush=True)
            tuning = ctx.get_tuning()
            tuning.extension_direction = d
            ctx.set_tuning(tuning)
            out[d] = solve(yg, method, batch=b, q=q)
    finally:
        ctx.set_tuning(old)
    assert out[0].iterations == out[2].iterations > 1
    assert np.array_equal(out[0].ranks, out[2].ranks)


@pytest.mark.parametrize("method", [3, 4], ids=["DF", "DFP"])
def test_pushed_solves_beyond_the_infinity_cache(ctx, method):
    """A graph whose in-CSR the pushed solves read with non-temporal loads (5M vertices, rows of every class): the same bits
    as pulled, where the loads are plain ones."""
    from pagerank_amd import Batch, apply_batch, solve
    x = degree_graph(5_000_003, 21)
    rest = 4 * (x.M + x.N) + 42 * x.N
    assert rest <= 1 << 28 < 4 * (x.M + x.N) + rest  # the rule of the dispatch
    q = solve(ctx.upload(x), 0).ranks
    b = Batch.random(x, 3000, 0.8, seed=5)
    yg = ctx.upload(apply_batch(x, b))
    old = ctx.get_tuning()
    out = {}
    try:
        for d in (0, 2):
            print(f"[stream csr] method={method} direction={d}", flush=True)
            tuning = ctx.get_tuning()
            tuning.extension_direction = d
            ctx.set_tuning(tuning)
            out[d] = solve(yg, method, batch=b, q=q)
    finally:
        ctx.set_tuning(old)
    assert out[0].iterations == out[2].iterations > 1
    assert np.array_equal(out[0].ranks, out[2].ranks)
