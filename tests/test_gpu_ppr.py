"""Batched personalized PageRank on the GPU (prh_ppr_batched) against the oracle's single-column solve.

Bars: every column within L-inf 1e-9 of orc_ppr (the FP64 single-column solve with the same stopping rule) and with
the same iteration count +-1; a column whose teleport is uniform over all vertices equals the static solve within
1e-9; every column sums to 1 (no dead ends); results do not depend on how many iterations one HIP-graph replay
holds (the captured run is replayed many times and checked every time against the eager CPU result).
"""
from __future__ import annotations

import numpy as np
import pytest

from conftest import star_graph

pytestmark = pytest.mark.gpu


def _seed_sets(n, k, max_size, rng):
    return [rng.choice(n, size=int(rng.integers(1, max_size + 1)), replace=False).astype(np.uint32) for _ in range(k)]


def _teleport(n, seeds):
    s = np.zeros(n)
    np.add.at(s, seeds, 1.0 / len(seeds))
    return s


@pytest.mark.parametrize("scale,k", [(11, 64), (13, 64), (12, 5)])
def test_batched_matches_single_column_oracle(ctx, oracle_mod, scale, k):
    from pagerank_amd import HostGraph, ppr_batched
    y = HostGraph.rmat(scale, 16, seed=scale + k)
    rng = np.random.default_rng(scale * 100 + k)
    seeds = _seed_sets(y.N, k, min(1000, y.N // 4), rng)
    print(f"[ppr] scale={scale} k={k} N={y.N} M={y.M}", flush=True)
    res = ppr_batched(ctx.upload(y, with_out=False), seeds)
    assert res.ranks.shape == (y.N, k)
    for j in range(k):
        s = _teleport(y.N, seeds[j])
        ref, it = oracle_mod.ppr(y, s)
        assert abs(int(res.iterations[j]) - it) <= 1, (j, res.iterations[j], it)
        assert np.abs(res.ranks[:, j] - ref).max() <= 1e-9, j
        assert abs(res.ranks[:, j].sum() - 1.0) < 1e-9


def test_uniform_column_equals_static(ctx, oracle_mod):
    from pagerank_amd import HostGraph, pagerankStaticHip, ppr_batched
    y = HostGraph.rmat(12, 16, seed=3)
    yg = ctx.upload(y, with_out=False)
    seeds = [np.arange(y.N, dtype=np.uint32), np.array([7], dtype=np.uint32)]
    res = ppr_batched(yg, seeds)
    st = pagerankStaticHip(yg)
    assert abs(int(res.iterations[0]) - st.iterations) <= 1
    assert np.abs(res.ranks[:, 0] - st.ranks).max() <= 1e-9


def test_heavy_vertex_chunks(ctx, oracle_mod):
    """A hub with in-degree above the chunk size is summed in chunks by many waves and combined."""
    from pagerank_amd import ppr_batched
    y = star_graph(6000)
    seeds = [np.array([0], np.uint32), np.array([1, 2, 3], np.uint32), np.arange(1, 6000, 7, dtype=np.uint32)]
    res = ppr_batched(ctx.upload(y, with_out=False), seeds)
    for j, sd in enumerate(seeds):
        ref, it = oracle_mod.ppr(y, _teleport(y.N, sd))
        assert abs(int(res.iterations[j]) - it) <= 1
        assert np.abs(res.ranks[:, j] - ref).max() <= 1e-9


@pytest.mark.parametrize("interval", [1, 3, 16])
def test_graph_replay_interval_does_not_change_results(ctx, interval):
    from pagerank_amd import HostGraph, Tuning, ppr_batched
    y = HostGraph.rmat(11, 16, seed=9)
    yg = ctx.upload(y, with_out=False)
    seeds = _seed_sets(y.N, 64, 100, np.random.default_rng(1))
    old = ctx.get_tuning()
    try:
        ctx.set_tuning(Tuning(old.switch_degree, old.huge_degree, old.low_width, 8))
        base = ppr_batched(yg, seeds)
        ctx.set_tuning(Tuning(old.switch_degree, old.huge_degree, old.low_width, interval))
        for _ in range(2):  # replays of a freshly captured graph, twice, with eager work in between
            again = ppr_batched(yg, seeds)
            assert np.array_equal(again.ranks, base.ranks)
            assert np.array_equal(again.iterations, base.iterations)
    finally:
        ctx.set_tuning(old)


def test_bad_seeds_rejected(ctx):
    from pagerank_amd import HostGraph, PagerankError, ppr_batched
    yg = ctx.upload(HostGraph.rmat(8, 4, seed=1), with_out=False)
    with pytest.raises(PagerankError):
        ppr_batched(yg, [np.array([10**6], np.uint32)])
    with pytest.raises(PagerankError):
        ppr_batched(yg, [np.zeros(0, np.uint32)])
    with pytest.raises(PagerankError):
        ppr_batched(yg, [np.array([1], np.uint32)] * 65)


def test_uncaptured_mode_matches_captured(monkeypatch):
    """PRH_GRAPH_CAPTURE=0 at context creation: the batched solve and the streaming session issue their launches
    one by one instead of replaying captured graphs; the results are the same bits (no order-dependent sums here:
    the row plan and the batched solver sum in a fixed order)."""
    from pagerank_amd import Batch, Context, HostGraph, Stream, engine
    y = HostGraph.rmat(12, 16, seed=8)
    rng = np.random.default_rng(2)
    sets = [rng.choice(y.N, size=int(rng.integers(1, 50)), replace=False).astype(np.uint32) for _ in range(5)]
    b = Batch.random(y, 60, 0.8, seed=3)
    out = {}
    for mode in ("1", "0"):
        monkeypatch.setenv("PRH_GRAPH_CAPTURE", mode)
        with Context(0) as c:
            yg = c.upload(y)
            res = engine.ppr_batched(yg, sets)
            st = Stream(yg, 4, max_batch=128)
            got = st.update(b)
            st.close()
            yg.close()
        out[mode] = (res.ranks, res.iterations, got.ranks, got.iterations)
    assert np.array_equal(out["0"][0], out["1"][0]) and np.array_equal(out["0"][1], out["1"][1])
    assert np.array_equal(out["0"][2], out["1"][2]) and out["0"][3] == out["1"][3]


@pytest.mark.parametrize("k", [1, 2, 3, 4, 5, 8, 9, 16, 17, 32, 33, 64])
def test_tile_widths_and_row_classes(ctx, oracle_mod, k):
    """Every tile width (and padded columns), on rows at the edges of the row classes: lane groups, waves, chunks.
    Seed sets overlap, repeat a seed, and include vertices nobody but themselves links to. Bound: the sums of at most
    40001 non-negative terms in two orders differ by 2 d 2^-53 of the sum, amplified by 1 / (1 - 0.85): 6e-11."""
    from pagerank_amd import ppr_batched
    from test_gpu_rows import degree_graph
    n = 40961
    y = degree_graph(n, 11)
    rng = np.random.default_rng(k)
    seeds = _seed_sets(n, k, 400, rng)
    seeds[0] = np.array([n - 1, n - 1, 5, n - 2, 5, n - 1], dtype=np.uint32)
    seeds[k - 1] = np.concatenate([seeds[k - 1], seeds[0]])
    print(f"[ppr] tiles k={k} N={y.N} M={y.M}", flush=True)
    res = ppr_batched(ctx.upload(y, with_out=False), seeds)
    for j in sorted({0, k // 3, k // 2, k - 1}):
        ref, it = oracle_mod.ppr(y, _teleport(n, seeds[j]))
        assert abs(int(res.iterations[j]) - it) <= 1
        if res.iterations[j] == it:
            assert np.all(np.abs(res.ranks[:, j] - ref) <= 6e-11 * ref)
        assert np.abs(res.ranks[:, j] - ref).max() <= 1e-9


def test_ranks_larger_than_the_staging_area(ctx, oracle_mod):
    """72 MB of ranks: copied to the host in slots of the 64 MB staging area by several threads, the last one in part."""
    from pagerank_amd import HostGraph, ppr_batched
    n, k = 140001, 64
    rng = np.random.default_rng(4)
    src = np.concatenate([rng.integers(0, n, 300000), np.arange(n)]).astype(np.uint32)
    dst = np.concatenate([rng.integers(0, n, 300000), (np.arange(n) + 1) % n]).astype(np.uint32)
    y = HostGraph.from_edges(n, src, dst)
    seeds = _seed_sets(n, k, 300, rng)
    print(f"[ppr] staging N={y.N} M={y.M}", flush=True)
    yg = ctx.upload(y, with_out=False)
    for _ in range(2):
        res = ppr_batched(yg, seeds)
        assert np.abs(res.ranks.sum(axis=0) - 1.0).max() < 1e-8
    for j in (0, 31, 63):
        ref, it = oracle_mod.ppr(y, _teleport(n, seeds[j]))
        assert abs(int(res.iterations[j]) - it) <= 1 and np.abs(res.ranks[:, j] - ref).max() <= 1e-9


@pytest.mark.parametrize("k", [3, 40])
def test_iteration_cap_with_heavy_rows(monkeypatch, k):
    """Caps before, at and after the end of a replay of eight iterations, reached unconverged, on rows cut into chunks:
    the loop ends while the last replay's heavy rows are still to be finished. Captured and launched one by one, three
    times over: the same bits."""
    from pagerank_amd import Context, PagerankOptions, ppr_batched
    from test_gpu_rows import degree_graph
    y = degree_graph(40961, 13)
    seeds = _seed_sets(y.N, k, 200, np.random.default_rng(k))
    out = {}
    for mode in ("0", "1"):
        monkeypatch.setenv("PRH_GRAPH_CAPTURE", mode)
        with Context(0) as c:
            yg = c.upload(y, with_out=False)
            for cap in (0, 1, 7, 8, 9, 16):
                for i in range(3 if mode == "1" else 1):
                    print(f"[ppr cap] k={k} capture={mode} cap={cap} pass={i}", flush=True)
                    res = ppr_batched(yg, seeds, PagerankOptions(tolerance=0.0, maxIterations=cap))
                    assert np.all(res.iterations == cap)
                    assert np.array_equal(res.ranks, out.setdefault(cap, res.ranks))
            yg.close()


def test_waiting_leaves_the_core(ctx):
    """The host waits 16 ms and more for each run of iterations (512 of at least 32 us): it polls for the first millisecond
    and sleeps after it, so the calling thread takes less than half of the call's time (the rest of it, the capture and
    the way back of 34 MB, is some ten milliseconds)."""
    import time

    from pagerank_amd import HostGraph, PagerankOptions, Tuning, ppr_batched
    y = HostGraph.rmat(16, 16, seed=4)
    seeds = _seed_sets(y.N, 64, 20, np.random.default_rng(5))
    yg = ctx.upload(y, with_out=False)
    old = ctx.get_tuning()
    try:
        ctx.set_tuning(Tuning(**{**old.__dict__, "check_interval": 512}))
        o = PagerankOptions(tolerance=0.0, maxIterations=2048)
        ppr_batched(yg, seeds, o)
        wall, cpu = time.perf_counter(), time.thread_time()
        ppr_batched(yg, seeds, o)
        wall, cpu = time.perf_counter() - wall, time.thread_time() - cpu
    finally:
        ctx.set_tuning(old)
    print(f"[wait] {wall * 1e3:.1f} ms, {cpu * 1e3:.1f} ms of the calling thread's", flush=True)
    assert cpu < 0.5 * wall


def test_repeated_seeds(ctx, oracle_mod):
    """Seed sets that repeat few vertices many times, in runs, shuffled and among seeds of their own: the shares are the
    counts over the size, whatever the order, and the results repeat bit for bit."""
    from pagerank_amd import HostGraph, ppr_batched
    y = HostGraph.rmat(11, 16, seed=6)
    rng = np.random.default_rng(8)
    runs = np.repeat(np.arange(10, dtype=np.uint32), 3001)
    seeds = [runs, rng.permutation(runs), np.full(50021, 7, np.uint32),
             rng.permutation(np.concatenate([np.arange(y.N, dtype=np.uint32), np.full(777, 3, np.uint32)])),
             np.array([5], np.uint32), np.arange(63, dtype=np.uint32), np.repeat(np.arange(65, dtype=np.uint32), 2)]
    print(f"[ppr repeats] N={y.N} M={y.M}", flush=True)
    yg = ctx.upload(y, with_out=False)
    res = ppr_batched(yg, seeds)
    assert np.array_equal(res.ranks[:, 0], res.ranks[:, 1])
    again = ppr_batched(yg, seeds)
    assert np.array_equal(again.ranks, res.ranks)
    for j, sd in enumerate(seeds):
        s = np.bincount(sd, minlength=y.N) / len(sd)
        ref, it = oracle_mod.ppr(y, s)
        assert abs(int(res.iterations[j]) - it) <= 1
        assert np.abs(res.ranks[:, j] - ref).max() <= 1e-9
