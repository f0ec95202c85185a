"""GPU tests of the SSSP sweeps on the weight-sorted adjacency: rows at the
edges of the sort's classes (4, 16, 64, 512 and 2048 edges, hub chunks), weights
that one key holds exactly (up to 63) and that share keys (up to 2^30), zero
weights, unsorted vertex orders, 8-byte offsets, shares, and initial distances
of every kind.  Distances are the unique fixpoint: equality with the oracle."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _stars(hc, degrees, max_weight, seed, extra=4000):
    """A graph with one hub of each given degree over a common pool of leaves,
    and random edges among the leaves."""
    rng = np.random.default_rng(seed)
    hubs = len(degrees)
    leaves = max(degrees) + 8
    src, dst = [], []
    for h, d in enumerate(degrees):
        src.append(np.full(d, h))
        dst.append(hubs + rng.choice(leaves, d, replace=False))
    src.append(hubs + rng.integers(0, leaves, extra))
    dst.append(hubs + rng.integers(0, leaves, extra))
    src, dst = np.concatenate(src), np.concatenate(dst)
    w = rng.integers(0, max_weight + 1, src.size).astype(np.int32)
    return hc.HostGraph.from_edges(src.astype(np.int32), dst.astype(np.int32), hubs + leaves,
                                   weights=w, relabel=bool(seed % 2))


@pytest.fixture(autouse=True)
def always_sorted(hc):
    """These graphs are below the size from which the copy is built."""
    hc.set_tuning("sssp.sorted", 2)
    yield
    hc.reset_tuning()


DEGREES = [1, 3, 4, 5, 15, 16, 17, 63, 64, 65, 511, 512, 513, 2047, 2048, 2049, 4095, 4096, 4097,
           20000, 40001]


@pytest.mark.parametrize("max_weight", [0, 1, 63, 64, 255, 70000, (1 << 30) - 2])
@pytest.mark.parametrize("seed", [0, 1])
def test_sorted_rows_exact(hc, gpu, oracle, max_weight, seed):
    g = _stars(hc, DEGREES, max_weight, seed)
    with hc.DeviceGraph(g) as dg:
        for s in (0, 7, g.num_nodes - 5):
            ref = oracle.sssp_dijkstra(g.index, g.neighbors, g.weights, s)
            for direction in (0, 1, 2):
                assert np.array_equal(hc.sssp(dg, s, direction=direction).values, ref), direction
            for delta in (max(1, max_weight // 16), max(1, max_weight)):
                dg.set_tuning("sssp.delta", delta)
                for direction in (0, 2):
                    assert np.array_equal(hc.sssp(dg, s, direction=direction).values, ref), delta
                dg.reset_tuning()


def test_sorted_matches_plain_wide_offsets_and_shares(hc, gpu, oracle, monkeypatch):
    monkeypatch.setenv("HC_FORCE_OFF64", "1")
    g = _stars(hc, DEGREES, 1000, 3)
    u = hc.HostGraph.generate("uniform", 12, 6, weighted=True, seed=4)
    for gg in (g, u):
        with hc.DeviceGraph(gg) as dg:
            assert dg.info()["offset_bytes"] == 8
            s = int(gg.pick_sources(1)[0])
            ref = oracle.sssp_dijkstra(gg.index, gg.neighbors, gg.weights, s)
            share = dg.share()
            for h in (dg, share):
                assert np.array_equal(hc.sssp(h, s).values, ref)
            share.set_tuning("sssp.sorted", 0)
            assert np.array_equal(hc.sssp(share, s).values, ref)
            share.free()


@pytest.mark.parametrize("init", ["one", "many", "low", "negative", "above"])
def test_sorted_pull_initial_distances(hc, gpu, oracle, init):
    """hc_sssp_pull from initial distances: the sorted sweeps give what the
    plain ones give, also for values outside the sentinel's range."""
    g = hc.HostGraph.generate("kron", 11, 8, weighted=True, seed=9)
    rng = np.random.default_rng(2)
    d0 = np.full(g.num_nodes, hc.INF_DIST, np.int32)
    some = rng.choice(g.num_nodes, 40, replace=False)
    if init == "one":
        d0[some[0]] = 0
    elif init == "many":
        d0[some] = rng.integers(0, 500, 40)
    elif init == "low":
        d0[:] = rng.integers(1000, 2000, g.num_nodes)
        d0[some] = 990
    elif init == "negative":
        d0[some] = rng.integers(-300, 300, 40)
    else:
        d0[some[:20]] = 5
        d0[some[20:]] = hc.INF_DIST + 77
    with hc.DeviceGraph(g) as dg:
        got = hc.sssp_pull(dg, d0).values
        dg.set_tuning("sssp.sorted", 0)
        assert np.array_equal(got, hc.sssp_pull(dg, d0).values)


def test_flat_buckets_cover_every_settling_path(hc, gpu, oracle):
    """A flat graph whose buckets are settled by pushes (few vertices done) and
    by sweeps (most done), with sweeps inside heavy buckets; narrow and wide
    weights, and parts that the source does not reach."""
    rng = np.random.default_rng(5)
    n = 30000
    src, dst = rng.integers(0, n - 500, 8 * n), rng.integers(0, n - 500, 8 * n)
    for top in (3, 255, 100000):
        w = rng.integers(1, top + 1, src.size).astype(np.int32)
        g = hc.HostGraph.from_edges(src.astype(np.int32), dst.astype(np.int32), n, weights=w)
        with hc.DeviceGraph(g) as dg:
            for s in (0, 123):
                ref = oracle.sssp_dijkstra(g.index, g.neighbors, g.weights, s)
                for delta in (-1, 1, max(1, top // 8), top, 4 * top):
                    if delta == 1 and top > 255:
                        continue  # tens of thousands of buckets
                    dg.set_tuning("sssp.delta", delta)
                    r = hc.sssp(dg, s)
                    assert np.array_equal(r.values, ref), (top, delta)
                    assert r.stats["pull_epochs"] == 0
                    assert np.array_equal(hc.sssp(dg, s, direction=2).values, ref), (top, delta)


@pytest.mark.parametrize("wide", [False, True])
@pytest.mark.parametrize("top", [3, 255, 100000])
def test_buckets_turn_light_and_heavy(hc, gpu, oracle, monkeypatch, top, wide):
    """Two dense cores of 800K edges joined by a long path, with a tail and
    unreached vertices behind: buckets start light (the far set), turn heavy in a
    core (scans and sweeps), light again on the path, and heavy in the second
    core."""
    if wide:
        monkeypatch.setenv("HC_FORCE_OFF64", "1")
    rng = np.random.default_rng(top)
    core, path = 40000, 600
    src, dst = [], []
    for base in (0, core + path):
        src.append(base + rng.integers(0, core, 10 * core))
        dst.append(base + rng.integers(0, core, 10 * core))
    for first in (core - 1, 2 * core + path - 1):
        src.append(first + np.arange(path))
        dst.append(first + 1 + np.arange(path))
    src, dst = np.concatenate(src), np.concatenate(dst)
    n = 2 * (core + path) + 500
    w = rng.integers(1, top + 1, src.size).astype(np.int32)
    for relabel in (False, True):
        g = hc.HostGraph.from_edges(src.astype(np.int32), dst.astype(np.int32), n, weights=w,
                                    relabel=relabel)
        with hc.DeviceGraph(g) as dg:
            for s in (0, int(g.pick_sources(1)[0]), n // 2):
                ref = oracle.sssp_dijkstra(g.index, g.neighbors, g.weights, s)
                for delta in (-1, max(1, top // 20), top, 20 * top):
                    dg.set_tuning("sssp.delta", delta)
                    for direction in (0, 2):
                        got = hc.sssp(dg, s, direction=direction).values
                        assert np.array_equal(got, ref), (s, delta, direction)


@pytest.mark.parametrize("wide", [False, True])
@pytest.mark.parametrize("knob,value", [("sssp.sorted", 0), ("sssp.filter", 1), ("sssp.dist16", 1),
                                        ("pull.col_shift", 10)])
def test_buckets_without_the_copy(hc, gpu, oracle, monkeypatch, knob, value, wide):
    """sssp.delta holds on the plain CSR too (no copy, or a knob that asks for a
    plain sweep): vertices past the threshold wait in the far set and are
    promoted, hubs and zero weights among them, and no epoch pulls."""
    if wide:
        monkeypatch.setenv("HC_FORCE_OFF64", "1")
    rng = np.random.default_rng(8)
    n = 20000
    src, dst = rng.integers(0, n - 300, 6 * n), rng.integers(0, n - 300, 6 * n)
    for top in (3, 255, (1 << 30) - 2):
        w = rng.integers(0, top + 1, src.size).astype(np.int32)
        flat = hc.HostGraph.from_edges(src.astype(np.int32), dst.astype(np.int32), n, weights=w)
        for g in (flat, _stars(hc, DEGREES, top, 1)):
            with hc.DeviceGraph(g) as dg:
                dg.set_tuning(knob, value)
                for s in (0, g.num_nodes // 3):
                    ref = oracle.sssp_dijkstra(g.index, g.neighbors, g.weights, s)
                    for delta in (max(1, top // 8), top, 0):
                        dg.set_tuning("sssp.delta", delta)
                        for direction in (0, 2, 1):
                            r = hc.sssp(dg, s, direction=direction)
                            assert np.array_equal(r.values, ref), (top, delta, direction)
                            modes = {e["mode"] for e in hc.epoch_trace(dg, "sssp")}
                            buckets = delta > 0 and direction != 1
                            assert ("promote" in modes) == (buckets and int(
                                (ref < hc.INF_DIST).sum() and ref[ref < hc.INF_DIST].max()) >= delta)
                            if buckets:
                                assert r.stats["pull_epochs"] == 0


def test_default_buckets_without_the_copy(hc, gpu):
    """A flat graph of more than 2^24 edges has buckets by default on the plain
    CSR as well, a smaller one does not."""
    for degree, buckets in ((9, True), (7, False)):
        g = hc.HostGraph.generate("uniform", 20, degree, weighted=True, seed=3)
        assert (g.num_edges >= 1 << 24) == buckets
        with hc.DeviceGraph(g) as dg:
            s = int(g.pick_sources(1)[0])
            ref = hc.sssp(dg, s).values
            dg.set_tuning("sssp.sorted", 0)
            assert np.array_equal(hc.sssp(dg, s).values, ref)
            assert ("promote" in {e["mode"] for e in hc.epoch_trace(dg, "sssp")}) == buckets


def test_sorted_sweeps_count_what_they_read(hc, gpu):
    """The trace and the byte count hold the pairs read, whether or not a distance
    is read for them: a star whose leaves lie at 1..200 is read once to lower the
    leaves and once more, but for the lightest, to find nothing; a heavy bucket's
    pushes read part of their frontier's edges."""
    d = 200
    g = hc.HostGraph.from_edges(np.zeros(d, np.int32), 1 + np.arange(d, dtype=np.int32), d + 1,
                                weights=1 + np.arange(d, dtype=np.int32))
    with hc.DeviceGraph(g) as dg:
        r = hc.sssp(dg, 0, direction=1)
        tr = hc.epoch_trace(dg, "sssp")
        assert [(e["frontier"], e["scanned"]) for e in tr] == [(d, d), (0, d - 1)]
        rows = 4 * (d + 2) + 4 * (d + 1)
        assert r.stats["alg_bytes"] == 2 * rows + 8 * (2 * d - 1) + 4 * d + 8 * d
    g = hc.HostGraph.generate("uniform", 16, 24, weighted=True, seed=2)
    with hc.DeviceGraph(g) as dg:
        dg.set_tuning("sssp.delta", 16)
        hc.sssp(dg, int(g.pick_sources(1)[0]))
        tr = hc.epoch_trace(dg, "sssp")
        pushes = [(e["scanned"], p["frontier_edges"]) for p, e in zip(tr, tr[1:])
                  if e["mode"] == "push" and p["frontier"] > 0]
        assert all(0 < got <= edges for got, edges in pushes)
        assert any(got < 0.8 * edges for got, edges in pushes)


def test_copy_is_built_once_there_is_memory(hc, gpu):
    """With the device's memory taken the queries run on the plain CSR; the first
    one after it is given back builds the copy."""
    g = hc.HostGraph.generate("uniform", 19, 16, weighted=True, seed=6)
    s = int(g.pick_sources(1)[0])
    with hc.DeviceGraph(g) as dg:
        dg.set_tuning("sssp.sorted", 0)
        ref = hc.sssp(dg, s).values
        dg.reset_tuning()
        hold = []
        try:
            while (free := hc.mem_get_info()[0]) > 96 << 20:
                hold.append(hc.DeviceArray(min(free - (64 << 20), 8 << 30) // 4, np.int32))
            print("held", sum(a.nbytes for a in hold) >> 20, "MiB", flush=True)
            short = hc.mem_get_info()[0]
            assert np.array_equal(hc.sssp(dg, s).values, ref)
            assert short - hc.mem_get_info()[0] < 8 * g.num_edges
        finally:
            for a in hold:
                a.free()
        free = hc.mem_get_info()[0]
        assert np.array_equal(hc.sssp(dg, s).values, ref)
        assert free - hc.mem_get_info()[0] >= 8 * g.num_edges


@pytest.mark.parametrize("max_weight,delta", [(0, -1), (255, -1), (255, 40), (70000, 9000)])
@pytest.mark.parametrize("seed", [0, 1])
def test_batched_sweeps_exact(hc, gpu, oracle, max_weight, delta, seed):
    """The batched sweep on the sorted adjacency, with and without buckets and
    push epochs: every column is the oracle's, and the plain sweep's."""
    g = _stars(hc, DEGREES, max_weight, seed)
    rng = np.random.default_rng(seed)
    for count, push_div in ((1, 16), (40, 0), (64, 4)):
        sources = rng.integers(0, g.num_nodes, count)
        with hc.DeviceGraph(g) as dg:
            dg.set_tuning("multi.delta", delta)
            dg.set_tuning("multi.push_div", push_div)
            r = hc.sssp_multi(dg, sources).values
            again = hc.sssp_multi(dg, sources).values
            dg.set_tuning("sssp.sorted", 0)
            assert np.array_equal(r, hc.sssp_multi(dg, sources).values)
        assert np.array_equal(r, again)
        for q in (0, count // 2, count - 1):
            ref = oracle.sssp_dijkstra(g.index, g.neighbors, g.weights, int(sources[q]))
            assert np.array_equal(r[q], ref), (count, q)
