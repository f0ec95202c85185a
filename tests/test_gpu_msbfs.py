"""GPU tests of the bit-parallel batched BFS at the sizes where its kernels
divide their work: rows at the edges of the degree classes and hub chunks,
push windows of one to several thousand vertices, chunks of one edge to a
hub's, every level forced into one direction, one to 64 sources, 8-byte
offsets and unsorted vertex orders.  Depths are unique: equality with the
oracle."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

DEGREES = [1, 4, 5, 64, 65, 128, 511, 513, 2047, 2048, 2049, 4097, 9000]


@pytest.fixture(autouse=True)
def restore(hc):
    yield
    hc.reset_tuning()


def _stars(hc, seed, relabel):
    rng = np.random.default_rng(seed)
    hubs, leaves = len(DEGREES), 12000
    src, dst = [], []
    for h, d in enumerate(DEGREES):
        src.append(np.full(d, h))
        dst.append(hubs + rng.choice(leaves, d, replace=False))
    # A path through the last leaves: many levels of one vertex.
    path = hubs + np.arange(leaves - 300, leaves - 1)
    src += [path, hubs + rng.integers(0, leaves - 400, 3000)]
    dst += [path + 1, hubs + rng.integers(0, leaves - 400, 3000)]
    return hc.HostGraph.from_edges(np.concatenate(src).astype(np.int32),
                                   np.concatenate(dst).astype(np.int32), hubs + leaves,
                                   relabel=relabel)


@pytest.mark.parametrize("alpha", [1, 16, 1 << 20])
@pytest.mark.parametrize("relabel,wide", [(True, False), (False, True)])
def test_depths_in_every_direction(hc, gpu, oracle, monkeypatch, alpha, relabel, wide):
    if wide:
        monkeypatch.setenv("HC_FORCE_OFF64", "1")
    g = _stars(hc, 3, relabel)
    hc.set_tuning("msbfs.alpha", alpha)
    rng = np.random.default_rng(alpha)
    with hc.DeviceGraph(g) as dg:
        for count in (1, 33, 64):
            sources = rng.integers(0, g.num_nodes, count)
            sources[count // 2] = sources[0]  # a source twice
            r = hc.bfs_multi(dg, sources)
            for q, s in enumerate(sources):
                ref = oracle.bfs_depth(g.index, g.neighbors, int(s))
                assert np.array_equal(r.values[q], ref), (count, q)


@pytest.mark.parametrize("size", [4095, 4096, 4097, 8193, 20000])
def test_push_windows(hc, gpu, oracle, size):
    """A frontier of `size` vertices in one level, each with one edge on (and
    one of them with many)."""
    mid = 1 + np.arange(size)
    end = 1 + size + np.arange(size)
    hub = np.full(700, 1 + size // 2)
    src = np.concatenate([np.zeros(size, int), mid, hub])
    dst = np.concatenate([mid, end, 1 + 2 * size + np.arange(700)])
    g = hc.HostGraph.from_edges(src.astype(np.int32), dst.astype(np.int32), 2 * size + 701)
    hc.set_tuning("msbfs.alpha", 1)
    with hc.DeviceGraph(g) as dg:
        sources = [0, 1, size, 2 * size]
        r = hc.bfs_multi(dg, sources)
        for q, s in enumerate(sources):
            assert np.array_equal(r.values[q], oracle.bfs_depth(g.index, g.neighbors, s)), q


@pytest.mark.parametrize("wide", [False, True])
@pytest.mark.parametrize("leaves", [1, 61, 62, 63, 190, 255, 256, 257, 1100])
def test_short_lists(hc, gpu, oracle, monkeypatch, leaves, wide):
    """A ladder of 40 rungs of 80 vertices whose every tenth rung has one vertex
    with `leaves` leaves: lists of some hundred edges, rows on both sides of a
    group's 64 edges and of a wavefront's 256 beyond them, and of the mean up to
    which a list is short."""
    if wide:
        monkeypatch.setenv("HC_FORCE_OFF64", "1")
    width, rungs = 80, 40
    v = np.arange(width * (rungs - 1))
    hubs = width * np.arange(0, rungs, 10) + 7
    n = width * rungs + leaves * hubs.size
    src = np.concatenate([v, v, np.repeat(hubs, leaves)])
    dst = np.concatenate([v + width, v // width * width + width + (v + 1) % width,
                          width * rungs + np.arange(leaves * hubs.size)])
    p = np.random.default_rng(leaves).permutation(n)
    g = hc.HostGraph.from_edges(p[src].astype(np.int32), p[dst].astype(np.int32), n)
    hc.set_tuning("msbfs.alpha", 1)
    with hc.DeviceGraph(g) as dg:
        for sources in ([p[0]], p[[7, 8, n - 1]], p[:64]):
            r = hc.bfs_multi(dg, sources)
            for q, s in enumerate(sources):
                assert np.array_equal(r.values[q], oracle.bfs_depth(g.index, g.neighbors, int(s)))
