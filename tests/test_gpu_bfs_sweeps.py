"""GPU tests of the BFS loop where its launches divide: top-down epochs on both
sides of the size from which they mark by plain stores and collect by a scan,
and bottom-up rows whose scan ends at, or just past, the neighbours read ahead
(one on skewed graphs, four on flat ones).  Depths are unique; parents are
valid, and bottom-up the first frontier neighbour."""
from __future__ import annotations

import os
import subprocess
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _check(hc, oracle, g, sources, directions=(0, 1, 2)):
    with hc.DeviceGraph(g) as dg:
        for s in sources:
            depth = oracle.bfs_depth(g.index, g.neighbors, s)
            for direction in directions:
                b = hc.bfs(dg, s, direction=direction)
                assert np.array_equal(b.values, depth), (s, direction)
                assert oracle.verify_parents(depth, b.parents, s) == 0, (s, direction)
            _, _, dirs = oracle.bfs_do(g.index, g.neighbors, s)
            hc.bfs(dg, s)
            tr = hc.epoch_trace(dg, "bfs")
            assert [e["mode"] == "pull" for e in tr] == [bool(x) for x in dirs]
            reached = int((depth >= 0).sum())
            assert 1 + sum(e["frontier"] for e in tr) == reached


@pytest.mark.parametrize("wide", [False, True])
@pytest.mark.parametrize("leaves", [5000, 560000, 900000])
def test_heavy_top_down_epochs(hc, gpu, oracle, monkeypatch, leaves, wide):
    """Twelve hubs over a pool of leaves and a tail behind the leaves: the
    second epoch pushes 12 * leaves / 8 edges, many to the same leaves."""
    if wide:
        monkeypatch.setenv("HC_FORCE_OFF64", "1")
    rng = np.random.default_rng(leaves)
    hubs, tail = 12, 70
    per = leaves // 8
    src = [np.zeros(hubs, int)] + [np.full(per, 1 + h) for h in range(hubs)]
    dst = [1 + np.arange(hubs)] + [1 + hubs + rng.choice(leaves, per, replace=False)
                                   for _ in range(hubs)]
    last = hubs + leaves
    src.append(last + np.arange(tail))
    dst.append(last + 1 + np.arange(tail))
    g = hc.HostGraph.from_edges(np.concatenate(src).astype(np.int32),
                                np.concatenate(dst).astype(np.int32), 1 + hubs + leaves + tail)
    _check(hc, oracle, g, [0, int(dst[1][0])])


@pytest.mark.parametrize("n", [4, 5, 9])
def test_path_of_parallel_edges(hc, gpu, n):
    """A path whose links are 2^19 + n parallel edges: every level after the
    first is a heavy top-down epoch, so the loop takes two launch pairs for
    nearly every vertex."""
    k = (1 << 19) + n
    rows = [[v for v in (u - 1, u + 1) if 0 <= v < n] for u in range(n)]
    index = np.concatenate([[0], np.cumsum([k * len(r) for r in rows])]).astype(np.int64)
    g = hc.HostGraph.from_csr(index, np.repeat(np.concatenate(rows), k).astype(np.int32))
    with hc.DeviceGraph(g) as dg:
        for s in (0, n - 1, n // 2):
            b = hc.bfs(dg, s, direction=2)
            assert b.values.tolist() == [abs(v - s) for v in range(n)]
            assert b.parents.tolist() == [v - np.sign(v - s) for v in range(n)]
            assert b.stats["epochs"] == max(s, n - 1 - s) + 1


@pytest.mark.parametrize("wide", [False, True])
@pytest.mark.parametrize("degree", [1, 2, 3, 9])
def test_flat_rows_read_ahead(hc, gpu, oracle, monkeypatch, degree, wide):
    """Flat graphs above the size from which four neighbours are read ahead:
    rows of zero to a few dozen edges, vertices the source does not reach."""
    if wide:
        monkeypatch.setenv("HC_FORCE_OFF64", "1")
    rng = np.random.default_rng(degree)
    n = (1 << 19) + 77
    src = rng.integers(0, n - 1000, degree * n).astype(np.int32)
    dst = rng.integers(0, n - 1000, degree * n).astype(np.int32)
    g = hc.HostGraph.from_edges(src, dst, n)
    _check(hc, oracle, g, [int(src[0])], directions=(0, 1))


@pytest.mark.parametrize("n", [1, 2, 31, 32, 33, 1023, 1025, 8193, 32767, 32768, 32769])
def test_small_graphs_around_the_one_workgroup_limit(hc, gpu, oracle, n):
    """Graphs of up to 2^15 vertices run as one workgroup: its levels, trace and
    totals are those of the epoch loop."""
    rng = np.random.default_rng(n)
    src = rng.integers(0, n, 6 * n).astype(np.int32)
    dst = rng.integers(0, n, 6 * n).astype(np.int32)
    hub = np.zeros(min(n, 3000), np.int32)
    g = hc.HostGraph.from_edges(np.concatenate([src, hub]),
                                np.concatenate([dst, rng.permutation(n)[:hub.size].astype(np.int32)]),
                                n)
    _check(hc, oracle, g, [0, n // 2, n - 1])
    with hc.DeviceGraph(g) as dg:
        one = hc.bfs(dg, n // 2)
        hc.set_tuning("profile.kernel_events", 1)  # the epoch loop
        loop = hc.bfs(dg, n // 2)
        hc.reset_tuning()
        assert np.array_equal(one.values, loop.values)
        for key in ("epochs", "push_epochs", "pull_epochs", "reached"):
            assert one.stats[key] == loop.stats[key], key


FIRST_QUERY = """
import importlib, sys
sys.path.insert(0, sys.argv[1])
hc = importlib.import_module("hetero-compute_amd")
hc.check(hc.lib().hc_init(0))
g = hc.HostGraph.generate("kron", 12, 16, weighted=False, seed=1)
dg = hc.DeviceGraph(g)
out = hc.DeviceArray(g.num_nodes, "int32")
hc.synchronize()
free, _ = hc.mem_get_info()
hc.bfs(dg, 0, want_parents=False, depth_out=out, fetch=False)
print("took", free - hc.mem_get_info()[0])
"""


def test_first_small_query_of_a_process_takes_little_memory(hc, gpu):
    """A small graph's query loads the BFS loop's code only, not the many-graph
    launch's with its 32 MiB scratch array (which is no part of a server's
    budget either)."""
    root = os.path.dirname(os.path.dirname(os.path.abspath(hc.__file__)))
    run = subprocess.run([sys.executable, "-c", FIRST_QUERY, root], capture_output=True, text=True,
                         timeout=100)
    assert run.returncode == 0, run.stderr[-2000:]
    assert int(run.stdout.split()[-1]) < 32 << 20
