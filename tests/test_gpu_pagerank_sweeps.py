"""GPU tests of the PageRank sweep where its work divides: rows at the edges of
the degree classes and of the chunks of long rows, row counts at the edges of a
wavefront's share, hubs held in LDS or not, and stops on either side of a batch
of launches."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# A score is rounded in its contribution, its compensated sum (2 units), the
# sum of its two parts, the product and the sum with the base: 6 * 2^-24 a step,
# carried on with factor 0.85: 6 * 2^-24 / 0.15 of the scores, which add up to
# at most 1.
L1_TOL = 6 * 2.0**-24 / 0.15


def _stars(hc, degrees, pool, rng, shuffle):
    """One vertex of each degree over a common pool of leaves, and 70 more
    vertices without edges."""
    src = np.repeat(np.arange(len(degrees)), degrees)
    dst = len(degrees) + np.concatenate([rng.permutation(pool)[:d] for d in degrees])
    n = len(degrees) + pool + 70
    if shuffle:
        p = rng.permutation(n)
        src, dst = p[src], p[dst]
    return hc.HostGraph.from_edges(src.astype(np.int32), dst.astype(np.int32), n)


@pytest.mark.parametrize("shuffle", [False, True])
@pytest.mark.parametrize("stage", [0, 7, 8192])
@pytest.mark.parametrize("degrees", [
    [1, 2, 4, 5, 6, 23, 24, 25, 63, 64, 65],
    [191, 192, 193, 255, 256, 257, 1023, 1024, 1025],
    [2047, 2048, 2049, 4095, 4096, 4097, 4099, 8191, 8193, 20000],
])
def test_rows_at_class_and_chunk_edges(hc, gpu, oracle, degrees, stage, shuffle):
    g = _stars(hc, degrees, 20000, np.random.default_rng(len(degrees)), shuffle)
    with hc.DeviceGraph(g) as dg:
        hc.set_tuning("pull.stage", stage)
        for iters in (1, 2, 3, 5):
            r = hc.pagerank(dg, tolerance=-1.0, max_iters=iters)
            assert r.stats["epochs"] == iters
            ref = oracle.pr_jacobi_f64(g.index, g.neighbors, 0.85, iters)
            assert np.abs(r.values.astype(np.float64) - ref).sum() <= L1_TOL
        hc.reset_tuning()


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 1023, 1025, 16383, 70001])
def test_row_counts_and_stops(hc, gpu, oracle, n):
    rng = np.random.default_rng(n)
    g = hc.HostGraph.from_edges(rng.integers(0, n, 8 * n).astype(np.int32),
                                rng.integers(0, n, 8 * n).astype(np.int32), n)
    with hc.DeviceGraph(g) as dg:
        for tol in (0.5, 1e-2, 1e-4, -1.0):
            r = hc.pagerank(dg, tolerance=tol)
            it = r.stats["epochs"]
            ref = oracle.pr_jacobi_f64(g.index, g.neighbors, 0.85, it)
            assert np.abs(r.values.astype(np.float64) - ref).sum() <= L1_TOL
            prev = oracle.pr_jacobi_f64(g.index, g.neighbors, 0.85, it - 1) if it > 1 else \
                np.full(n, 1.0 / n)
            assert abs(r.stats["residual"] - np.abs(ref - prev).sum()) <= 2 * L1_TOL
            assert it == 20 if tol < 0 else r.stats["residual"] < tol or it == 20
        assert np.array_equal(hc.pagerank(dg).values, hc.pagerank(dg).values)


@pytest.mark.parametrize("held", [False, True])
@pytest.mark.parametrize("shuffle", [False, True])
def test_epochs_over_ranges(hc, gpu, shuffle, held):
    """One epoch range by range, of the whole graph or of a handle that holds the
    range's rows only: rows are cut into chunks by the range's own edges.  Each
    score is rounded six times (see L1_TOL)."""
    rng = np.random.default_rng(4)
    g = _stars(hc, [1, 5, 24, 192, 1023, 1024, 1025, 2047, 2049, 4097, 8193, 20000], 20000, rng,
               shuffle)
    n = g.num_nodes
    contrib = (rng.random(n) / n).astype(np.float32)
    s_in = rng.random(n).astype(np.float32)
    inv = 1.0 / np.maximum(1, np.diff(g.index))
    sums = np.add.reduceat(np.append(contrib[g.neighbors].astype(np.float64), 0.0), g.index[:-1])
    ref = np.float32(0.15) / n + np.float32(0.85) * np.where(np.diff(g.index) > 0, sums, 0.0)
    bufs = [hc.DeviceArray.from_host(x) for x in (s_in, contrib, inv)]
    s_out, c_out = (hc.DeviceArray.from_host(np.zeros(n, np.float32)) for _ in range(2))
    whole = None if held else hc.DeviceGraph(g)
    cuts = [0, 1, 6, 12, 13, 500, n // 2, n // 2 + 64, n]
    resid = 0.0
    for a, b in zip(cuts, cuts[1:]):
        dg = hc.DeviceGraph(g, a, b) if held else whole
        resid += hc.pr_pull_epoch(dg, a, b, 0.85, *bufs, s_out, c_out)
        if held:
            dg.free()
    got = s_out.get().astype(np.float64)
    assert (np.abs(got - ref) <= 6 * 2.0**-24 * ref).all()
    assert np.abs(c_out.get() - got * inv).max() <= 2.0**-24 * (got * inv).max()
    assert abs(resid - np.abs(got - s_in).sum()) <= 1e-9 * resid
