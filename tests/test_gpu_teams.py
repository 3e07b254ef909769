"""Several results repaired side by side in one launch: fewer results than teams, as many, and more (a
second launch), different sources and weight columns, with and without parallel edges, small and large
batches. Every tree and count equals the oracle's."""

from __future__ import annotations

import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dg():
    import dyng_amd

    assert dyng_amd.available(), "no HIP device"
    return dyng_amd


@pytest.mark.parametrize("count", [2, 3, 4, 5, 9])
@pytest.mark.parametrize("parallel", [False, True])
def test_results_side_by_side(dg, count, parallel):
    print(f"[teams] {count} results, parallel edges {parallel}", flush=True)
    rng = np.random.default_rng(count)
    n, m, K = 5000, 30_000, 2
    src, dst, w = rng.integers(0, n, m), rng.integers(0, n, m), rng.integers(1, 90, (m, K))
    op = oracle.Props(allow_parallel=parallel)
    gp = dg.GraphProperties(parallel_edges="allow" if parallel else "forbid")
    og = oracle.build_from_edges(n, src, dst, w, op)
    g = dg.Graph.from_edges(src, dst, w, num_vertices=n, properties=gp)
    sources = rng.permutation(n)[:count]
    trees, results = [], []
    for i, s in enumerate(sources):
        trees.append(oracle.compute(og, int(s), i % K)[0])
        results.append(dg.sssp.compute(g, int(s), objective=i % K))
    for b, ops in enumerate([1, 60, 3000, 70_000]):
        rows = np.repeat(np.arange(og.n), np.diff(og.row_ptr))
        pick = rng.choice(og.m, min(ops // 2, og.m // 2), replace=False)
        dels = (rows[pick], og.col[pick].copy())
        k = ops - ops // 2
        ins = (rng.integers(0, n, k), rng.integers(0, n, k), rng.integers(1, 90, (k, K)))
        stats = dg.update(g, dg.EdgeBatch(insert=ins, delete=dels), *results)
        og, _, counters = oracle.update_many(og, trees, ins[0], ins[1], ins[2], dels[0], dels[1], props=op)
        for i, (r, tree, c) in enumerate(zip(results, trees, counters)):
            d, p = r.to_numpy()
            assert np.array_equal(d, tree.dist) and np.array_equal(p, tree.parent), (b, i)
            assert (stats[i].invalidated, stats[i].affected) == (c.invalidated, c.affected), (b, i)
