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


def test_a_heavy_result_beside_light_ones(dg):
    """A result whose last repair scanned millions of edges more than the others' has a launch of its own in
    the next one (all the device's workgroups, where the others have a share each)."""
    rng = np.random.default_rng(11)
    n0, m, light, K = 200_000, 5_000_000, 3, 1
    n = n0 + 500 * light
    src, dst = [rng.integers(1, n0, m)], [rng.integers(1, n0, m)]
    for i in range(light):  # small components of their own
        lo = n0 + 500 * i
        src.append(rng.integers(lo, lo + 500, 4000))
        dst.append(rng.integers(lo, lo + 500, 4000))
    src, dst = np.concatenate([[0], *src]), np.concatenate([[1], *dst])  # 0 -> 1, its only edge
    w = rng.integers(1, 90, (len(src), K))
    og = oracle.build_from_edges(n, src, dst, w)
    g = dg.Graph.from_edges(src, dst, w[:, 0], num_vertices=n)
    sources = [n0, 0, n0 + 500, n0 + 1000]
    trees = [oracle.compute(og, s)[0] for s in sources]
    results = [dg.sssp.compute(g, s) for s in sources]
    for b in range(3):  # the source's edge moves: its whole tree is invalidated
        few = rng.integers(n0, n, 40)
        ins = (np.concatenate([[0], few]), np.concatenate([[2 + b], n0 + (few - n0) // 500 * 500 + rng.integers(0, 500, 40)]),
               rng.integers(1, 90, (41, K)))
        dels = (np.array([0]), np.array([1 + b]))
        stats = dg.update(g, dg.EdgeBatch(insert=(ins[0], ins[1], ins[2][:, 0]), delete=dels), *results)
        og, _, counters = oracle.update_many(og, trees, ins[0], ins[1], ins[2], dels[0], dels[1])
        for i, (r, tree, c) in enumerate(zip(results, trees, counters)):
            d, p = r.to_numpy()
            assert np.array_equal(d, tree.dist) and np.array_equal(p, tree.parent), (b, i)
            assert (stats[i].invalidated, stats[i].affected) == (c.invalidated, c.affected), (b, i)
        edges = [s.device.pull_edges + s.device.relax_edges for s in stats]
        blocks = [s.device.blocks for s in stats]
        print(f"[teams] batch {b}: edges {edges}, workgroups {blocks}", flush=True)
        assert edges[1] > (4 << 20) + max(edges[0], *edges[2:]), edges
        assert len(set(blocks)) == 1 if b == 0 else blocks[1] > 2 * max(blocks[0], *blocks[2:]), blocks
