"""Long rows on the device: lengths around the limits past which the engine cuts a row into chunks for
the whole grid (128 edges in a solve, 1024 in a repair's pull and relax phases, 2048 in its subtree
walk; chunks of 256 edges), and the frontiers without them, bit-exact against the oracle."""

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


def _hub_graph(degree: int, seed: int):
    """0 -> hub 1 -> `degree` vertices -> hub 2 (an in-row of `degree`) -> a tail of 40 vertices, and
    a costly detour 0 -> 3 -> both hubs that a cut tree edge falls back to; random cross edges."""
    rng = np.random.default_rng(seed)
    first, tail = 4, 4 + degree
    n = tail + 40
    leaves = np.arange(first, tail)
    chain = np.arange(tail, n)
    src = [np.array([0, 0, 3, 3]), np.full(degree, 1), leaves, np.concatenate([[2], chain[:-1]]),
           rng.integers(first, n, degree // 2)]
    dst = [np.array([1, 3, 1, 2]), leaves, np.full(degree, 2), chain, rng.integers(first, n, degree // 2)]
    w = [np.array([1, 5, 900, 4000]), rng.integers(1, 60, degree), rng.integers(1, 60, degree),
         rng.integers(1, 9, len(chain)), rng.integers(200, 400, degree // 2)]
    src, dst, w = np.concatenate(src), np.concatenate(dst), np.concatenate(w)
    _, keep = np.unique(src * n + dst, return_index=True)
    return n, src[keep], dst[keep], w[keep]


@pytest.mark.parametrize("degree", [127, 128, 129, 1023, 1024, 1025, 2047, 2048, 2049, 5 * 256, 5 * 256 + 1, 20_001])
def test_rows_around_the_chunk_limits(dg, degree):
    print(f"[long rows] degree {degree}", flush=True)
    n, src, dst, w = _hub_graph(degree, degree)
    og = oracle.build_from_edges(n, src, dst, w.reshape(-1, 1))
    g = dg.Graph.from_edges(src, dst, w, num_vertices=n)
    tree, _ = oracle.compute(og, 0)
    r = dg.sssp.compute(g, 0)
    d, p = r.to_numpy()
    assert np.array_equal(d, tree.dist) and np.array_equal(p, tree.parent), "compute"
    batches = [
        (([3], [4], [7]), ([0], [1])),  # the hub's tree edge: its whole row is walked, pulled and relaxed
        (([0], [1], [2]), ([3], [4])),  # back: one insertion lowers the whole row
        (([0, 2], [2, 1], [90, 3]), ([0], [3])),
    ]
    for b, (ins, dels) in enumerate(batches):
        ins, dels = tuple(np.array(x) for x in ins), tuple(np.array(x) for x in dels)
        og, _, c = oracle.update(og, tree, ins[0], ins[1], ins[2].reshape(-1, 1), dels[0], dels[1])
        st = dg.sssp.update(g, dg.EdgeBatch(insert=ins, delete=dels), r)
        d, p = r.to_numpy()
        assert np.array_equal(d, tree.dist) and np.array_equal(p, tree.parent), f"batch {b}"
        assert st.invalidated == c.invalidated and st.affected == c.affected, f"batch {b}"


@pytest.mark.parametrize("length,width", [(3000, 1), (700, 40)])
def test_a_deep_solve_runs_in_local_rounds(dg, length, width):
    """`width` chains of `length` vertices: narrow frontiers, which a solve relaxes in workgroup-local
    rounds too."""
    print(f"[deep solve] {width} chains of {length}", flush=True)
    rng = np.random.default_rng(length)
    n = 1 + length * width
    ids = 1 + np.arange(length * width).reshape(width, length)
    src = np.concatenate([np.zeros(width, np.int64), ids[:, :-1].reshape(-1), rng.integers(0, n, n // 10)])
    dst = np.concatenate([ids[:, 0], ids[:, 1:].reshape(-1), rng.integers(0, n, n // 10)])
    w = np.concatenate([rng.integers(1, 1001, width * length), rng.integers(50_000, 60_000, n // 10)])
    og = oracle.build_from_edges(n, src, dst, w.reshape(-1, 1))
    tree, _ = oracle.compute(og, 0)
    d, p = dg.sssp.compute(dg.Graph.from_edges(src, dst, w, num_vertices=n), 0).to_numpy()
    assert np.array_equal(d, tree.dist) and np.array_equal(p, tree.parent)


@pytest.mark.parametrize("recompute", [False, True])
def test_every_row_is_cut_into_chunks(dg, recompute):
    """A frontier of all vertices whose rows are all past the limit, in the smallest chunks: as many as the
    chunk list is made for, one per vertex and one per 16 slots of the long rows."""
    rng = np.random.default_rng(16)
    n, long_rows = 20_000, 40
    rest = np.arange(2, n)
    src = [np.array([0]), np.full(n - 2, 1), np.repeat(rest, 2), np.repeat(np.arange(2, 2 + long_rows), 1000)]
    dst = [np.array([1]), rest, rng.integers(0, n, 2 * (n - 2)), rng.integers(0, n, 1000 * long_rows)]
    src, dst = np.concatenate(src), np.concatenate(dst)
    _, keep = np.unique(src * n + dst, return_index=True)
    src, dst = src[keep], dst[keep]
    w = rng.integers(1, 9, len(src))
    og = oracle.build_from_edges(n, src, dst, w.reshape(-1, 1))
    g = dg.Graph.from_edges(src, dst, w, num_vertices=n)
    tree, _ = oracle.compute(og, 0)
    r = dg.sssp.compute(g, 0)
    r.set_tuning(dg.sssp.Tuning(light_degree=1, chunk_edges=16, recompute=recompute))
    none = np.zeros(0, np.int64)
    for b, (ins, dels) in enumerate([((0, 1, 7), (0, 1)), ((0, 1, 3), None), ((0, 2, 5), (0, 1))]):
        ins = tuple(np.array([x]) for x in ins)
        dels = tuple(np.array([x]) for x in dels) if dels else (none, none)
        og, _, c = oracle.update(og, tree, ins[0], ins[1], ins[2].reshape(-1, 1), dels[0], dels[1])
        st = dg.sssp.update(g, dg.EdgeBatch(insert=ins, delete=dels), r)
        d, p = r.to_numpy()
        assert np.array_equal(d, tree.dist) and np.array_equal(p, tree.parent), f"batch {b}"
        if not recompute:
            assert st.invalidated == c.invalidated and st.affected == c.affected, f"batch {b}"
