"""The apply's groups of rows on the device: batch sizes around the groups' (one group holds 256 to 512
operations, a workgroup takes 512 at a time and a group 4096 at most), batches with more operations
on one row than a group takes, several operations on one pair, and the next batches after one that
did not fit. Rows, counts and trees equal the oracle's."""

from __future__ import annotations

import numpy as np
import pytest

import oracle
from tests.test_gpu_sssp import _assert_same_rows

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dg():
    import dyng_amd

    assert dyng_amd.available(), "no HIP device"
    return dyng_amd


def _graph(dg, n, m, K, directed, parallel, existing, seed):
    rng = np.random.default_rng(seed)
    src, dst, w = rng.integers(0, n, m), rng.integers(0, n, m), rng.integers(1, 60, (m, K))
    op = oracle.Props(directed=directed, allow_parallel=parallel, on_existing_insert=existing)
    sem = dg.BatchSemantics(on_existing_insert="upsert" if existing == 0 else "ignore")
    gp = dg.GraphProperties(directed=directed, parallel_edges="allow" if parallel else "forbid", semantics=sem)
    return (op, oracle.build_from_edges(n, src, dst, w, op),
            dg.Graph.from_edges(src, dst, w if K > 1 else w[:, 0], num_vertices=n, properties=gp), rng)


def _check(dg, op, og, hg, ot, r, ins, dels, label):
    og, a, c = oracle.update(og, ot, ins[0], ins[1], ins[2], dels[0], dels[1], props=op)
    st = dg.sssp.update(hg, dg.EdgeBatch(insert=(ins[0], ins[1], ins[2] if ins[2].shape[1] > 1 else ins[2][:, 0]),
                                         delete=dels), r)
    d, p = r.to_numpy()
    assert np.array_equal(d, ot.dist) and np.array_equal(p, ot.parent), label
    assert (st.invalidated, st.affected) == (c.invalidated, c.affected), label
    for f in ("inserted_edges", "updated_edges", "deleted_edges", "ignored_deletions", "ignored_insertions"):
        assert getattr(st.batch, f) == a.summary[f], (label, f)
    _assert_same_rows(hg, og)
    return og


@pytest.mark.parametrize("directed,parallel,K,existing",
                         [(True, False, 1, 0), (True, True, 1, 0), (False, False, 2, 0), (True, True, 3, 2),
                          (False, True, 1, 0), (True, False, 5, 2)])
def test_batch_sizes_around_the_groups(dg, directed, parallel, K, existing):
    print(f"[groups] directed {directed} parallel {parallel} K {K}", flush=True)
    op, og, hg, rng = _graph(dg, 1500, 9000, K, directed, parallel, existing, 5 + K)
    n = og.n
    ot, _ = oracle.compute(og, 0)
    r = dg.sssp.compute(hg, 0)
    for b, ops in enumerate([1, 2, 255, 256, 257, 511, 512, 513, 1023, 1025, 4097]):
        half = ops // 2
        rows = np.repeat(np.arange(og.n), np.diff(og.row_ptr))
        pick = rng.integers(0, og.m, half)
        dels = (rows[pick], og.col[pick].copy())
        few = 40 if b % 2 else n  # few rows: several operations on a pair
        ins = (rng.integers(0, few, ops - half), rng.integers(0, few, ops - half),
               rng.integers(1, 60, (ops - half, K)))
        if b == 5:
            n += 100  # the batch brings new vertices
            ins[0][-1] = n - 1
        og = _check(dg, op, og, hg, ot, r, ins, dels, f"batch {b}: {ops} operations")


@pytest.mark.parametrize("directed,parallel", [(True, False), (False, True)])
def test_more_operations_on_a_row_than_a_group_takes(dg, directed, parallel):
    op, og, hg, rng = _graph(dg, 6000, 20000, 1, directed, parallel, 0, 77)
    ot, _ = oracle.compute(og, 0)
    r = dg.sssp.compute(hg, 0)
    for b, on_hub in enumerate([4096, 4097, 300, 5000, 2000]):
        print(f"[groups] {on_hub} operations on row 7", flush=True)
        hub = rng.permutation(np.arange(8, og.n))[:on_hub]
        other = rng.integers(8, og.n, 200)
        ins = (np.concatenate([np.full(on_hub, 7), other]), np.concatenate([hub, rng.integers(8, og.n, 200)]),
               rng.integers(1, 60, (on_hub + 200, 1)))
        rows = np.repeat(np.arange(og.n), np.diff(og.row_ptr))
        pick = rng.choice(og.m, 50, replace=False)
        og = _check(dg, op, og, hg, ot, r, ins, (rows[pick], og.col[pick].copy()), f"batch {b}")
