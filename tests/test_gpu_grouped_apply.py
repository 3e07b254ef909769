"""The apply's groups of rows on the device (groups of 32 operations and more, by the batch's size; a
workgroup of 256 threads takes one, keeps fewer than 1024 operations in LDS and takes 4096 at most):
batch sizes around those, several operations on one pair, rows with as many operations as a group
takes and more, and the batches after one that did not fit. Rows, counts and trees equal the
oracle's. Which way a batch goes shows in no result, so the tests work out the fullest group from the
constants and the hash in dyng_amd/csrc/graph.hip."""

from __future__ import annotations

import pathlib
import re

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


SOURCE = (pathlib.Path(__file__).resolve().parents[1] / "dyng_amd" / "csrc" / "graph.hip").read_text()


def _constant(name):
    return int(re.search(rf"\b{name} = (\w+?)u?[,;]", SOURCE).group(1), 0)


CAP, LDS, PAUSE = _constant("kGroupCap"), _constant("kGroupLds"), _constant("kGroupPause")


def _fullest(n, src, dst, directed):
    """Operations of the fullest out-row and in-row group of a batch with these endpoints."""
    if not directed:
        loops = src == dst
        src, dst = np.concatenate([src, dst[~loops]]), np.concatenate([dst, src[~loops]])
        total = 2 * (len(loops))
    else:
        total = len(src)
    vbits, lb = int(n).bit_length(), 0
    while lb < min(_constant("kGroupBits"), vbits):
        ops = _constant("kGroupOpsFew") if lb < _constant("kGroupBitsFew") else \
            _constant("kGroupOpsSome") if lb < _constant("kGroupBitsSome") else _constant("kGroupOps")
        if (total // ops) >> (lb + 1) == 0:
            break
        lb += 1
    hashed = [((np.asarray(x, np.uint64) * np.uint64(_constant("kGroupHash"))) & np.uint64((1 << vbits) - 1))
              >> np.uint64(vbits - lb) for x in (src, dst)]
    return [int(np.bincount(h.astype(np.int64)).max()) for h in hashed]


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


@pytest.mark.parametrize("directed,parallel", [(True, False), (True, True), (False, False), (False, True)])
@pytest.mark.parametrize("on_row", [1, LDS - 1, LDS, LDS + 1, 2 * LDS, CAP - 1, CAP, CAP + 1])
def test_operations_on_one_row(dg, directed, parallel, on_row):
    """A new graph's first batch, all on one row: a group in LDS, a group in memory, a full one, and one that
    its workgroup cannot take. Another new graph's on the row's in-edges, and the row emptied."""
    op, og, hg, rng = _graph(dg, 6000, 20000, 1, directed, parallel, 0, on_row)
    ot, _ = oracle.compute(og, 0)
    r = dg.sssp.compute(hg, 0)
    ends = rng.permutation(np.arange(8, og.n))[:on_row]
    hub, w = np.full(on_row, 7), rng.integers(1, 60, (on_row, 1))
    fullest = _fullest(og.n, hub, ends, directed)
    print(f"[groups] {on_row} operations on a row, fullest groups {fullest}, directed {directed}, parallel {parallel}",
          flush=True)
    assert fullest[0] == on_row if directed else on_row <= fullest[0] <= on_row + 300
    none = np.zeros(0, np.int64)
    og = _check(dg, op, og, hg, ot, r, (hub, ends, w), (none, none), "out-row")
    _, og2, hg2, _ = _graph(dg, 6000, 20000, 1, directed, parallel, 0, on_row)  # another: not behind a pause
    ot2, _ = oracle.compute(og2, 0)
    _check(dg, op, og2, hg2, ot2, dg.sssp.compute(hg2, 0), (ends, hub, w), (none, none), "in-row")
    _check(dg, op, og, hg, ot, r, (none, none, np.zeros((0, 1), np.int64)), (hub, ends), "emptied")


@pytest.mark.parametrize("ops,on_row,fits", [(70_000, 3000, True), (100_000, 4000, False), (140_000, 3000, True),
                                             (140_000, 5000, False)])
@pytest.mark.parametrize("parallel", [False, True])
def test_a_full_row_in_a_large_batch(dg, ops, on_row, fits, parallel):
    """Rows with thousands of operations among many others: below and past the size up to which the merges
    are queued without the host, in groups and sorted."""
    op, og, hg, rng = _graph(dg, 30_000, 100_000, 1, True, parallel, 0, ops + on_row)
    ot, _ = oracle.compute(og, 0)
    r = dg.sssp.compute(hg, 0)
    rest = ops - on_row
    src = np.concatenate([np.full(on_row, 7), rng.integers(8, og.n, rest - rest // 3)])
    dst = np.concatenate([rng.permutation(np.arange(8, og.n))[:on_row], rng.integers(8, og.n, rest - rest // 3)])
    rows = np.repeat(np.arange(og.n), np.diff(og.row_ptr))
    pick = rng.choice(og.m, rest // 3, replace=False)
    dels = (rows[pick], og.col[pick].copy())
    fullest = _fullest(og.n, np.concatenate([src, dels[0]]), np.concatenate([dst, dels[1]]), True)
    print(f"[groups] {ops} operations, fullest groups {fullest}", flush=True)
    assert (max(fullest) <= CAP) == fits
    _check(dg, op, og, hg, ot, r, (src, dst, rng.integers(1, 60, (len(src), 1))), dels, f"{ops} operations")


def test_groups_again_after_the_pause(dg):
    """A batch that a group cannot take, the batches sorted after it, groups again, and a second such batch."""
    op, og, hg, rng = _graph(dg, 6000, 20000, 1, True, False, 0, 9)
    ot, _ = oracle.compute(og, 0)
    r = dg.sssp.compute(hg, 0)
    none = np.zeros(0, np.int64)
    for b in range(PAUSE + 5):
        on_row = CAP + 1 if b in (0, PAUSE + 3) else LDS + 200 if b > PAUSE else 300
        print(f"[groups] batch {b}: {on_row} operations on a row", flush=True)
        ends = rng.permutation(np.arange(8, og.n))[:on_row]
        assert (_fullest(og.n, np.full(on_row, 7), ends, True)[0] > CAP) == (on_row > CAP)
        og = _check(dg, op, og, hg, ot, r, (np.full(on_row, 7), ends, rng.integers(1, 60, (on_row, 1))), (none, none),
                    f"batch {b}")
