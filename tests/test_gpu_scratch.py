"""The applies' scratch on the device: graphs updated in turn and from several threads share their device's
pool, hold none of it between updates, and keep the oracle's rows and trees."""

from __future__ import annotations

import ctypes
import threading

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


def _free_bytes(dg):
    """The device's free memory, from the HIP runtime that the library is linked to."""
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    dg.synchronize()
    assert dg._lib.lib().hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


def test_graphs_hold_no_scratch_between_updates(dg):
    """The scratch of a batch of 300,000 operations is about 150 MB; a graph keeps its rows and the batch's
    operations only (a few MB)."""
    n, ops = 2000, 300_000
    rng = np.random.default_rng(3)
    src, dst, w = rng.integers(0, n, 8000), rng.integers(0, n, 8000), rng.integers(1, 60, 8000)
    ins = (rng.integers(0, n, ops), rng.integers(0, n, ops), rng.integers(1, 60, ops))
    graphs, free = [], []
    for i in range(5):
        print(f"[scratch] graph {i}", flush=True)
        g = dg.Graph.from_edges(src, dst, w, num_vertices=n)
        g.apply(dg.EdgeBatch(insert=ins))
        graphs.append(g)
        free.append(_free_bytes(dg))
    per_graph = (free[0] - free[-1]) / (len(graphs) - 1)
    print(f"[scratch] {per_graph / 1e6:.1f} MB a graph", flush=True)
    assert per_graph < 40e6


def test_graphs_on_several_threads(dg):
    """Batches of very different sizes at the same time: a block each."""
    errors = []

    def work(seed):
        try:
            rng = np.random.default_rng(seed)
            n, m = 3000, 20_000
            src, dst, w = rng.integers(0, n, m), rng.integers(0, n, m), rng.integers(1, 60, (m, 1))
            og = oracle.build_from_edges(n, src, dst, w)
            g = dg.Graph.from_edges(src, dst, w[:, 0], num_vertices=n)
            tree, _ = oracle.compute(og, 0)
            r = dg.sssp.compute(g, 0)
            for ops in (7, 3000, 20, 15_000, 600, 15_000):
                ops += seed
                ins = (rng.integers(0, n, ops), rng.integers(0, n, ops), rng.integers(1, 60, (ops, 1)))
                rows = np.repeat(np.arange(og.n), np.diff(og.row_ptr))
                pick = rng.choice(og.m, ops // 3, replace=False)
                dels = (rows[pick], og.col[pick].copy())
                og, _, c = oracle.update(og, tree, ins[0], ins[1], ins[2], dels[0], dels[1])
                st = dg.sssp.update(g, dg.EdgeBatch(insert=(ins[0], ins[1], ins[2][:, 0]), delete=dels), r)
                d, p = r.to_numpy()
                assert np.array_equal(d, tree.dist) and np.array_equal(p, tree.parent), (seed, ops)
                assert (st.invalidated, st.affected) == (c.invalidated, c.affected), (seed, ops)
                _assert_same_rows(g, og)
        except BaseException as e:  # noqa: BLE001  (reported by the test's thread)
            errors.append(e)

    threads = [threading.Thread(target=work, args=(s,)) for s in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors
