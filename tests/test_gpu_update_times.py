"""The times an update reports: the apply's and the engine's stream time."""

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


def test_an_apply_planned_again_counts_its_second_plan(dg):
    """Vertex 0's row outgrows its tail: the first full merge needs staging that the graph does not have, so
    the merges are held back and planned again on the host, two synchronizations and copies later than the
    same growth of another row afterwards. The apply's time holds them."""
    rng = np.random.default_rng(5)
    n, m = 3000, 30_000
    src, dst, w = rng.integers(2, n, m), rng.integers(2, n, m), rng.integers(1, 60, m)
    for hub in (0, 1):
        src = np.concatenate([src, np.full(200, hub)])
        dst = np.concatenate([dst, rng.permutation(np.arange(2, n))[:200]])
        w = np.concatenate([w, rng.integers(1, 60, 200)])
    og = oracle.build_from_edges(n, src, dst, w.reshape(-1, 1))
    g = dg.Graph.from_edges(src, dst, w, num_vertices=n)
    tree, _ = oracle.compute(og, 2)
    r = dg.sssp.compute(g, 2)
    plans, apply_ms = [], []
    for hub in (2, 3, 0, 1):  # two batches of short tails first: the scratch is there
        far = rng.permutation(np.arange(2, n))[:300]
        ins_src = np.full(300, hub) if hub < 2 else rng.integers(2, n, 300)
        ins = (ins_src, far, rng.integers(1, 60, 300))
        none = np.zeros(0, np.int64)
        og, _, c = oracle.update(og, tree, ins[0], ins[1], ins[2].reshape(-1, 1), none, none)
        st = dg.sssp.update(g, dg.EdgeBatch(insert=ins), r)
        d, p = r.to_numpy()
        assert np.array_equal(d, tree.dist) and np.array_equal(p, tree.parent)
        assert (st.invalidated, st.affected) == (c.invalidated, c.affected)
        plans.append(st.batch.host_plans)
        apply_ms.append(st.apply_ms)
        assert st.engine_ms == st.device.kernel_ms > 0
    print(f"[times] host plans {plans}, apply ms {apply_ms}", flush=True)
    assert plans == [0, 0, 1, 0]
    assert apply_ms[2] > 1.5 * apply_ms[3]
