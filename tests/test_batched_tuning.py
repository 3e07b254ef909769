"""The autotuner's grid of schedules (dyng_amd.batched.candidate_tunings). Host logic only; no device."""

from __future__ import annotations

import pytest

from dyng_amd import batched, sssp


@pytest.mark.parametrize("delta", [1, 7, 400])
def test_the_untuned_schedule_is_a_candidate(delta):
    grid = batched.candidate_tunings(delta)
    assert (sssp.Tuning(), delta) in grid
    assert all(width >= 1 for _, width in grid)
    assert len(grid) == len({(t.light_degree, t.chunk_edges, i % 3) for i, (t, _) in enumerate(grid)})
