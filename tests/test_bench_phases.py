"""bench.py's phases of the plain step: every ms of the timings goes to one
phase, named after the kernels that ran it, and every phase but the queue
passes has its own minimum traffic."""
import sys

import pytest

from conftest import ROOT

sys.path.insert(0, ROOT)
import bench  # noqa: E402


@pytest.mark.parametrize("row", [False, True])
@pytest.mark.parametrize("slots", [1, 2, 4])
@pytest.mark.parametrize("k", [3, 5, 10, 16])
def test_phases_cover_the_step(k, slots, row):
    kt = [0.01, 0.09, 0.0, 0.0 if row else 0.05, 0.0 if row or (k in (5, 10) and slots == 2) else 0.03, 0.02]
    p = bench.plain_phases(kt, k, slots, row)
    assert abs(sum(p.values()) - (kt[0] + kt[1] + kt[3])) < 1e-12
    assert ("row_step" in p) == row and ("orca_queues" in p) == (not row)
    assert ("knn_orca_main" in p) == (not row and k in (5, 10) and slots == 2)
    assert all(v >= 0.0 for v in p.values())
    own = bench.own_bytes_per_agent(k, 4.0)
    assert set(p) - {"orca_queues"} <= set(own)
