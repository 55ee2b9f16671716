"""The bench line's counted figures exist only for the sequence that was counted, and
the line stays valid JSON without them (no device needed)."""
import json
import os
import sys

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _plan(*counts):
    from khepri_amd.ops import Doublings
    return {k: Doublings(np.array(c)) for k, c in enumerate(counts)}


@pytest.mark.parametrize("counts,mean", [((), None), (([2, 2],), 2.0), (([1, 2], [3, 3]), 2.25), (([2, -1],), None)])
def test_counted_figures(counts, mean):
    sys.path.insert(0, ROOT)
    import bench
    doublings = bench.plan_doublings(_plan(*counts))
    assert doublings == mean
    roofline = bench.solve_roofline(doublings, 162, 1024, 1, 5.0, 5, "another workload")
    counted = bench.counted_line(doublings, 162, 30000.0)
    assert (roofline is None) == (counted is None) == (mean is None)
    json.dumps([roofline, counted], allow_nan=False)
