"""Hierarchical graphs at the lengths of two paths: a change of the tuning keys
that decide which buffers a call needs ("wide", "big_chunk_mb") runs the next
call eagerly, so that a capture finds them all."""
import numpy as np
import pytest

import apogee_amd as mf
from test_gpu_wide import bank

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [32768, 65536])
def test_tuning_changes_between_captured_calls(n, gpu_device):
    D, T = bank(n, 4, 12, n + 9)
    h = mf.HierarchicalFilter(n, 4, 12, band=1024)
    h.set_data(D)
    h.set_templates(T)
    h.set_coarse_threshold(3.8)
    first = h.run(binsize=n // 8, threshold=3.0)
    assert (first["index"] >= 0).any() and (first["index"] < 0).any()
    h._gpu.set_tuning("graphs", 1)
    for key, value in [("wide", 1), ("wide", 2), ("big_chunk_mb", 1), ("big_chunk_mb", 128), ("wide", 1), ("wide", 0)]:
        h._gpu.set_tuning(key, value)
        for i in range(5):
            assert np.array_equal(h.run(binsize=n // 8, threshold=3.0), first), (key, value, i)
