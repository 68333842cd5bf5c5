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


@pytest.mark.parametrize("n,cap,left", [(65536, 150, 80), (65536, 68, 40), (32768, 60, 8)])
def test_capture_by_capacity_after_eager_calls_by_length(n, cap, left, gpu_device):
    """An eager call goes by the survivors of the call before, a captured one by
    the list's capacity, maybe on the other path, after calls of other shapes."""
    D, T = bank(n, 1, 160, n + 11)
    h = mf.HierarchicalFilter(n, 1, 160, band=512)
    h.set_data(D)
    h.set_templates(T)
    h.set_coarse_threshold(1e6)
    h.run(binsize=n, threshold=3.0)   # sets the band
    coarse = np.sort(h._gpu.hier_coarse_max(0, 1, 0, cap, 0, n, 0).ravel())[::-1]
    h.set_coarse_threshold(float((coarse[left - 1] + coarse[left]) / 2))
    kw = dict(binsize=n // 4, threshold=3.0, templates=(0, cap))
    want = h.run(**kw)
    assert h.run(**kw).shape == want.shape
    h._gpu.set_tuning("graphs", 1)
    h.run(binsize=n // 4, threshold=3.0, templates=(0, 100))
    h.run(binsize=n // 2, threshold=3.0)
    for i in range(5):
        assert np.array_equal(h.run(**kw), want), i
    assert h._gpu.last_refinements == left
