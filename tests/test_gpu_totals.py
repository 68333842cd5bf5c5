"""The total of reported bins that runs with host results return through the C
ABI: counted by default and whenever per-pair counts are asked for, 0 when
tuning key "totals" turns the pass off; the results are the same."""
import ctypes

import numpy as np
import pytest

import apogee_amd as mf
from apogee_amd import _hip

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pinned", [True, False])
@pytest.mark.parametrize("nb", [1, 5])
def test_totals_key(pinned, nb, gpu_device):
    rng = np.random.default_rng(nb)
    n, nd, nt = 1024, 3, 7
    D = (rng.standard_normal((nd, n)) + 1j * rng.standard_normal((nd, n))).astype(np.complex64)
    T = (rng.standard_normal((nt, n)) + 1j * rng.standard_normal((nt, n))).astype(np.complex64)
    f = mf.MatchedFilter(n, nd, nt)
    f.set_data(D)
    f.set_templates(T)
    L, c = _hip.lib(), f._gpu
    bs = -(-n // nb)
    thr = float(np.median(np.abs(f.run(binsize=bs)["value"])))

    def call(counts):
        rec = _hip._records_array((nd, nt, nb), mf.PEAK_DTYPE) if pinned else np.empty((nd, nt, nb), mf.PEAK_DTYPE)
        cnt = np.full((nd, nt), -1, np.int32)
        total = L.mfh_flat_peaks_rec(c.handle, 0, nd, 0, nt, bs, thr, 0, n, ctypes.c_void_p(rec.ctypes.data),
                                     ctypes.c_void_p(cnt.ctypes.data) if counts else None)
        return total, rec.copy(), cnt

    c.set_tuning("totals", 1)
    total, rec, _ = call(False)
    assert 0 < total == int((rec["index"] >= 0).sum()) < rec.size
    c.set_tuning("totals", 0)
    off, same, _ = call(False)
    assert off == 0 and np.array_equal(rec, same)
    again, same, cnt = call(True)
    assert again == total and np.array_equal(rec, same)
    assert np.array_equal(cnt, (rec["index"] >= 0).sum(axis=2))
    with pytest.raises(RuntimeError):
        c.set_tuning("totals", 2)
