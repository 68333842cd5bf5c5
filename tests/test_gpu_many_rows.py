"""More data rows than a launch grid's second dimension holds, whatever tile is
tuned: the same results as in two halves."""
import numpy as np
import pytest

import apogee_amd as mf

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,nd,nt", [(64, 65536, 1), (64, 131075, 5), (1024, 70001, 2)])
def test_more_rows_than_the_grid(n, nd, nt, gpu_device):
    rng = np.random.default_rng(nd)
    f = mf.MatchedFilter(n, nd, nt)
    f.set_data(rng.standard_normal((nd, 2 * n), dtype=np.float32).view(np.complex64))
    f.set_templates(rng.standard_normal((nt, 2 * n), dtype=np.float32).view(np.complex64))
    half = nd // 2
    f._gpu.set_tuning("dpw", 4)
    parts = [f.run(threshold=0.0, data=s) for s in ((0, half), (half, nd - half))]
    for dpw in (0, 1, 3):
        f._gpu.set_tuning("dpw", dpw)
        got = f.run(threshold=0.0)
        assert np.array_equal(got[:half], parts[0]) and np.array_equal(got[half:], parts[1]), dpw
