"""Both sides of the lines at which n = 32768 and 65536 change their path, bit
for bit: parts merged by a pair's last part or by a finish launch (few or many
workgroups, small or large bin tables)."""
import numpy as np
import pytest

import apogee_amd as mf
from test_gpu_wide import bank, both

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [32768, 65536])
@pytest.mark.parametrize("nd,nt", [(1, 1), (2, 4), (4, 4), (1, 17), (5, 7)])
def test_part_tables_merged_in_either_place(n, nd, nt, gpu_device):
    D, T = bank(n, nd, nt, n + nd * nt)
    f = mf.MatchedFilter(n, nd, nt)
    f.set_data(D)
    f.set_templates(T)
    for bs, thr in [(n, 0.0), (n, 5.5), (n // 64, 0.0), (n // 64 - 1, 3.0), (n // 128, 0.0), (n // 1024, 0.0)]:
        wide, two = both(f, binsize=bs, threshold=thr)
        assert np.array_equal(wide, two), (n, nd, nt, bs, thr)
