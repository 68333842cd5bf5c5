"""Both sides of the lines at which n = 32768 and 65536 change their path, bit
for bit: parts merged by a pair's last part or by a finish launch (few or many
workgroups, small or large bin tables), and the one-workgroup or the two-kernel
path by pairs, bins and threshold, in plain calls, series and allocation-free
lists."""
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


@pytest.mark.parametrize("n,pairs", [(8192, (256, 257, 512, 513)), (32768, (31, 32, 103, 104)),
                                     (65536, (71, 72, 103, 104, 128, 129, 191, 192, 257, 268))])
def test_automatic_choice_on_either_side_of_its_lines(n, pairs, gpu_device):
    D, T = bank(n, 1, max(pairs), n + 5)
    f = mf.MatchedFilter(n, 1, max(pairs))
    f.set_data(D)
    f.set_templates(T)
    for p in pairs:
        for bs, thr in [(n, 5.5), (n // 8, 0.0), (1000, 0.0)]:
            f._gpu.set_tuning("wide", 0)
            auto = f.run(binsize=bs, threshold=thr, templates=(0, p))
            wide, two = both(f, binsize=bs, threshold=thr, templates=(0, p))
            assert np.array_equal(auto, wide) and np.array_equal(auto, two), (n, p, bs, thr)


@pytest.mark.parametrize("n,nt", [(8192, 130), (32768, 30), (65536, 27)])
def test_series_windows_on_either_path(n, nt, gpu_device):
    """Blocks with windows of their own, with a threshold and without one (whose
    lines differ): the blocks' windows reach the path that the run takes."""
    rng = np.random.default_rng(n)
    _, T = bank(n, 1, nt, n + 6)
    x = (rng.standard_normal(3 * n) + 1j * rng.standard_normal(3 * n)).astype(np.complex64)
    f = mf.MatchedFilter(n, 1, nt)
    f.set_templates(T)
    c = f._gpu
    starts = np.array([0, n // 2, n, 3 * n // 2])
    lo = np.array([0, n // 4, n // 4, n // 2 + 1])
    hi = lo + n // 2 - 1
    for bs, thr in [(n, 0.0), (n // 16, 0.0), (n // 16, 3.0)]:
        got = []
        for mode in (0, 1, 2):
            c.set_tuning("wide", mode)
            got.append(c.run_series(x, starts, lo, hi, 0, nt, bs, thr, records=mf.PEAK_DTYPE)[0])
        assert np.array_equal(got[0], got[1]) and np.array_equal(got[0], got[2]), (n, bs, thr)
        for b in range(4):
            one = c.run_series(x, starts[b:b + 1], lo[b:b + 1], hi[b:b + 1], 0, nt, bs, thr, records=mf.PEAK_DTYPE)[0]
            assert np.array_equal(got[0][b:b + 1], one), (n, bs, thr, b)


@pytest.mark.parametrize("n", [8192, 16384, 32768, 65536])
def test_winners_found_either_way(n, gpu_device):
    """256 bins, whose winners a wave visits, and a few more, which the samples
    look up: all samples candidates, some, a few."""
    D, T = bank(n, 2, 3, n + 8)
    f = mf.MatchedFilter(n, 2, 3)
    f.set_data(D)
    f.set_templates(T)
    for bs, window in [(n // 256, None), (n // 256 - 1, None), (n // 256, (1, n)), (17, (3, 3 + 17 * 256 + 1))]:
        for thr in (0.0, 2.5, 5.0):
            wide, two = both(f, binsize=bs, threshold=thr, window=window)
            assert np.array_equal(wide, two), (n, bs, window, thr)


@pytest.mark.parametrize("n,pairs,bs", [(8192, 600, 24), (8192, 300, 200), (32768, 48, 8), (32768, 130, 100), (65536, 66, 16),
                                        (65536, 120, 128)])
def test_automatic_choice_by_bin_width(n, pairs, bs, gpu_device):
    D, T = bank(n, 1, pairs, n + 7)
    f = mf.MatchedFilter(n, 1, pairs)
    f.set_data(D)
    f.set_templates(T)
    for thr in (0.0, 4.0):
        f._gpu.set_tuning("wide", 0)
        auto = f.run(binsize=bs, threshold=thr)
        wide, two = both(f, binsize=bs, threshold=thr)
        assert np.array_equal(auto, wide) and np.array_equal(auto, two), thr
