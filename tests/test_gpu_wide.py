"""The one-workgroup path of n = 8192 ... 65536 (tuning key "wide") against the
path it replaces for many pairs, bit for bit, and against the FP64 oracle: one
bin and many, edges that fall inside a wave, more bins than one table and than
a wave looks up at once, thresholds that nothing, a few or every sample beats,
pair counts that are no multiple of the eight XCDs, NaN and infinity in a row.
"""
import numpy as np
import pytest

import apogee_amd as mf
from _parity import assert_peaks_match

pytestmark = pytest.mark.gpu

LENGTHS = [8192, 16384, 32768, 65536]
ALWAYS, NEVER = 1, 2


def bank(n, nd, nt, seed):
    rng = np.random.default_rng(seed)
    D = (rng.standard_normal((nd, n)) + 1j * rng.standard_normal((nd, n)))
    T = (rng.standard_normal((nt, n)) + 1j * rng.standard_normal((nt, n)))
    T /= np.sqrt((np.abs(T) ** 2).sum(axis=1, keepdims=True))
    f = np.arange(n)
    for d in range(nd):  # one planted peak per row, at an odd or even lag
        lag = int(rng.integers(n))
        D[d] += 9.0 * T[d % nt] * np.exp(-2j * np.pi * f * lag / n)
    return D.astype(np.complex64), T.astype(np.complex64)


def both(f, **kw):
    out = []
    for mode in (ALWAYS, NEVER):
        f._gpu.set_tuning("wide", mode)
        out.append(f.run(**kw))
    return out


@pytest.mark.parametrize("n", LENGTHS)
def test_paths_agree_bit_for_bit(n, gpu_device):
    D, T = bank(n, 3, 5, n)
    f = mf.MatchedFilter(n, 3, 5)
    f.set_data(D)
    f.set_templates(T)
    for bs, thr, win in [(n, 0.0, None), (n, 5.5, None), (n, 1000.0, None), (n, 0.0, (37, n - 11)),
                         (n // 8, 0.0, None), (n // 8, 5.5, None), (1024, 3.0, (64, n)), (1000, 0.0, (37, n - 11)),
                         (1000, 5.0, (37, n - 11)), (100, 0.0, None), (33, 0.0, (1, n - 1)), (7, 0.0, None),
                         (1, 0.0, (5, 700)), (1, 2.0, None), (64, 0.0, (n // 2, n // 2 + 65))]:
        a, b = both(f, binsize=bs, threshold=thr, window=win)
        assert np.array_equal(a, b), (n, bs, thr, win)
        if bs >= 1000:
            assert_peaks_match(D, T, a["index"], a["value"], bs, thr, win, context=str((n, bs, thr, win)))
    sub = f.run(binsize=n // 8, data=(1, 2), templates=(2, 3))
    f._gpu.set_tuning("wide", ALWAYS)
    assert np.array_equal(sub, f.run(binsize=n // 8)[1:3, 2:5])


@pytest.mark.parametrize("n", LENGTHS)
def test_nonfinite_rows_agree(n, gpu_device):
    D, T = bank(n, 4, 2, n + 1)
    D[1, 17] = np.nan
    D[2, 18] = np.inf
    D[3] = 0.0
    f = mf.MatchedFilter(n, 4, 2)
    f.set_data(D)
    f.set_templates(T)
    for bs, thr in [(n, 0.0), (1000, 0.0), (1000, 4.0)]:
        a, b = both(f, binsize=bs, threshold=thr)
        assert np.array_equal(a["index"], b["index"])
        assert np.array_equal(a["value"], b["value"], equal_nan=True)
        assert (a["index"][1] == -1).all() and (a["index"][3] == -1).all()


@pytest.mark.parametrize("n,nd,nt", [(8192, 13, 23), (16384, 7, 41), (32768, 5, 7), (65536, 9, 7)])
def test_automatic_choice_on_many_pairs(n, nd, nt, gpu_device):
    D, T = bank(n, nd, nt, n + 2)
    f = mf.MatchedFilter(n, nd, nt)
    f.set_data(D)
    f.set_templates(T)
    auto = f.run(binsize=1024, threshold=5.0)
    a, b = both(f, binsize=1024, threshold=5.0)
    assert np.array_equal(auto, a) and np.array_equal(a, b)
    assert (auto["index"] >= 0).any()


@pytest.mark.parametrize("n", LENGTHS)
def test_refine_lists_agree(n, gpu_device):
    D, T = bank(n, 5, 6, n + 3)
    h = mf.HierarchicalFilter(n, 5, 6, band=1024)
    h.set_data(D)
    h.set_templates(T)
    for gate in (0.0, 3.6, 4.4, 100.0):  # every pair, some, none; a shrinking and a growing list
        h.set_coarse_threshold(gate)
        for bs, thr in [(n, 0.0), (n // 8, 3.0)]:
            a, b = both(h, binsize=bs, threshold=thr)
            assert np.array_equal(a, b), (n, gate, bs)
            h._gpu.set_tuning("wide", 0)
            for _ in range(2):
                assert np.array_equal(a, h.run(binsize=bs, threshold=thr))


@pytest.mark.parametrize("n,nd,nt", [(32768, 3, 11), (65536, 3, 5), (262144, 1, 5)])
def test_parts_merge_alike_every_time(n, nd, nt, gpu_device):
    """Pairs whose parts run on different XCDs, merged by whichever part comes
    last: repeated calls, and calls of another shape between them, agree."""
    D, T = bank(n, nd, nt, n + 3)
    f = mf.MatchedFilter(n, nd, nt)
    f.set_data(D)
    f.set_templates(T)
    if n <= 65536:
        f._gpu.set_tuning("wide", ALWAYS)
    first = f.run(binsize=n // 16)
    assert_peaks_match(D, T, first["index"], first["value"], n // 16, 0.0, None, context=str(n))
    for i in range(40):
        assert np.array_equal(f.run(binsize=n // 16), first), i
        f.run(binsize=n // 8, data=(0, 1), templates=(i % nt, 1))
