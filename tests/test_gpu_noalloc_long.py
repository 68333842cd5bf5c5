"""mfh_hier_peaks_noalloc at n = 32768 and 65536, where a call may take the
one-workgroup or the two-kernel path: after one allocating call over the whole
bank, calls over any part of it and with other bins find their buffers,
allocate nothing and give the same results."""
import ctypes

import numpy as np
import pytest

from test_zz_no_alloc import lib, make_ctx

pytestmark = pytest.mark.gpu

_vp = ctypes.c_void_p


def call(L, fn, h, d0, nd, t0, nt, binsize, thr, n, cthr):
    import torch
    nb = -(-n // binsize)
    idx = torch.full((nd, nt, nb), -7, dtype=torch.int64, device="cuda")
    val = torch.full((nd, nt, nb), 7.0, dtype=torch.complex64, device="cuda")
    torch.cuda.synchronize()
    args = [h, d0, nd, t0, nt, binsize, thr, 0, n, cthr, _vp(idx.data_ptr()), _vp(val.data_ptr())]
    if fn is L.mfh_hier_peaks_async:
        args.append(None)
    free0 = torch.cuda.mem_get_info()[0]
    assert fn(*args) == 0, L.mfh_last_error()
    assert L.mfh_sync(h) == 0
    if fn is L.mfh_hier_peaks_noalloc:
        assert torch.cuda.mem_get_info()[0] == free0
    return idx.cpu().numpy(), val.cpu().numpy()


@pytest.mark.parametrize("n", [32768, 65536])
def test_part_of_the_bank_after_a_call_over_all_of_it(n):
    L = lib()
    nd, nt = 4, 16
    h = make_ctx(L, n, nd, nt, 1024, 0, seed=n)
    try:
        fi, fv = call(L, L.mfh_hier_peaks_async, h, 0, nd, 0, nt, 4096, 3.0, n, 3.8)
        assert (fi >= 0).any() and (fi < 0).any()
        for d0, cd, t0, ct in [(1, 2, 3, 9), (0, 1, 0, 1), (2, 1, 15, 1), (0, 4, 9, 7), (0, 4, 0, 8), (0, 4, 0, 16)]:
            i, v = call(L, L.mfh_hier_peaks_noalloc, h, d0, cd, t0, ct, 4096, 3.0, n, 3.8)
            np.testing.assert_array_equal(i, fi[d0:d0 + cd, t0:t0 + ct])
            np.testing.assert_array_equal(v, fv[d0:d0 + cd, t0:t0 + ct])
        # one pair with as many bins in all as the bank had
        i, v = call(L, L.mfh_hier_peaks_noalloc, h, 3, 1, 5, 1, n // 512, 3.0, n, 0.0)
        ai, av = call(L, L.mfh_hier_peaks_async, h, 3, 1, 5, 1, n // 512, 3.0, n, 0.0)
        np.testing.assert_array_equal(i, ai)
        np.testing.assert_array_equal(v, av)
    finally:
        L.mfh_destroy(h)


@pytest.mark.parametrize("n,nd,nt,binsize", [(65536, 16, 32, 8), (32768, 16, 40, 8)])
def test_fewer_bins_than_the_call_that_built_the_buffers(n, nd, nt, binsize):
    """The part tables hold fewer pairs at once the more bins a pair has: the
    call with one bin, and so more pairs at once, finds its buffers too."""
    L = lib()
    h = make_ctx(L, n, nd, nt, 1024, 0, seed=n + 1)
    try:
        call(L, L.mfh_hier_peaks_async, h, 0, nd, 0, nt, binsize, 4.0, n, 3.8)
        i, v = call(L, L.mfh_hier_peaks_noalloc, h, 0, nd, 0, nt, n, 4.0, n, 3.8)
        ai, av = call(L, L.mfh_hier_peaks_async, h, 0, nd, 0, nt, n, 4.0, n, 3.8)
        np.testing.assert_array_equal(i, ai)
        np.testing.assert_array_equal(v, av)
        assert (ai >= 0).any() and (ai < 0).any()
    finally:
        L.mfh_destroy(h)
