"""Planning a refine queue whose requests all have parameters of their own: the
time grows with the number of requests, not with its square."""
import time

import numpy as np
import pytest

import apogee_amd as mf

pytestmark = pytest.mark.gpu


def test_plan_of_many_parameter_sets():
    """A window per request is a group per request.  Compared with requests of
    one group, so the limit holds on any host: at 40000 requests a search of the
    groups for each of them takes over a hundred times as long."""
    n, nreq = 8192, 40000
    pool = np.zeros(2 * n, dtype=np.complex64)
    q = mf.RefineQueue()
    took = []
    for spread in (0, 1):
        start = np.arange(nreq, dtype=np.int64) % 4096 * spread
        end = n - np.arange(nreq, dtype=np.int64) // 4096 * spread
        best = np.inf
        for _ in range(2):
            t0 = time.perf_counter()
            q.plan(pool, n=np.full(nreq, n), data_offset=0, template_offset=n, candidates=1, binsize=n,
                   threshold=5.0, window=np.stack([start, end], axis=1))
            best = min(best, time.perf_counter() - t0)
        took.append(best)
        assert q.total == nreq
    assert took[1] < 20 * took[0], took
