"""Refine queue plans: the time for requests that all have parameters of their own
grows with their number, not with its square; groups of 8192 and 16384 points on
either side of the lines from which they get a list launch."""
import time

import numpy as np
import pytest

import apogee_amd as mf
from test_gpu_refine import check_against_per_request, cnoise, stage

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


@pytest.mark.parametrize("n,bins,thr,line", [(8192, 1, 60.0, 350), (16384, 16, 60.0, 300), (8192, 8, 60.0, 512),
                                             (16384, 8, 60.0, 400), (8192, 1, 0.0, 512), (16384, 16, 0.0, 400),
                                             (8192, 8, 0.0, 1024), (16384, 8, 0.0, 1024)])
def test_groups_on_either_side_of_their_lines(n, bins, thr, line, gpu_device):
    """One pair short of a list launch and just enough for one, by threshold and
    bins, beside shorter requests: the results of the flat filter, each time."""
    rng = np.random.default_rng(n + line)
    data, bank = cnoise(rng, n), cnoise(rng, (line, n))
    for c in (line - 1, line):
        reqs = [(data, bank[:c], n // bins, thr, None),
                (cnoise(rng, 1024), cnoise(rng, (3, 1024)), 100, 0.0, None),
                (cnoise(rng, n), cnoise(rng, (2, n)), 999, 300.0, (5, n - 3))]
        q = mf.RefineQueue()
        stage(q, reqs)
        for _ in range(3):      # eager, captured, replayed
            check_against_per_request(reqs, q.run(), gpu_device, "%d of %d" % (c, line))
