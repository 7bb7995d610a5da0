"""The persistent kernel's claims at the ends of its grid: one workgroup (its
four waves share one poller), a few, and more than stay resident; bursts of
one-item passes longer than the 64 passes a claim looks at, with integer
requests that need a second pass, a pass of many items among them, and a
pause long enough for the launch to end between two bursts."""
import time

import numpy as np
import pytest

import permanent_amd as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("grid", [1, 3, 1024])
def test_bursts_on_every_grid(grid):
    mats = [P.synthetic_matrix(9 + i % 9, 0.3 + 0.05 * (i % 11), 900 + i, full_support=True)
            for i in range(200)]
    mats += [P.synthetic_matrix(20 + i % 4, 0.5, 950 + i, binary=True).astype(np.int32)
             for i in range(6)]
    mats.append(P.synthetic_matrix(25, 0.4, 77, full_support=True))  # many items
    reqs = P.RequestBatch([P.Request(m) for m in mats])
    want = [P.dense(m) for m in mats]
    first = None
    with P.Server(grid=grid, idle_us=500.0) as s:
        for burst in range(3):
            ids = s.submit_batch(reqs)
            res, _ = s.wait_many_raw(ids)
            got = [(r.value, r.sum_lo, r.mode, r.certified) for r in res]
            if first is None:
                first = got
            assert got == first, burst
            if burst == 1:
                time.sleep(0.05)  # the launch ends; the next burst starts another
    for m, r, w in zip(mats, res, want):
        assert abs(r.value - w.value) <= max(r.err_bound, r.err_est) + w.stated, (m.shape, w)
        assert r.certified
