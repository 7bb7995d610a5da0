"""perm_batch_compute_dense at every kind of work split: its room for each
matrix comes from the order alone, before the matrix is prepared, also where
the split leaves the class walk out (items below 2^11 or above 2^21 subsets)."""
import numpy as np
import pytest

import permanent_amd as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("item_log2", [0, 6, 8, 10, 11, 21, 22, 30])
def test_one_call_has_the_bits_of_add_and_run(item_log2):
    """Orders on both sides of the class walk's smallest (12) and of the split
    past its longest walk table (n = 23 at 2^22), sparse to full."""
    mats = [P.synthetic_matrix(n, d, 700 + 10 * n + k, full_support=True)
            for n in (4, 11, 12, 16, 22, 23, 24) for k, d in enumerate((0.2, 0.5, 1.0))]
    mats.append(P.synthetic_matrix(20, 0.4, 3, binary=True).astype(np.int32))
    b = P.Batch(item_log2=item_log2)
    b.add_many(mats)
    want, _ = b.run()
    b.close()
    b = P.Batch(item_log2=item_log2)
    out = (P.PermResultC * len(mats))()
    b.compute_prepared(P.BatchInputs(mats), out, threads=4)
    again, _ = b.run()
    b.close()
    for m, w, c, a in zip(mats, want, out, again):
        r = P.PermResult.from_c(c)
        key = (w.value, w.sum_hi, w.sum_lo, w.abs_sum, w.err_est, w.mode, w.certified)
        for q in (r, a):
            assert (q.value, q.sum_hi, q.sum_lo, q.abs_sum, q.err_est, q.mode,
                    q.certified) == key, (m.shape, item_log2)
