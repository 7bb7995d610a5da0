"""Sparse integer matrices whose passes are a search (dense, sparse, plan and
chunked calls from n = 29 on): the calls that share it, and what their results
say about it."""
import numpy as np
import pytest

import permanent_amd as P

pytestmark = pytest.mark.gpu


def threes(n, density):
    """Entries 0 and 3: values of 2^53 and more, which stay FP64 results."""
    a = 3 * P.synthetic_matrix(n, density, 3 * n, binary=True, full_support=True).astype(np.int32)
    a[np.arange(n), (np.arange(n) + 1) % n] = 3
    return a


@pytest.mark.parametrize("n,density", [(29, 0.12), (30, 0.12), (33, 0.12)])
def test_chunked_without_the_cpu_has_the_bits_of_one_launch(n, density):
    a = threes(n, density)
    one = P.dense(a)
    assert one.mode == 0 and abs(one.value) >= 2.0 ** 53, one
    for sparse in (False, True):
        c, cpu_chunks = P.chunked(a, use_cpu=False, sparse_path=sparse)
        assert cpu_chunks == 0
        assert (c.value, c.sum_hi, c.sum_lo, c.abs_sum, c.err_est, c.mode, c.certified) == (
            one.value, one.sum_hi, one.sum_lo, one.abs_sum, one.err_est, one.mode, one.certified)
    h, _ = P.chunked(a, use_cpu=True, threads=4)
    assert abs(h.value - one.value) <= h.stated + one.stated
