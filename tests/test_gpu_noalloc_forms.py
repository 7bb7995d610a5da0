"""perm_dense_noalloc over the walks a call may take -- one workgroup, the
class walk at its smallest and at the largest order that fits, the search of
a sparse integer matrix, double-double products -- has perm_dense's bits: its
runs report through a record in device memory, perm_dense's through a pinned
one."""
import ctypes

import numpy as np
import pytest

import permanent_amd as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,density,binary", [(2, 1.0, False), (12, 0.5, False), (13, 0.5, False),
                                              (24, 0.5, False), (30, 0.1, True), (33, 0.18, True),
                                              (35, 0.3, False)])
def test_noalloc_has_the_bits_of_dense(n, density, binary):
    a = P.synthetic_matrix(n, density, seed=900 + n, binary=binary)
    a[np.arange(n), (np.arange(n) + 1) % n] = 1.0  # a perfect matching
    if binary:
        a = a.astype(np.int32)
    a = np.ascontiguousarray(a)
    ref = P.dense(a, 4)
    for _ in range(2):
        c = P.PermResultC()
        st = P.lib().perm_dense_noalloc(P._DT[a.dtype], a.ctypes.data, n, 4, ctypes.byref(c))
        assert st == 0, P.lib().perm_last_error()
        r = P.PermResult.from_c(c)
        assert (r.value, r.sum_hi, r.sum_lo, r.abs_sum, r.mode, r.certified) == (
            ref.value, ref.sum_hi, ref.sum_lo, ref.abs_sum, ref.mode, ref.certified)
        assert r.kernel_ms > 0.0
