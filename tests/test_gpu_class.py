"""The class walk (FP64 pass of the single-matrix paths, n = 24..48): its
column classes, records and splits at the orders where they change, against
exact values and the double-double oracle, and against the double-double X
mode over the same workgroups where no oracle finishes."""
import numpy as np
import pytest

import oracle as O
import permanent_amd as P
from conftest import assert_target

pytestmark = pytest.mark.gpu


def patterns(n):
    """0/1 matrices whose rows fall into few, many, or one-sided classes:
    name -> (matrix, its permanent)."""
    eye = np.eye(n, dtype=np.int32)
    band = eye + np.roll(eye, 1, axis=1)          # circulant, two ones per row: 2
    tri = np.triu(np.ones((n, n), dtype=np.int32))
    hat = eye.copy()                               # a full first row and column
    hat[0, :] = hat[:, 0] = 1                      # 1 + (n - 1)
    pairs = np.kron(np.eye(n // 2, dtype=np.int32), np.ones((2, 2), dtype=np.int32))
    return {"identity": (eye, 1), "circulant": (band, 2), "triangular": (tri, 1),
            "arrow": (hat, n), "pairs": (pairs, 2 ** (n // 2))}


@pytest.mark.parametrize("name", ["identity", "circulant", "triangular", "arrow", "pairs"])
@pytest.mark.parametrize("n", [24, 30])
def test_structured_patterns_exact(n, name):
    a, want = patterns(n)[name]
    g = np.random.default_rng(n)
    for m in (a, a[g.permutation(n)][:, g.permutation(n)], 3 * a):
        m = np.ascontiguousarray(m, dtype=np.int32)
        scale = 3 ** n if m.max() == 3 else 1
        r = P.dense(m)
        # within the stated error; exact where that is below one half (the
        # sum of |terms| of 3 a, n = 30, is 4e26 times its permanent: there
        # no double-double product sum is)
        assert abs(r.value - float(want * scale)) <= r.stated, (n, name, r)
        if r.stated < 0.5:
            assert r.value == want * scale, (n, name, r)
        assert r.stated < 0.5 or scale > 1, (n, name, r)


@pytest.mark.parametrize("n,density,signed", [(24, 0.15, False), (24, 0.6, True), (25, 0.35, False),
                                              (25, 0.8, False), (26, 0.5, False),
                                              (26, 0.25, True)])
def test_against_exact_and_natural_order(monkeypatch, n, density, signed):
    a = P.synthetic_matrix(n, density, 90 + n, full_support=True)
    if signed:
        a = a * np.where(P.uniforms(7, n * n).reshape(n, n) < 0.5, -1.0, 1.0)
    hi, lo = O.ryser_dd(a)
    ex = hi + lo
    r = P.dense(a)
    assert_target(r, ex, ctx=(n, density, signed))
    with monkeypatch.context() as m:
        m.setenv("PERMAN_PAIR", "0")
        plain = P.dense(a)
    assert abs(r.value - plain.value) <= r.stated + plain.stated
    # the sum of |terms| does not depend on the walk: n roundings of a term, at
    # most 2^10 of a lane's sum
    assert abs(r.abs_sum - plain.abs_sum) <= (n + 1024) * 2.0 ** -52 * plain.abs_sum
    if not signed:
        s = P.sparse(a)
        assert (s.value, s.abs_sum) == (r.value, r.abs_sum)


@pytest.mark.parametrize("n,density", [(27, 0.1), (28, 0.7), (31, 0.3), (32, 0.5), (36, 0.2),
                                       (37, 0.6), (42, 0.45), (43, 0.2), (48, 0.5)])
def test_workgroups_cover_the_same_subsets_in_every_mode(n, density):
    """One workgroup of the class walk against the double-double X mode over
    the same subsets (the first, one in the middle, the last)."""
    plan = P.Plan(P.synthetic_matrix(n, density, 300 + n, full_support=True))
    try:
        w, h, blocks = plan.geometry()
        assert blocks == 1 << (n - 1 - w - 8)
        for b in (0, blocks // 3, blocks - 1):
            fp = plan.run_blocks(b, b + 1, mode=0)
            dd = plan.run_blocks(b, b + 1, mode=2)
            diff = abs((fp.sum_hi - dd.sum_hi) + (fp.sum_lo - dd.sum_lo))
            # n + 9 roundings of a term (product and row sums) and at most 256
            # of a run's sum
            assert diff <= min(fp.err_est / 2.0, (n + 9 + 256) * 2.0 ** -53 * fp.abs_sum / 2.0), \
                (n, b, fp, dd)
            # a lane's sum of |terms| is not folded: a rounding per subset
            assert abs(fp.abs_sum - dd.abs_sum) <= (n + 9 + 2.0 ** w) * 2.0 ** -52 * dd.abs_sum
    finally:
        plan.close()


@pytest.mark.parametrize("item_log2", [8, 10, 11, 12, 15, 21, 22])
def test_batch_splits(item_log2):
    """Batches at every kind of split: items too small for a group of class
    subsets per lane (8, 10: the variant kernels), one group (11), fewer
    groups than waves (12), more (15), the longest walk table (21: 2^10
    groups) and past it (22), for orders from below the class walk's smallest
    on, full matrices (which keep the variant kernels) and empty columns
    among them.  Every result within the stated errors of the single-matrix
    path, and the same bits alone and among the others."""
    mats = [P.synthetic_matrix(n, d, 500 + 10 * n + k, full_support=True)
            for n in (11, 12, 13, 15, 18, 23, 28) for k, d in enumerate((0.2, 0.5, 1.0))]
    mats.append((P.synthetic_matrix(22, 0.4, 3, binary=True)).astype(np.int32))
    mats.append(P.synthetic_matrix(20, 0.05, 9))
    b = P.Batch(item_log2=item_log2)
    b.add_many(mats)
    first, _ = b.run()
    again, _ = b.run()
    b.close()
    for m, r, r2 in zip(mats, first, again):
        one = P.dense(m)
        n = m.shape[0]
        assert abs(r.value - one.value) <= r.stated + one.stated, (n, item_log2, r, one)
        assert r.certified and r.zero_pattern == one.zero_pattern
        assert (r.value, r.sum_lo, r.abs_sum, r.err_est) == (r2.value, r2.sum_lo, r2.abs_sum,
                                                             r2.err_est)
    for i in (1, 7, 13, 19):
        b = P.Batch(item_log2=item_log2)
        b.add(mats[i])
        (alone,), _ = b.run()
        b.close()
        assert (alone.value, alone.sum_lo, alone.abs_sum) == (first[i].value, first[i].sum_lo,
                                                              first[i].abs_sum), i


@pytest.mark.parametrize("n,exponent", [(24, 20), (24, 60), (24, 100), (24, 300), (30, 20),
                                        (30, 60), (30, 100), (30, 300), (30, 450)])
def test_rows_of_far_apart_magnitudes(n, exponent):
    """Rows scaled by 2^e and 2^-e in turn: the permanent is the unscaled
    one's, whichever walk the rows' range leaves (a class's product of twelve
    rows of 2^100 is out of range).  The two runs' stated errors bound the
    difference."""
    a = P.synthetic_matrix(n, 0.6, n, full_support=True)
    base = P.dense(a)
    b = a.copy()
    b[::2] *= 2.0 ** exponent
    b[1::2] *= 2.0 ** -exponent
    r = P.dense(b)
    assert np.isfinite(r.value), (n, exponent, r)
    assert abs(r.value - base.value) <= r.stated + base.stated, (n, exponent, r, base)


@pytest.mark.parametrize("n", [12, 17, 23, 26])
def test_batch_of_both_trees(n):
    """One batch whose matrices take the thin tree (two class columns without
    a common row), the full one, or neither, against the double-double
    oracle (the single runs from 24 rows on)."""
    mats = [P.synthetic_matrix(n, d, 40 * n + i, full_support=True)
            for i, d in enumerate((0.12, 0.2, 0.3, 0.45, 0.6, 0.9, 1.0, 0.15))]
    b = P.Batch()
    for m in mats:
        b.add(m)
    out, _ = b.run()
    b.close()
    for d, (m, r) in enumerate(zip(mats, out)):
        if r.zero_pattern:  # no perfect matching: exactly 0, no walk
            assert r.value == 0.0
        elif n < 24:
            hi, lo = O.ryser_dd(m)
            assert abs(r.value - (hi + lo)) <= r.stated, (n, d, r)
        else:
            s = P.dense(m)
            assert abs(r.value - s.value) <= r.stated + s.stated, (n, d, r, s)
