"""Whole passes in double-double of matrices whose FP64 pass is the class walk:
the Gray walk runs them on its own split and, where a call is not cut into
ranges of workgroups, with the walk shape that all columns allow, as it does
where the class walk is off (PERMAN_WALK_BITS at the Gray walk's own value);
ranges of workgroups keep the class walk's split."""
import numpy as np
import pytest

import permanent_amd as P

pytestmark = pytest.mark.gpu

GRAY_WALK_BITS = {27: 8, 29: 10, 31: 10, 32: 10, 33: 10}


def runs(a, modes):
    plan = P.Plan(a)
    out = [plan.run(mode=m) for m in modes]
    g = plan.geometry()
    plan.close()
    return out, g


@pytest.mark.parametrize("n,density,binary", [(27, 0.4, False), (27, 0.5, True), (29, 0.3, False),
                                              (31, 0.5, True), (32, 0.5, True), (32, 0.5, False),
                                              (33, 0.3, True), (33, 0.5, True)])
def test_split_is_the_gray_walks(monkeypatch, n, density, binary):
    a = P.synthetic_matrix(n, density, 60 + n, binary=binary, full_support=True)
    if binary:
        a = a.astype(np.int32)
    modes = (1, 2) if n <= 29 else (1,)
    got, g = runs(a, modes)
    with monkeypatch.context() as m:
        m.setenv("PERMAN_WALK_BITS", str(GRAY_WALK_BITS[n]))
        want, g0 = runs(a, modes)
    assert g0[0] == GRAY_WALK_BITS[n]
    for r, w in zip(got, want):
        assert abs(r.value - w.value) <= r.stated + w.stated, (r, w)
        # the bound of a pass is stated for its walks' length, 2^(w+1) of 2^-104
        # (2^-102 in mode 2) of the sum of |terms| among it: the same split
        # (results rounded to an integer have none)
        if r.mode == 2 or r.err_bound > 0.0 and w.err_bound > 0.0 and binary:
            start = 0.0 if binary else n * 2.0 ** -106
            per_term = [(q.err_bound - start * abs(q.value)) / q.abs_sum for q in (r, w)]
            assert per_term[0] == pytest.approx(per_term[1], rel=1e-6, abs=0.0), (r, w)
        if r.mode == 2:
            assert (r.nu, r.nu1, r.nu2) == (n, n, n)


@pytest.mark.parametrize("n", [30, 32, 33, 34])
@pytest.mark.parametrize("density", [0.3, 0.5, 0.7])
def test_shape_of_an_integer_matrix_is_the_gray_walks(monkeypatch, n, density):
    """Dense, sparse and chunked calls (without the CPU): the shape their passes
    with double-double products walk."""
    a = P.synthetic_matrix(n, density, 60 + n, binary=True, full_support=True).astype(np.int32)
    calls = [P.dense(a), P.sparse(a), P.chunked(a)[0]]
    with monkeypatch.context() as m:
        m.setenv("PERMAN_WALK_BITS", "10")
        want = P.dense(a)
    for r in calls:
        assert (r.nu, r.nu1, r.nu2) == (want.nu, want.nu1, want.nu2), (r, want)
        assert abs(r.value - want.value) <= r.stated + want.stated, (r, want)


@pytest.mark.parametrize("n,density,binary", [(24, 0.5, False), (29, 0.3, False), (32, 0.5, True),
                                              (33, 0.3, False), (37, 0.5, False)])
def test_block_ranges_cover_the_same_subsets(n, density, binary):
    """A workgroup's sum in FP64 (the class walk), with double-double products
    and with double-double X (both the Gray walk): the same subsets."""
    a = P.synthetic_matrix(n, density, 80 + n, binary=binary, full_support=True)
    if binary:
        a = a.astype(np.int32)
    plan = P.Plan(a)
    w, h, blocks = plan.geometry()
    plan.run(mode=2) if n <= 29 else None  # (a whole pass leaves the ranges' split alone)
    for b in (0, blocks // 3, blocks - 1):
        fp, d1, d2 = (plan.run_blocks(b, b + 1, mode=m) for m in (0, 1, 2))
        for r in (fp, d1):
            diff = abs((r.sum_hi - d2.sum_hi) + (r.sum_lo - d2.sum_lo))
            # n + 9 roundings of a term (product and row sums), at most 256 of
            # a run's sum and, in the Gray walk, the drift of 2^w steps
            assert diff <= (n + 9 + 256 + 2.0 ** w) * 2.0 ** -53 * d2.abs_sum / 2.0, (n, b, r, d2)
    plan.close()


@pytest.mark.parametrize("n", [29, 30, 33])
def test_search_takes_the_passes_its_plan_gives_it(n):
    """A sparse 0/1 matrix is searched in both passes, whatever room the Gray
    walk's own split would need for its records."""
    a = P.synthetic_matrix(n, 0.12, 3 * n, binary=True, full_support=True).astype(np.int32)
    (r0, r1), _ = runs(a, (0, 1))
    assert r0.main_subsets == r1.main_subsets < 0.1 * r0.subsets, (r0, r1)
