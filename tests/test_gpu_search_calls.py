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


@pytest.mark.parametrize("n,density", [(29, 0.1), (30, 0.12), (33, 0.12)])
def test_main_subsets_are_those_the_search_formed(n, density):
    """main_subsets: subsets the first pass evaluated, which the search and
    the skipper (the same search) agree on; other passes evaluate all."""
    a = threes(n, density) // 3
    plan = P.Plan(a)
    runs = [P.dense(a), P.sparse(a), P.chunked(a)[0], plan.run(), plan.run(mode=0)]
    part = plan.run_blocks(0, 1)
    plan.close()
    want = P.skip(a).main_subsets
    assert 0 < want < 0.1 * 2.0 ** (n - 1)
    for r in runs:
        assert r.main_subsets == want and r.subsets == 2.0 ** (n - 1), r
        assert r.clock_ghz == 0.0  # (the search measures none)
    assert part.main_subsets < part.subsets
    full = P.synthetic_matrix(n, 0.5, n)
    assert P.dense(full).main_subsets == 2.0 ** (n - 1)


@pytest.mark.parametrize("n,density", [(29, 0.12), (33, 0.12), (33, 0.18)])
def test_bound_of_a_search_counts_its_own_additions(monkeypatch, n, density):
    """err_bound with double-double products covers the additions a lane made
    (tens here), not those of a walk's lane of 2^9 subsets and more (2^10
    additions of 2^-104 each), and the exact difference to the Gray walk's
    sum stays within both bounds."""
    a = threes(n, density)
    plan = P.Plan(a)
    r = plan.run(mode=1)
    plan.close()
    assert r.clock_ghz == 0.0 and r.main_subsets < r.subsets, "not the search"
    assert (n + 48) * r.abs_sum * 2.0 ** -104 <= r.err_bound <= 512 * r.abs_sum * 2.0 ** -104, r
    with monkeypatch.context() as m:
        m.setenv("PERMAN_PAIR", "0")
        plan = P.Plan(a)
        w = plan.run(mode=1)
        plan.close()
    diff = abs((r.sum_hi - w.sum_hi) + (r.sum_lo - w.sum_lo))
    assert 2.0 * diff <= r.err_bound + w.err_bound, (r, w)


def integers(n, density, kind, seed):
    """A sparse pattern with entries 1 and, by kind, some of them negative
    (whole rows or here and there) or 2: rows of one or of several values."""
    a = P.synthetic_matrix(n, density, seed, binary=True, full_support=True).astype(np.int32)
    g = np.random.default_rng(seed)
    if kind == "signed":
        a = a * np.where(g.random((n, n)) < 0.3, -1, 1)
    if kind in ("twos", "signed twos"):
        a = a * np.where(g.random((n, n)) < 0.15, 2, 1)
    if kind == "signed twos":
        a = a * np.where(g.random((n, n)) < 0.3, -1, 1)
    if kind == "negative rows":
        a[::2] *= -1
    a[np.arange(n), (np.arange(n) + 1) % n] = 2 if kind == "signed twos" else 1
    return np.ascontiguousarray(a.astype(np.int32))


@pytest.mark.parametrize("kind,n,density", [("signed", 29, 0.1), ("signed", 30, 0.1),
                                            ("signed", 33, 0.12), ("twos", 33, 0.1),
                                            ("signed twos", 30, 0.08),
                                            ("negative rows", 30, 0.18)])
def test_rows_of_several_values_and_signs(monkeypatch, kind, n, density):
    """Searched matrices with rows of several values (one record per value),
    against the Gray walk in the columns' own order."""
    a = integers(n, density, kind, 11 * n)
    plan = P.Plan(a)
    fp, dd, auto = plan.run(mode=0), plan.run(mode=1), plan.run()
    plan.close()
    assert fp.main_subsets < fp.subsets and dd.main_subsets < dd.subsets, "not searches"
    calls = [fp, dd, auto, P.dense(a)]
    if (a >= 0).all():  # (the sparse path's columns are the entries > 0)
        calls.append(P.sparse(a))
    with monkeypatch.context() as m:
        m.setenv("PERMAN_PAIR", "0")
        want = P.dense(a)
    for r in calls:
        assert abs(r.value - want.value) <= r.stated + want.stated, (kind, n, r, want)
        assert abs(r.abs_sum - want.abs_sum) <= 1e-12 * want.abs_sum, (kind, n, r, want)


@pytest.mark.parametrize("n,density,scale", [(29, 0.08, 7), (29, 0.1, 7), (30, 0.1, 5), (30, 0.12, 7),
                                             (31, 0.1, 5), (33, 0.1, 3), (33, 0.12, 5)])
def test_estimate_of_a_search(n, density, scale):
    """The error of a searched FP64 pass against the double-double one: within
    err_est (three standard deviations).  Its model takes the terms' products
    as rounded independently, while the prefixes of a subtree share theirs."""
    for k, kind in enumerate(("ones", "signed")):
        for seed in range(3):
            a = scale * integers(n, density, kind, 1000 * k + 100 * seed + n)
            plan = P.Plan(a)
            f, d = plan.run(mode=0), plan.run(mode=1)
            plan.close()
            if f.main_subsets == f.subsets or f.err_est == 0.0:
                continue  # (a walk here, or exact)
            diff = 2.0 * abs((f.sum_hi - d.sum_hi) + (f.sum_lo - d.sum_lo))
            print(f"n={n} {kind} seed {seed}: error {diff / f.err_est:.3f} of err_est")
            assert diff <= f.err_est, (kind, seed, f, d)
