"""Sparse skipper (ID 7): zero-run skipping on integer matrices.

* grid-graph matrices of the reference's generator (util.h:403-520):
  exact domino-tiling counts, most of the walk skipped;
* random sparse 0/1 and small-integer matrices against the exact oracle and
  the plain sparse path;
* non-integer matrices and n < 16 fall back to the sparse path (same sum);
* the drop-in entry point for each element type."""
import numpy as np
import pytest

import oracle as O
import permanent_amd as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,cols", [(6, 6), (6, 8), (8, 8), (8, 9), (8, 10)])
def test_grid_graphs_exact(rows, cols):
    G = O.grid_graph_matrix(rows, cols).astype(np.int32)
    want = float(O.domino_tilings(rows, cols))
    r = P.skip(G)
    assert r.value == want, (rows, cols, r.value, want)
    frac = r.main_subsets / r.subsets
    print(f"grid {rows}x{cols} n={G.shape[0]}: walked {frac:.4%} of the subsets, "
          f"{r.kernel_ms:.2f} ms")
    if G.shape[0] >= 32:
        assert frac < 0.1


@pytest.mark.parametrize("n,density,seed", [(16, 0.25, 1), (18, 0.2, 2), (20, 0.3, 3),
                                            (22, 0.15, 4), (24, 0.2, 5), (26, 0.12, 6)])
def test_random_binary_vs_exact(n, density, seed):
    a = P.synthetic_matrix(n, density, seed=800 + seed, binary=True,
                           full_support=True).astype(np.int32)
    ex = O.exact_permanent(a)
    r = P.skip(a)
    s = P.sparse(a, algo_id=4)
    assert r.value == s.value
    if ex < 2 ** 53:
        assert r.value == float(ex)


@pytest.mark.parametrize("n", [17, 21])
def test_small_integers_vs_exact(n):
    rng = np.random.default_rng(n)
    a = (rng.integers(0, 4, size=(n, n)) * (rng.random((n, n)) < 0.3)).astype(np.int32)
    np.fill_diagonal(a, 1)
    ex = O.exact_permanent(a)
    r = P.skip(a)
    assert r.value == float(ex) or abs(r.value - float(ex)) <= r.stated


def test_fallbacks_follow_the_sparse_path():
    real = P.synthetic_matrix(20, 0.3, seed=12, full_support=True)
    assert P.skip(real).value == P.sparse(real, algo_id=4).value
    small = P.synthetic_matrix(12, 0.4, seed=13, binary=True).astype(np.int32)
    assert P.skip(small).value == float(O.exact_permanent(small))


@pytest.mark.parametrize("dtype", [np.int32, np.float32, np.float64])
def test_dropin_skipper(dtype):
    G = O.grid_graph_matrix(6, 6).astype(dtype)
    assert P.dropin_skipper(G) == float(O.domino_tilings(6, 6))


def _skip_cases():
    """name, matrix: the search's levels from one to many, rows of one and of
    many values, both precisions."""
    def binary(n, d):
        return P.synthetic_matrix(n, d, 70 + n, binary=True, full_support=True).astype(np.int32)

    rng = np.random.default_rng(9)

    def integer(n, d):
        a = rng.integers(0, 4, size=(n, n)) * (rng.random((n, n)) < d)  # (CCS: entries > 0)
        np.fill_diagonal(a, 1)
        return a.astype(np.int32)

    cases = [(f"binary{n}", binary(n, d)) for n, d in ((16, 0.3), (18, 0.9), (19, 0.3), (20, 0.2),
                                                       (21, 0.5), (22, 0.25), (24, 0.3))]
    cases += [(f"integer{n}", integer(n, d)) for n, d in ((16, 0.6), (20, 0.3), (23, 0.2))]
    arrow = np.eye(20, dtype=np.int32)          # a row of the last column only
    arrow[0, :] = arrow[:, 0] = 1
    cases += [("identity", np.eye(24, dtype=np.int32)), ("arrow", arrow),
              ("rotated arrow", np.ascontiguousarray(arrow[::-1, ::-1])),
              ("dense", np.ones((17, 17), dtype=np.int32))]
    return cases


@pytest.mark.parametrize("name,a", _skip_cases(), ids=lambda v: v if isinstance(v, str) else "")
def test_search_and_walk_vs_exact(monkeypatch, name, a):
    ex = O.exact_permanent(a)
    r = P.skip(a)
    monkeypatch.setenv("PERMAN_SKIP_CHECK_BITS", "3")  # the walk
    w = P.skip(a)
    for q in (r, w):
        assert abs(q.value - float(ex)) <= q.stated + 2.0 ** -53 * abs(float(ex)), (name, q, ex)
    assert r.value == w.value or r.stated > 0 or w.stated > 0
    again = [P.skip(a).value for _ in range(3)]
    assert again == [again[0]] * 3


@pytest.mark.parametrize("n,density", [(28, 0.15), (30, 0.3), (33, 0.15), (36, 0.1)])
def test_search_vs_walk_at_larger_orders(monkeypatch, n, density):
    a = P.synthetic_matrix(n, density, 5 * n, binary=True, full_support=True).astype(np.int32)
    r = P.skip(a)
    with monkeypatch.context() as m:
        m.setenv("PERMAN_SKIP_CHECK_BITS", "3")
        w = P.skip(a)
    assert r.main_subsets <= w.main_subsets
    assert r.value == w.value or abs(r.value - w.value) <= r.stated + w.stated
    assert [P.skip(a).value for _ in range(3)] == [r.value] * 3


@pytest.mark.parametrize("n,density", [(28, 0.15), (29, 0.12), (30, 0.2), (31, 0.3), (33, 0.12),
                                       (34, 0.2)])
def test_plain_calls_of_sparse_integer_matrices(monkeypatch, n, density):
    """The dense, sparse and plan calls search where that is the faster pass
    (in one mode, both or none of them); the Gray walk in the columns' own
    order (PERMAN_PAIR=0) and the sum over block ranges never do."""
    a = P.synthetic_matrix(n, density, 3 * n, binary=True, full_support=True).astype(np.int32)
    calls = [P.dense(a), P.sparse(a)]
    plan = P.Plan(a)
    calls += [plan.run(), plan.run(mode=0), plan.run(mode=1), plan.run()]
    plan.close()
    with monkeypatch.context() as m:
        m.setenv("PERMAN_PAIR", "0")
        want = P.dense(a)
    for r in calls:
        assert abs(r.value - want.value) <= r.stated + want.stated, (n, density, r, want)
        if r.zero_pattern == want.zero_pattern:  # (no walk, no sum of |terms|)
            assert abs(r.abs_sum - want.abs_sum) <= 1e-12 * want.abs_sum
    assert calls[2].value == calls[5].value == calls[0].value
