"""Host plans of the class walk and of the search (class_plan.cpp,
perman_skip_plan.cpp): the invariants their kernels rely on, over random and
structured patterns, and their tables evaluated subset by subset against the
exact permanent."""
import ctypes
import os
import re
import subprocess

import numpy as np
import pytest

import oracle as O
import permanent_amd as P
from conftest import ROOT

CSRC = os.path.join(ROOT, "matrix-permanent-calculator_amd", "csrc")


@pytest.fixture(scope="module")
def shim(tmp_path_factory):
    so = tmp_path_factory.mktemp("plans") / "libplan_shim.so"
    subprocess.run(["g++", "-O2", "-std=c++17", "-mpopcnt", "-ffp-contract=off", "-shared", "-fPIC",
                    os.path.join(ROOT, "tests", "plan_shim.cpp"),
                    os.path.join(CSRC, "class_plan.cpp"), os.path.join(CSRC, "perman_skip_plan.cpp"),
                    "-o", str(so)], check=True)
    L = ctypes.CDLL(str(so))
    L.shim_class_limit.restype = ctypes.c_double
    L.shim_class_tables.restype = L.shim_class_tables_room.restype = ctypes.c_long
    L.shim_tree_plan.restype = ctypes.c_double
    return L


def ptr(a):
    return a.ctypes.data_as(ctypes.c_void_p)


def supports(a):
    n = a.shape[0]
    return np.array([sum(1 << j for j in range(n) if a[j, k]) for k in range(n - 1)] + [0],
                    dtype=np.uint64)


def class_plan(L, a):
    n = a.shape[0]
    out = np.zeros(3 * n + 2, dtype=np.int32)
    L.shim_class_plan(n, ptr(supports(a)), ptr(out))
    return out[:n - 1], out[n - 1:2 * n - 1], out[2 * n - 1:3 * n - 1], *map(int, out[3 * n - 1:])


def patterns(n, rng):
    yield "empty", np.zeros((n, n), dtype=bool)
    yield "identity", np.eye(n, dtype=bool)
    yield "last column", np.arange(n * n).reshape(n, n) % n == n - 1
    yield "triangular", np.triu(np.ones((n, n), dtype=bool))
    yield "full", np.ones((n, n), dtype=bool)
    yield "one column short", np.ones((n, n), dtype=bool) & (np.arange(n) > 0)
    yield "circulant", np.eye(n, dtype=bool) | np.roll(np.eye(n, dtype=bool), 1, axis=1)
    yield "halves", np.kron(np.eye(2, dtype=bool), np.ones((n // 2 + 1, n // 2 + 1), bool))[:n, :n]
    for d in (0.05, 0.1, 0.2, 0.3, 0.4, 0.5, 0.7, 0.9):
        for _ in range(4):
            yield f"density {d}", rng.random((n, n)) < d


@pytest.mark.parametrize("n", [12, 13, 20, 23, 24, 31, 32, 33, 40, 48])
def test_class_plan_invariants(shim, n):
    L = shim
    K = L.shim_class_bits()
    half = (1 << (K - 1)) - 1
    for name, a in patterns(n, np.random.default_rng(n)):
        cols, rows, classes, live, thin, cost = class_plan(L, a)
        assert sorted(cols) == list(range(n - 1)) and sorted(rows) == list(range(n)), name
        root = L.shim_root(thin)
        count = [0] * (1 << K)
        for r, t in zip(rows, classes):
            own = sum(1 << k for k in range(K) if a[r, cols[k]])
            assert own & ~int(t) == 0, (name, r)  # the row's own class or a superset
            assert L.shim_allowed(thin, int(t)), name
            count[t] += 1
        assert live & 0xffffffff == sum(1 << t for t in range(1 << K) if count[t]), name
        assert count[root] > 0, name  # the walk starts there
        want = 3 * (1 << K) // 2 if thin else 2 << K
        for t in range(1 << K):
            if count[t]:
                m = bin(t).count("1")
                want += (2 * count[t] - 1) << m
                if t not in (root, half):
                    p = L.shim_parent(thin, t)
                    assert count[p] > 0, (name, t, p)  # its array starts from a row
                    want += 1 << bin(p).count("1")
        assert cost == want, name
        # the rows of a class stand together
        assert len([i for i in range(1, n) if classes[i] != classes[i - 1]]) + 1 == \
            sum(c > 0 for c in count), name


@pytest.mark.parametrize("n,walk_bits,density", [(12, 0, 0.2), (12, 0, 0.6), (13, 1, 0.3),
                                                 (13, 0, 0.45), (14, 2, 0.25), (14, 1, 0.8)])
def test_class_tables_hold_every_row_sum(shim, n, walk_bits, density):
    """The rows' records, the lane columns, the block columns and the walk
    offsets, read as the kernel reads them: the products over all subsets add
    up to the permanent."""
    L = shim
    K = L.shim_class_bits()
    a = P.synthetic_matrix(n, density, 17 * n + walk_bits, full_support=True)
    cols, rows, classes, live, thin, _ = class_plan(L, a)
    x0 = np.zeros(2 * n)
    data = np.zeros(L.shim_class_tables_room(n, walk_bits))
    at = np.zeros(3, dtype=np.int64)
    used = L.shim_class_tables(n, ptr(supports(a)), ptr(a), walk_bits, ptr(x0), ptr(data), ptr(at))
    assert used <= len(data)
    B = n - 1
    # offsets of each row by the subset of its class's columns
    offsets, pos, i = [], 0, 0
    while i < n:
        t, m = int(classes[i]), bin(int(classes[i])).count("1")
        c = sum(1 for q in classes if q == t)
        pair = m <= 2
        control = int(data[pos + 7:pos + 8].view(np.uint64)[0])
        end, first = i + c, True
        while i < end:
            two = pair and (not first or bool(control & 0x100))
            if first:
                assert control & 0xff == (c - (2 if two else 1)) // (2 if pair else 1)
            took = 2 if two else 1
            if m <= 3:
                for q in range(took):
                    o = data[pos + q * ((1 << m) - 1):pos + (q + 1) * ((1 << m) - 1)]
                    offsets.append(np.concatenate([[0.0], o]))
                pos += 8
            else:
                o = np.concatenate([data[pos:pos + 7], data[pos + 8:pos + (1 << m)]])
                offsets.append(np.concatenate([[0.0], o]))
                pos += 1 << m
            i += took
            first = False
    assert pos + 8 == at[0]
    lane0, block0 = K + walk_bits, K + walk_bits + 6
    blockcols = data[at[0]:][:(B - K) * n].reshape(B - K, n)
    lane = data[at[1]:][:8 * n].reshape(n, 8)
    walk = data[at[2]:][:n << walk_bits].reshape(1 << walk_bits, n)
    for k in range(K, B):
        assert (blockcols[k - K] == a[rows, cols[k]]).all()
    assert (lane[:, 6] == x0[rows]).all() and (lane[:, 7] == x0[n + rows]).all()
    assert (data[at[0] + (B - K) * n:][:2 * n] == np.concatenate([x0[rows], x0[n + rows]])).all()
    for b in range(6):
        assert (lane[:, b] == a[rows, cols[lane0 + b]]).all()
    s = np.arange(1 << B)
    bit = [(s >> k) & 1 for k in range(B)]
    prod = np.ones(1 << B)
    for r in range(n):
        t, sub, q = int(classes[r]), np.zeros(1 << B, dtype=np.int64), 0
        for k in range(K):
            if (t >> k) & 1:
                sub |= bit[k] << q
                q += 1
        x = lane[r, 6] + offsets[r][sub] + walk[(s >> K) & ((1 << walk_bits) - 1), r]
        for b in range(6):
            x = x + bit[lane0 + b] * lane[r, b]
        for k in range(block0, B):
            x = x + bit[k] * blockcols[k - K, r]
        direct = x0[rows[r]] + sum(bit[k] * a[rows[r], cols[k]] for k in range(B))
        assert np.abs(x - direct).max() <= n * 2.0 ** -52 * max(1.0, np.abs(direct).max())
        prod *= x
    total = float((prod * (1 - 2 * (sum(bit) % 2))).sum()) * (4 * (n & 1) - 2)
    ex = float(O.exact_permanent(a))
    assert abs(total - ex) <= 2.0 ** -53 * (2 * n + B) * 2 * np.abs(prod).sum()


def test_benchmark_matrix_plan(shim):
    """bench.py's roofline counts this plan's FP64 instructions per subset."""
    text = open(os.path.join(ROOT, "bench.py")).read()
    n, density, seed, instr = (float(re.search(rf"^{k} = ([0-9.]+)$", text, re.M).group(1))
                               for k in ("N", "DENSITY", "SEED", "FP64_INSTR_N40"))
    *_, cost = class_plan(shim, P.synthetic_matrix(int(n), density, seed=int(seed)))
    assert cost < shim.shim_class_limit(int(n))  # it runs the class walk
    assert instr == pytest.approx(cost / 32.0, abs=0.005)


def integers(n, density, kind, seed):
    g = np.random.default_rng(seed)
    a = (g.random((n, n)) < density).astype(float)
    a[np.arange(n), g.permutation(n)] = 1.0
    if kind == "signed":
        a *= g.choice((-1.0, 1.0), (n, n))
    if kind == "values":
        a *= g.integers(-2, 4, (n, n))
    return a


@pytest.mark.parametrize("kind", ["ones", "signed", "values"])
@pytest.mark.parametrize("n,density", [(7, 0.6), (8, 0.5), (12, 0.3), (16, 0.2), (16, 0.6)])
def test_search_plan(shim, n, density, kind):
    """Levels and records: they split the columns, a row is known where its
    records stand, they give its value at every subset, and the terms add up
    to the permanent; each row's share of zeros is the counted one."""
    L = shim
    a = integers(n, density, kind, 31 * n)
    B = n - 1
    x0, order, zero = np.zeros(2 * n), np.zeros(B, dtype=np.int32), np.zeros(n)
    levels = np.zeros((64, 4), dtype=np.int32)
    masks, recs = np.zeros(8192, dtype=np.uint64), np.zeros((8192, 3))
    counts, cost = np.zeros(5, dtype=np.int32), ctypes.c_double()
    share = L.shim_tree_plan(n, ptr(a), ptr(x0), ptr(order), ptr(zero), ptr(levels), ptr(masks),
                             ptr(recs), ptr(counts), ctypes.byref(cost))
    n_levels, n_records, top, waves, single = map(int, counts)
    max_levels, max_bits, max_top, step, room = (L.shim_tree_limits(i) for i in range(5))
    assert sorted(order) == list(range(B)) and n_levels <= max_levels
    assert 6 <= top <= max_top and levels[0][0] == top and waves <= 1 << (top - 6)
    at, seen = B, 0
    s = np.arange(1 << B, dtype=np.int64)
    direct = {}
    for j in range(n):
        direct[j] = x0[j] + sum(((s >> c) & 1) * a[j, order[c]] for c in range(B))
        assert zero[j] == pytest.approx(float((direct[j] == 0.0).mean()), rel=1e-12, abs=1e-15), j
    assert share == pytest.approx(float(np.prod(1.0 - zero)), rel=1e-9, abs=1e-12)
    left = list(range(n))
    prod, multiple = np.ones(1 << B), False
    for i, (bits, base, begin, end) in enumerate(levels[:n_levels].tolist()):
        assert begin == seen and end % step == 0 and base == at - bits
        if i:
            assert 1 <= bits <= max_bits and 64 + (64 >> bits) <= room
        at, seen = base, end
        x, parts = np.zeros(1 << B), 0
        for r in range(begin, end):
            value, start, last = recs[r]
            assert int(masks[r]) >> base << base == int(masks[r])  # known from here on
            pop = sum(((s & int(masks[r])) >> c) & 1 for c in range(B))
            x = x + value * pop + start
            parts += 1
            if last:
                multiple |= parts > 1
                hit = [j for j in left if (direct[j] == x).all()]
                if hit:
                    left.remove(hit[0])
                else:
                    assert (x == 1.0).all(), (i, r)  # a filler row
                prod *= x
                x, parts = np.zeros(1 << B), 0
        assert parts == 0
    assert at == 0 and seen == n_records and not left and single == (not multiple)
    sign = 1 - 2 * (sum((s >> c) & 1 for c in range(B)) % 2)
    total = float((prod * sign).sum()) * (4 * (n & 1) - 2)
    assert total == float(O.exact_permanent(a.astype(np.int32))), (n, kind)
