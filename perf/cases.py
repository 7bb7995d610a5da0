"""Performance cases of the framework: the work its users have it do, through
its public entry points (permanent_amd).

Every case computes permanents exactly: one-call drop-ins over the orders the
reference's users compute (small orders, where the call itself counts; the
middle; orders whose walk takes all the time), resident plans, the sparse
path, the skipping walk on grid graphs, a batch of mixed orders in one call
and replayed, and a stream of requests through the server.  Element types are
the three the library takes (int32, float32, float64); densities run from
sparse patterns to full matrices.

  dense   permanent_amd.solve on a prepared dense Request (perm_dense)
  sparse  permanent_amd.solve on a prepared sparse Request (perm_sparse)
  plan    Plan(mat).run(): the matrix resident on the device
  skip    permanent_amd.skip on a grid graph (dimer coverings)
  batch   Batch().compute_prepared: prepare, upload and run in one call
  replay  Batch.run() on a resident batch
  serve   Server.submit_batch + wait_many_raw on a running server

Outputs: the value(s), the sum(s) of |terms| and whether each is certified.
"""
import ctypes
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "matrix-permanent-calculator_amd"))
# loading the library (and libgomp with it) may pin this thread to one core;
# the threads that batches and servers start should see the full set
_CPUS = os.sched_getaffinity(0)
import permanent_amd as P  # noqa: E402

P.lib()
os.sched_setaffinity(0, _CPUS)
THREADS = min(16, len(_CPUS))

KINDS = ("dense", "sparse", "plan", "skip", "batch", "replay", "serve")


def listed():
    return [
        # the smallest calls: a drop-in call whose walk is a few microseconds
        {"name": "dense_n12_i32", "kind": "dense", "n": 12, "density": 0.5, "dtype": "i32",
         "signed": False},
        # the order of the reference's small synthetic runs (n = 20, FP64)
        {"name": "dense_n20_f64", "kind": "dense", "n": 20, "density": 0.5, "dtype": "f64",
         "signed": False},
        # an odd order in single precision, fairly full
        {"name": "dense_n27_f32", "kind": "dense", "n": 27, "density": 0.7, "dtype": "f32",
         "signed": False},
        # a full matrix with entries of both signs (heavy cancellation)
        {"name": "dense_n28_signed", "kind": "dense", "n": 28, "density": 1.0, "dtype": "f64",
         "signed": True},
        # a 0/1 matrix: the exact integer
        {"name": "dense_n32_01", "kind": "dense", "n": 32, "density": 0.5, "dtype": "i32",
         "signed": False},
        # the headline: n = 40, density 0.5, resident
        {"name": "plan_n40_f64", "kind": "plan", "n": 40, "density": 0.5, "dtype": "f64",
         "signed": False},
        # the sparse path at its benchmark's order and density
        {"name": "sparse_n36_f64", "kind": "sparse", "n": 36, "density": 0.2, "dtype": "f64",
         "signed": False},
        # counting perfect matchings of a sparse 0/1 pattern
        {"name": "sparse_n33_01", "kind": "sparse", "n": 33, "density": 0.25, "dtype": "i32",
         "signed": False},
        # dimer coverings of a grid with a few bonds missing (n = 40)
        {"name": "skip_grid8x10", "kind": "skip", "rows": 8, "cols": 10, "missing": 0.04},
        # a new batch of mixed orders, in one call
        {"name": "batch_512", "kind": "batch", "count": 512, "n_lo": 12, "n_hi": 27},
        # the same kind of batch resident and run again
        {"name": "replay_512", "kind": "replay", "count": 512, "n_lo": 12, "n_hi": 27},
        # a stream of small requests through a running server
        {"name": "serve_2000", "kind": "serve", "count": 2000, "n_lo": 14, "n_hi": 26},
    ]


def draw(rng):
    kind = rng.choice(("dense", "dense", "dense", "sparse", "sparse", "plan", "skip", "batch",
                       "replay", "serve"))
    if kind == "dense":
        return {"kind": kind, "n": rng.randint(8, 34), "density": round(rng.uniform(0.3, 1.0), 3),
                "dtype": rng.choice(("i32", "f32", "f64")), "signed": rng.random() < 0.25}
    if kind == "plan":
        return {"kind": kind, "n": rng.randint(26, 39), "density": round(rng.uniform(0.3, 0.7), 3),
                "dtype": rng.choice(("i32", "f32", "f64")), "signed": False}
    if kind == "sparse":
        return {"kind": kind, "n": rng.randint(14, 37), "density": round(rng.uniform(0.12, 0.35), 3),
                "dtype": rng.choice(("i32", "f32", "f64")), "signed": False}
    if kind == "skip":
        r, c = rng.choice(((4, 9), (6, 7), (6, 9), (6, 11), (7, 8), (8, 8), (7, 10), (8, 9)))
        return {"kind": kind, "rows": r, "cols": c, "missing": round(rng.uniform(0.0, 0.1), 3)}
    lo = rng.randint(10, 18)
    if kind == "serve":
        return {"kind": kind, "count": int(round(2.0 ** rng.uniform(6, 11))), "n_lo": lo,
                "n_hi": rng.randint(lo + 4, 26)}
    return {"kind": kind, "count": int(round(2.0 ** rng.uniform(4, 9))), "n_lo": lo,
            "n_hi": rng.randint(lo + 4, 27)}


def _matrix(n, density, dtype, signed, rng):
    """Random pattern of the given density with a random permutation in it
    (so the permanent does not vanish by pattern), entries 1 (int32) or
    uniform in (0, 1] -- (-1, 1) when signed; signed integers are -1 and 1."""
    mask = rng.random((n, n)) < density
    mask[np.arange(n), rng.permutation(n)] = True
    if dtype == "i32":
        v = rng.choice((-1, 1), size=(n, n)) if signed else np.ones((n, n))
        return (mask * v).astype(np.int32)
    v = 2.0 * rng.random((n, n)) - 1.0 if signed else 1.0 - rng.random((n, n))
    return (mask * v).astype(np.float32 if dtype == "f32" else np.float64)


def _grid(rows, cols, missing, rng):
    """Biadjacency matrix of the rows x cols grid (an even number of cells)
    with a share of its bonds missing: its permanent counts the dimer
    coverings.  The bonds of one covering, by dominoes along an even side,
    always stay."""
    cells = [(i, j) for i in range(rows) for j in range(cols)]
    black = [c for c in cells if (c[0] + c[1]) % 2 == 0]
    white = {c: k for k, c in enumerate(c for c in cells if (c[0] + c[1]) % 2)}
    m = np.zeros((len(black), len(white)), dtype=np.int32)
    for r, (i, j) in enumerate(black):
        if cols % 2 == 0:
            mate = (i, j + 1 if j % 2 == 0 else j - 1)
        else:
            mate = (i + 1 if i % 2 == 0 else i - 1, j)
        for c in ((i + 1, j), (i - 1, j), (i, j + 1), (i, j - 1)):
            if c in white:
                kept = rng.random() >= missing
                m[r, white[c]] = 1 if kept or c == mate else 0
    return m


def _matrices(case, seed):
    rng = np.random.default_rng([int(seed), 20])
    kind = case["kind"]
    if kind in ("dense", "sparse", "plan"):
        return [_matrix(case["n"], case["density"], case["dtype"], case["signed"], rng)]
    if kind == "skip":
        return [_grid(case["rows"], case["cols"], case["missing"], rng)]
    mats = []
    span = case["n_hi"] - case["n_lo"]
    for i in range(case["count"]):
        if kind == "serve":  # mostly small requests, half of them 0/1
            n = case["n_lo"] + min(span, int(-np.log2(1.0 - rng.random())))
            mats.append(_matrix(n, rng.uniform(0.1, 0.9), "i32" if i % 2 else "f64", False, rng))
        else:                # orders uniform, every size in use
            n = case["n_lo"] + int(rng.integers(0, span + 1))
            mats.append(_matrix(n, rng.uniform(0.2, 0.8), "f64", False, rng))
    return mats


def prepare(case, seed):
    mats = _matrices(case, seed)
    kind = case["kind"]
    state = {"kind": kind}
    if kind in ("dense", "sparse"):
        state["req"] = P.Request(mats[0], sparse_path=kind == "sparse")
    elif kind == "plan":
        state["plan"] = P.Plan(mats[0])
    elif kind == "skip":
        state["mat"] = mats[0]
    elif kind == "serve":
        state["server"] = P.Server(prep_threads=4, arena_mb=64.0)
        state["requests"] = P.RequestBatch([P.Request(m, sparse_path=i % 3 == 2)
                                            for i, m in enumerate(mats)])
    else:
        state["inputs"] = P.BatchInputs(mats)
        state["results"] = (P.PermResultC * len(mats))()
        if kind == "replay":
            state["batch"] = P.Batch()
            state["batch"].add_prepared(state["inputs"], threads=THREADS)
            state["batch"].run()
    return state


def _many(res):
    """The results' fields as arrays (the C array is reused by the next run)."""
    a = np.ctypeslib.as_array(ctypes.cast(res, ctypes.POINTER(ctypes.c_ubyte)),
                              shape=(ctypes.sizeof(res),))
    size = ctypes.sizeof(P.PermResultC)
    a = a.reshape(len(res), size)

    def field(name, dtype):
        f = getattr(P.PermResultC, name)
        return np.ascontiguousarray(a[:, f.offset:f.offset + f.size]).view(dtype).reshape(-1)

    return {"value": field("value", np.float64), "abs_sum": field("abs_sum", np.float64),
            "certified": field("certified", np.int32)}


def _one(r):
    return {"value": np.array([r.value]), "abs_sum": np.array([r.abs_sum]),
            "certified": np.array([r.certified], dtype=np.int32)}


def run(state):
    kind = state["kind"]
    if kind in ("dense", "sparse"):
        return _one(P.solve(state["req"]))
    if kind == "plan":
        return _one(state["plan"].run())
    if kind == "skip":
        return _one(P.skip(state["mat"]))
    if kind == "batch":
        b = P.Batch()
        b.compute_prepared(state["inputs"], state["results"], threads=THREADS)
        b.close()
        return _many(state["results"])
    if kind == "replay":
        res = state["results"]
        ms = ctypes.c_double()
        P._check(P.lib().perm_batch_run(state["batch"]._h, res, ctypes.byref(ms)))
        return _many(res)
    ids = state["server"].submit_batch(state["requests"])
    res, _ = state["server"].wait_many_raw(ids)
    return _many(res)


def _subsets(case):
    """Sum over the case's matrices of (2^(n-1), n, density): expected values
    for the mixed cases."""
    kind = case["kind"]
    if kind in ("dense", "sparse", "plan"):
        return [(2.0 ** (case["n"] - 1), case["n"], case["density"], 1.0)]
    if kind == "skip":
        n = case["rows"] * case["cols"] // 2
        # about 0.05 % of the subsets have a nonzero term
        return [(2.0 ** (n - 1) * 5e-4, n, 4.0 / n, 1.0)]
    ns = range(case["n_lo"], case["n_hi"] + 1)
    if kind == "serve":
        w = [0.5 ** (n - case["n_lo"] + 1) for n in ns]
        w[-1] *= 2
    else:
        w = [1.0 / len(ns)] * len(ns)
    return [(2.0 ** (n - 1), n, 0.5, case["count"] * p) for n, p in zip(ns, w)]


def work(case):
    """Ryser's sum: per subset one product of n row sums and the update of the
    row sums that the flipped column touches; the matrix in, a result out."""
    size = {"i32": 4, "f32": 4}.get(case.get("dtype", "f64"), 8)
    flops = sum(k * s * (n + d * n) for s, n, d, k in _subsets(case))
    moved = sum(k * (n * n * size + 24) for s, n, d, k in _subsets(case))
    return {"bytes": moved, "flops": flops}


def _ryser(m):
    """The permanent in float64 by Ryser's formula over all subsets of the
    first n-1 columns, in the Nijenhuis-Wilf form, with torch."""
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    a = torch.tensor(np.asarray(m, dtype=np.float64), device=dev)
    n = a.shape[0]
    x0 = a[:, n - 1] - a.sum(dim=1) / 2
    low = min(n - 1, 20)
    s = torch.arange(1 << low, device=dev)
    bits = ((s[:, None] >> torch.arange(low, device=dev)) & 1).to(torch.float64)
    sign = 1.0 - 2.0 * (bits.sum(dim=1) % 2)
    # row sums of the low columns, one row per product factor
    y = [bits @ a[j, :low] for j in range(n)]
    total = 0.0
    parts = []
    for h in range(1 << (n - 1 - low)):
        hb = [(h >> b) & 1 for b in range(n - 1 - low)]
        x = x0.clone()
        for b, on in enumerate(hb):
            if on:
                x += a[:, low + b]
        p = sign * (y[0] + x[0])
        for j in range(1, n):
            p *= y[j] + x[j]
        parts.append(p.sum() * (-1.0 if sum(hb) % 2 else 1.0))
    total = torch.stack(parts).sum()
    return float(total) * (4 * (n & 1) - 2)


def exact(case, seed):
    n = case["rows"] * case["cols"] // 2 if case["kind"] == "skip" else case.get("n", 0)
    if n > 33 or sum(s * k for s, _, _, k in _subsets(case)) > 6e9:
        return None  # more than a few seconds
    v = np.array([_ryser(m) for m in _matrices(case, seed)])
    return {"value": v, "abs_sum": None, "certified": None}
