"""Benchmark: exact dense Ryser permanent on one MI355X.

Workload (one "step"): the permanent of one 40x40 FP64 matrix, density 0.5,
nonzeros uniform in (0,1], splitmix64 seed 2 -- 2^39 Gray-code subsets --
with the matrix resident on the device (a plan) before the timed region.

Prints ONE JSON line: subsets/s (whole job), ms per step, the roofline of
the Ryser kernel (FP64 instructions issued per lane over the kernel's time by
its own ticks, against the 39.3 T/s the chip can issue), and a
CPU baseline: the restated float-X parallel_perman64 (algo.h:662-746) timed
on the host cores over a bounded Gray slice of the same matrix.

Usage: python bench.py [--gpus 1] [--steps K] [--warmup W] [--no-cpu]
"""
import argparse
import contextlib
import json
import os
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, os.path.join(ROOT, "matrix-permanent-calculator_amd"))
# OpenMP threads of the CPU legs stay on their cores (read when libgomp loads)
os.environ.setdefault("OMP_PROC_BIND", "close")
# The process's CPU set before libgomp loads: under OMP_PROC_BIND, loading
# it pins the loading thread to one core at once, and every thread started
# after that (the server's scheduler and prep threads, the batch's host
# threads) would inherit the one-core mask.
FULL_CPU_SET = os.sched_getaffinity(0)

# HBM bytes per launch of the n=40 kernel on this workload: rocprofv3 FETCH_SIZE
# + WRITE_SIZE (profiles/ryser_class.md): 1698 KiB read + 65536 KiB written
# (2^20 workgroup records of 48 B, each one 64-B line write).
TRAFFIC_BYTES_N40 = (1697.9 + 65536.0) * 1024
FP64_PEAK_TFLOPS = 78.6
# FP64 lane-instructions the chip issues per second (an FMA is one: half the
# flop rate), in T/s
FP64_ISSUE_PEAK = FP64_PEAK_TFLOPS / 2
# FP64 instructions per subset the class walk needs for this workload's matrix
# (its plan: row additions and products per column class, the classes' joins
# and two FMAs per subset; a CPU test holds it to the plan); all VALU
# instructions by counter: 21.1 (profiles/ryser_class.md)
FP64_INSTR_N40 = 19.34
N = 40
DENSITY = 0.5
SEED = 2


@contextlib.contextmanager
def affinity_kept():
    """OpenMP under OMP_PROC_BIND pins the calling thread to one core (at
    load, and at its first parallel region), and threads started later (the
    server's scheduler and prep threads) inherit that mask; the CPU legs run
    inside this so the GPU legs that follow them get the process's full CPU
    set back."""
    try:
        yield
    finally:
        os.sched_setaffinity(0, FULL_CPU_SET)


def load_library(P):
    """Load the library (and libgomp with it) and give this thread its full
    CPU set back."""
    P.lib()
    os.sched_setaffinity(0, FULL_CPU_SET)


def cpu_share() -> int:
    """Host threads the CPU legs use: OMP_NUM_THREADS when the environment
    sets it (the CPU share given to one GPU on a shared host), else every
    core this process may run on."""
    env = os.environ.get("OMP_NUM_THREADS", "")
    if env.isdigit() and int(env) > 0:
        return int(env)
    return len(FULL_CPU_SET)


def cpu_model() -> str:
    try:
        with open("/proc/cpuinfo") as fh:
            for line in fh:
                if line.startswith("model name"):
                    return line.split(":", 1)[1].strip()
    except OSError:
        pass
    return "unknown CPU"


def cpu_baseline(mat, log2_sample: int, threads: int):
    """Time the float-X CPU baseline over the Gray slice [1, 1 + 2^log2_sample)."""
    sys.path.insert(0, os.path.join(ROOT, "oracle"))
    import oracle as O  # the CPU restatement; a checker/baseline only

    start, end = 1, 1 + (1 << log2_sample)
    t0 = time.perf_counter()
    O.parallel_perman64_slice(mat, threads, start, end, parallel=True)
    dt = time.perf_counter() - t0
    return {
        "value": (end - start) / dt,
        "unit": "subsets/s",
        "cores": threads,
        "kind": "port",
        "cpu": cpu_model(),
        "nproc": os.cpu_count(),
        "affinity_cpus": len(FULL_CPU_SET),
        "omp_num_threads": os.environ.get("OMP_NUM_THREADS"),
        "sample": (f"parallel_perman64 float-X restatement (algo.h:662-746), OpenMP "
                   f"{threads} threads (OMP_PROC_BIND={os.environ.get('OMP_PROC_BIND')}), "
                   f"Gray slice of 2^{log2_sample} subsets of the same "
                   f"n=40 matrix ({dt:.2f} s); full n=40 run extrapolated "
                   f"x{2 ** (N - 1 - log2_sample)}: {dt * 2 ** (N - 1 - log2_sample):.0f} s"),
    }


def sparse_leg(P, reps: int):
    """Sparse path (-s, ID 4) at n=36, density 0.2, every row and column
    nonzero, U(0,1], seed 4, resident plan: subsets/s, the dense-equivalent
    2n flops/subset and the sparse-minimal n + nnz/n flops/subset."""
    m = P.synthetic_matrix(36, 0.2, seed=4, full_support=True)
    nnz = int((m > 0).sum())
    plan = P.Plan(m, sparse_path=True)
    plan.run()
    t0 = time.perf_counter()
    for _ in range(reps):
        r = plan.run()
    wall = (time.perf_counter() - t0) / reps
    plan.close()
    subsets = 2.0 ** 35
    # the same pattern, all-ones (-b): an integer matrix, exact integer result
    mb = (m > 0).astype("int32")
    planb = P.Plan(mb, sparse_path=True)
    planb.run()
    t0 = time.perf_counter()
    for _ in range(reps):
        rb = planb.run()
    wall_b = (time.perf_counter() - t0) / reps
    planb.close()
    binary = {
        "workload": "sparse path -b: the same n=36 pattern, every entry 1, 2^35 subsets",
        "subsets_per_s": subsets / wall_b,
        "ms_per_run": wall_b * 1e3,
        "kernel_ms": rb.kernel_ms,
        "modes_run": "FP64 pass then double-double products" if rb.mode == 1 else "FP64 pass",
        "value": rb.value,
        "exact_integer": rb.err_bound == 0.0 and rb.value == round(rb.value),
    }
    return {
        "workload": "sparse path, n=36, density 0.2 (every row/column nonzero), U(0,1], "
                    "seed 4, 2^35 subsets, matrix resident",
        "binary": binary,
        "certified": r.certified,
        "rel_err_est": r.err_est / abs(r.value),
        "subsets_per_s": subsets / wall,
        "ms_per_run": wall * 1e3,
        "kernel_ms": r.kernel_ms,
        "shape": [r.nu, r.nu1, r.nu2],
        "pct_fp64_peak_dense_equivalent": 100.0 * 72.0 * subsets / wall / 1e12 / FP64_PEAK_TFLOPS,
        "pct_fp64_peak_sparse_minimal": 100.0 * (36.0 + nnz / 36.0) * subsets / wall / 1e12
                                        / FP64_PEAK_TFLOPS,
        "value": r.value,
        "err_bound": r.err_bound,
    }


def binary_leg(P, reps: int):
    """The 0/1 variant of the n=40 configuration (density 0.5, seed 3),
    resident plan: subsets/s and % of FP64 peak (2n flops per subset)."""
    m = P.synthetic_matrix(N, DENSITY, seed=3, binary=True).astype("int32")
    plan = P.Plan(m)
    plan.run()
    t0 = time.perf_counter()
    for _ in range(reps):
        r = plan.run()
    wall = (time.perf_counter() - t0) / reps
    plan.close()
    subsets = 2.0 ** (N - 1)
    return {
        "workload": "dense 0/1, n=40, density 0.5, splitmix64 seed 3, 2^39 subsets, matrix resident",
        "subsets_per_s": subsets / wall,
        "ms_per_run": wall * 1e3,
        "pct_fp64_peak_algorithmic": 100.0 * 2.0 * N * subsets / wall / 1e12 / FP64_PEAK_TFLOPS,
        "shape": [r.nu, r.nu1, r.nu2],
        "value": r.value,
        "err_bound": r.err_bound,
    }


def cpu_leg(P, threads: int, reps: int = 11):
    """`perman -c` (the library's OpenMP FP64 Ryser) at n=20, density 0.5,
    U(0,1], seed 1: median of `reps` runs."""
    m = P.synthetic_matrix(20, 0.5, seed=1)
    ts = []
    for _ in range(reps):
        t0 = time.perf_counter()
        v = P.cpu_dense(m, threads)
        ts.append(time.perf_counter() - t0)
    ts.sort()
    med = ts[len(ts) // 2]
    return {"workload": "CPU path (-c), n=20 FP64, density 0.5, U(0,1], seed 1",
            "threads": threads, "median_s": med, "subsets_per_s": 2.0 ** 19 / med, "value": v}


def batched_leg(P, count: int, seed: int):
    """Batched mixed-size stream (4096 matrices, n uniform in [12, 28],
    density uniform in [0.2, 0.8], nonzeros U(0,1], seed 5): one resident
    batch replayed as a graph, against one drop-in call per matrix (the
    reference's usage: host setup, upload, launch, download per matrix).
    Both sides are timed around their C calls only: the matrices' C
    arguments are built beforehand and the results land in C arrays
    (converted to Python objects after the timed region)."""
    import ctypes

    mats = P.mixed_batch(count, 12, 28, 0.2, 0.8, seed)
    subsets = sum(2.0 ** (m.shape[0] - 1) for m in mats)
    L = P.lib()
    inputs = P.BatchInputs(mats)
    res_c = (P.PermResultC * count)()
    ms = ctypes.c_double()
    # the process is warm: the batch kernels of every order were loaded by a
    # small batch with one matrix per order (the plain loop below is warm too)
    warm = P.Batch()
    warm_in = P.BatchInputs([next(m for m in mats if m.shape[0] == n)
                             for n in sorted({m.shape[0] for m in mats})])
    warm.add_prepared(warm_in, threads=cpu_share())
    warm.run()
    warm.close()
    # end to end: one call prepares (host threads), uploads and runs a new
    # batch, the preparation of the smaller orders overlapped with the
    # kernels of the largest (perm_batch_compute_dense); three new batches,
    # the first of which also pays the process's one-time host memory growth
    e2e = []
    for rep in range(3):
        if rep:
            b.close()
        t0 = time.perf_counter()
        b = P.Batch()
        b.compute_prepared(inputs, res_c, threads=cpu_share())
        e2e.append(time.perf_counter() - t0)
    t_first = e2e[0]
    t_e2e = sorted(e2e)[1]
    t0 = time.perf_counter()
    tuned = b.autotune(reps=2)  # picks the work split on this batch
    t_tune = time.perf_counter() - t0
    P._check(L.perm_batch_run(b._h, res_c, ctypes.byref(ms)))  # rebuild with the chosen split
    reps = 3
    t0 = time.perf_counter()
    dev = []
    for _ in range(reps):
        P._check(L.perm_batch_run(b._h, res_c, ctypes.byref(ms)))
        dev.append(ms.value)
    t_batch = (time.perf_counter() - t0) / reps
    b.close()
    res = [P.PermResult.from_c(r) for r in res_c]
    # plain: one perm_dense call per matrix (ID 4), arguments prebuilt
    args = [(P._DT[m.dtype], m.ctypes.data, m.shape[0]) for m in inputs.mats]
    one = P.PermResultC()
    plain_c = (P.PermResultC * count)()
    t0 = time.perf_counter()
    for i, (dt, ptr, n) in enumerate(args):
        P._check(L.perm_dense(dt, ptr, n, 4, ctypes.byref(one)))
        plain_c[i] = one
    t_plain = time.perf_counter() - t0
    plain = [P.PermResult.from_c(r) for r in plain_c]
    worst, worst_err = _diff_vs_plain(res, plain)
    oracle_err = _vs_c4_fixture(mats, res)
    return {
        "workload": f"{count} matrices, n~U{{12..28}}, density~U[0.2,0.8], U(0,1], seed {seed}",
        "timing": "C calls only (arguments prebuilt, results into C arrays) on both sides",
        "subsets": subsets,
        "batched_perms_per_s": count / t_batch,
        "batched_subsets_per_s": subsets / t_batch,
        "batched_device_ms": sum(dev) / len(dev),
        "batched_first_run_s": t_first,
        "batched_end_to_end_runs_s": e2e,
        "end_to_end": "a new batch in a warm process, median of 3: perm_batch_compute_dense "
                      "(prepare on host threads, upload, run; the smaller orders prepared while "
                      "the largest run); the first of the 3 also reported",
        "autotuned_split": tuned,
        "autotune_s": t_tune,
        "batched_end_to_end_perms_per_s": count / t_e2e,
        "plain_perms_per_s": count / t_plain,
        "speedup_vs_plain": t_plain / t_batch,
        "speedup_end_to_end_vs_plain": t_plain / t_e2e,
        "speedup_end_to_end_first_vs_plain": t_plain / t_first,
        "max_rel_diff_vs_plain": worst,
        "max_diff_over_stated_error": worst_err,
        "certified_fraction": sum(r.certified for r in res) / len(res),
        "zero_pattern": sum(r.zero_pattern for r in res),
        "passes": {f"mode{m}": sum(r.mode == m for r in res) for m in (0, 1, 2)},
        "vs_oracle_fixture": oracle_err,
    }


def _diff_vs_plain(res, plain):
    """Largest difference between two result lists relative to the
    permanent (0 when both are exactly 0), and in units of the sum of their
    stated errors."""
    rel = err = 0.0
    for r, v in zip(res, plain):
        d = abs(r.value - v.value)
        if d == 0.0:
            continue
        rel = max(rel, d / abs(v.value) if v.value != 0.0 else float("inf"))
        err = max(err, d / max(r.stated + v.stated, 1e-300))
    return rel, err


def _vs_c4_fixture(mats, res):
    """Largest relative error of the batch results against the oracle values
    of tests/golden/c4_mix.json (the members with n <= 26; data only)."""
    path = os.path.join(ROOT, "tests", "golden", "c4_mix.json")
    if not os.path.exists(path) or len(mats) != 4096:
        return None
    members = json.load(open(path))["members"]
    worst, zeros_exact = 0.0, 0
    for rec in members:
        ex = rec["hi"] + rec["lo"]
        v = res[rec["i"]].value
        if ex == 0.0:
            zeros_exact += v == 0.0
        else:
            worst = max(worst, abs(v - ex) / abs(ex))
    return {"members": len(members), "max_rel_err": worst,
            "exact_zeros": zeros_exact,
            "zeros": sum(rec["hi"] + rec["lo"] == 0.0 for rec in members)}


def served_leg(P, count: int, load: float, seed: int, decay: float = 4.0):
    """Served stream: `count` requests, n in [16, 36] with
    P(n) ~ 2^(-(n-16)/decay), density U[0.1, 0.9], half 0/1 and half FP64, a
    third through the sparse path.  The server's work split is first
    autotuned on a sample of the same mix (another seed).  Capacity: every
    request submitted at once (closed loop).  Then an open loop of Poisson
    arrivals at `load` x capacity driven from C (perm_server_drive); p50/p99
    of arrival-to-result latency (a submitter that falls behind its
    arrival times counts against it).  Plain: one perm_dense / perm_sparse call
    per request.  Every side is timed around its C calls only (arguments
    prebuilt, results into C arrays)."""
    import ctypes

    import numpy as np

    reqs = [P.Request(m, sp) for m, sp in P.served_workload(count, seed, decay=decay)]
    work = sum(2.0 * q.a.shape[0] * 2.0 ** (q.a.shape[0] - 1) for q in reqs)
    batch = P.RequestBatch(reqs)
    # the tuning sample: a few times the server's resident capacity for the
    # small-request mix (a 1000-request trial lasts only milliseconds there)
    sample_n = min(count, 1000 if decay > 2 else 8000)
    sample = [P.Request(m, sp)
              for m, sp in P.served_workload(sample_n, seed + 100, decay=decay)]
    t0 = time.perf_counter()
    cfg, tuned_rate = P.autotune_server(sample)
    t_tune = time.perf_counter() - t0
    progress(f"  autotuned in {t_tune:.1f} s: {cfg}")
    with P.Server(**cfg) as srv:
        srv.wait_many(srv.submit_many(reqs[:32]))  # warm the host paths and the kernel
        t0 = time.perf_counter()
        ids = srv.submit_batch(batch)  # one call; preparation runs in the server's pool
        res_c, _ = srv.wait_many_raw(ids)
        t_closed = time.perf_counter() - t0
        stats = srv.stats()
    closed = [P.PermResult.from_c(r) for r in res_c]
    capacity = count / t_closed
    progress(f"  closed loop {capacity:.0f} req/s")
    rate = load * capacity
    gaps = -np.log(1.0 - P.uniforms((seed << 20) + (1 << 18), count)) / rate
    arrivals = np.cumsum(gaps)
    with P.Server(**cfg) as srv:
        open_c, lat_c, t_open = srv.drive(batch, arrivals)
    lat_ms = np.array(list(lat_c))
    open_modes = np.array([r.mode for r in open_c])
    open_n = np.array([q.a.shape[0] for q in reqs])
    slowest = int(np.argmax(lat_ms))
    tail = {}
    for label, sel in (("fp64_pass_only", open_modes == 0),
                       ("escalated", open_modes != 0)):
        if sel.any():
            tail[label] = {"requests": int(sel.sum()),
                           "p50_ms": float(np.percentile(lat_ms[sel], 50)),
                           "p99_ms": float(np.percentile(lat_ms[sel], 99)),
                           "max_ms": float(lat_ms[sel].max())}
    progress(f"  open loop done in {t_open:.1f} s")
    plain_c = (P.PermResultC * count)()
    one = P.PermResultC()
    L = P.lib()
    t0 = time.perf_counter()
    for i, q in enumerate(reqs):
        if q.sparse:
            P._check(L.perm_sparse(*q._args, 4, ctypes.byref(one)))
        else:
            P._check(L.perm_dense(*q._args, 4, ctypes.byref(one)))
        plain_c[i] = one
    t_plain = time.perf_counter() - t0
    plain = [P.PermResult.from_c(r) for r in plain_c]
    worst, worst_err = _diff_vs_plain(closed, plain)
    return {
        "workload": f"{count} requests, n in [16,36] with P(n)~2^(-(n-16)/{decay:g}), density "
                    f"U[0.1,0.9], half 0/1 half FP64, 1/3 sparse path, seed {seed}",
        "timing": "C calls only (arguments prebuilt, results into C arrays)",
        "algorithmic_flops": work,
        "autotuned_config": cfg,
        "autotune_s": t_tune,
        "autotune_sample_req_per_s": tuned_rate,
        "capacity_req_per_s": capacity,
        "capacity_tflops": work / t_closed / 1e12,
        "offered_load": load,
        "offered_req_per_s": rate,
        "achieved_req_per_s": count / t_open,
        "latency_origin": "scheduled arrival time (Poisson), to the result",
        "latency_p50_ms": float(np.percentile(lat_ms, 50)),
        "latency_p99_ms": float(np.percentile(lat_ms, 99)),
        "latency_max_ms": float(lat_ms.max()),
        "latency_worst_request": {"n": int(open_n[slowest]), "mode": int(open_modes[slowest])},
        "latency_by_passes": tail,
        "plain_req_per_s": count / t_plain,
        "capacity_vs_plain": t_plain / t_closed,
        "max_rel_diff_vs_plain": worst,
        "max_diff_over_stated_error": worst_err,
        "certified_fraction": sum(r.certified for r in closed) / len(closed),
        "passes": {f"mode{m}": sum(r.mode == m for r in closed) for m in (0, 1, 2)},
        "server_stats_closed_loop": stats,
    }


def progress(msg: str):
    """A progress line on stderr (the result is the one JSON line on stdout)."""
    print(f"[bench {time.strftime('%H:%M:%S')}] {msg}", file=sys.stderr, flush=True)


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=5)
    ap.add_argument("--warmup", type=int, default=1)
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--cpu-sample-log2", type=int, default=32)
    ap.add_argument("--cpu-threads", type=int, default=cpu_share())
    ap.add_argument("--no-mixed", action="store_true",
                    help="skip the 0/1, batched and served legs")
    ap.add_argument("--batch-count", type=int, default=4096,
                    help="matrices of the batched leg (0: no batched leg)")
    ap.add_argument("--serve-count", type=int, default=20000,
                    help="requests of each served leg (0: no served legs)")
    ap.add_argument("--serve-mixes", choices=("both", "heavy", "small"), default="both",
                    help="served legs: P(n) ~ 2^(-(n-16)/4) (heavy), ~ 2^-(n-16) (small)")
    ap.add_argument("--serve-load", type=float, default=0.7)
    args = ap.parse_args()
    if args.gpus != 1:
        print(f"bench.py measures one GPU; --gpus {args.gpus} is not supported in this "
              f"single-GPU build (the Gray range would shard as independent slices, "
              f"see DESIGN.md)", file=sys.stderr)
        sys.exit(2)

    import permanent_amd as P
    load_library(P)

    progress("dense n=40 steps")
    mat = P.synthetic_matrix(N, DENSITY, SEED)
    plan = P.Plan(mat)
    for _ in range(args.warmup):
        plan.run()
    kernel_ms, main_ms_l = [], []
    t0 = time.perf_counter()
    for _ in range(args.steps):  # each run() waits for its stream
        r = plan.run()
        kernel_ms.append(r.kernel_ms)
        main_ms_l.append(r.main_ms)
    wall = time.perf_counter() - t0
    plan.close()

    subsets = 2.0 ** (N - 1)
    ms_per_step = wall * 1e3 / args.steps
    value = subsets / (ms_per_step / 1e3)
    k_ms = sum(kernel_ms) / len(kernel_ms)
    main_ms = sum(main_ms_l) / len(main_ms_l)
    flops = 2.0 * N * r.main_subsets
    algorithmic = flops / (main_ms / 1e3) / 1e12
    achieved = FP64_INSTR_N40 * r.main_subsets / (main_ms / 1e3) / 1e12
    out = {
        "metric": "Ryser subsets/s + %FP64 peak at n=40; mixed-size perms/s & p99 vs plain",
        "value": value,
        "unit": "subsets/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": ms_per_step,
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f64",
        "data": "synthetic",
        "config": {
            "workload": "dense Ryser permanent, n=40 FP64, density 0.5, nonzeros U(0,1], "
                        "splitmix64 seed 2, 2^39 Gray subsets per step, matrix resident",
            "n": N,
            "density": DENSITY,
            "seed": SEED,
            "subsets_per_step": subsets,
        },
        "pct_fp64_peak_algorithmic": 100.0 * algorithmic / FP64_PEAK_TFLOPS,
        "pct_fp64_peak_whole_step": 100.0 * 2.0 * N * subsets / (ms_per_step / 1e3) / 1e12
                                    / FP64_PEAK_TFLOPS,
        "result": {"value": r.value, "err_est": r.err_est, "err_bound": r.err_bound,
                   "rel_err_est": r.err_est / abs(r.value), "certified": r.certified,
                   "mode": r.mode, "abs_sum": r.abs_sum, "shape": [r.nu, r.nu1, r.nu2]},
        "shader_clock_ghz": r.clock_ghz,
        "roofline": {
            "bound": "fp64_valu",
            "bound_detail": "FP64 vector (VALU) issue: the kernel issues FP64 additions, "
                            "multiplications and a few FMAs, no MFMA; the chip issues 39.3 T FP64 "
                            "lane-instructions per second (256 CUs x 64 per clk x 2.4 GHz, the "
                            "78.6 TFLOP/s FP64 vector peak when all are FMAs); HBM does not bound "
                            "it (traffic below, ~0.2 GB/s)",
            "clock_ghz": r.clock_ghz,
            "peak_at_measured_clock": FP64_ISSUE_PEAK * r.clock_ghz / 2.4 if r.clock_ghz else None,
            "frac_at_measured_clock": achieved / (FP64_ISSUE_PEAK * r.clock_ghz / 2.4)
                                      if r.clock_ghz else None,
            "achieved": achieved,
            "peak": FP64_ISSUE_PEAK,
            "unit": "T FP64 lane-instructions/s",
            "frac": achieved / FP64_ISSUE_PEAK,
            "traffic": TRAFFIC_BYTES_N40,
            "kernel": "perm::ryser_class_kernel<false>",
            "kernel_ms": main_ms,
            "all_kernels_ms": k_ms,
            "subsets_per_launch": r.main_subsets,
            "algorithmic_flops_per_launch": flops,
            "fp64_instructions_per_subset": FP64_INSTR_N40,
            "note": "FP64 VALU-bound. The plain walk needs 2n FP64 instructions per subset (n "
                    "additions, n multiplications). The class walk groups the rows by which of "
                    "five columns touch them and forms each class's product once per value it "
                    "takes over those columns' 32 subsets: 19.3 per subset on this matrix, so the "
                    "2n-flop rate (pct_fp64_peak_algorithmic) exceeds the FP64 peak; the roofline "
                    "counts the instructions that are issued",
        },
    }
    if not args.no_mixed:
        progress("0/1 n=40 leg")
        out["binary_n40"] = binary_leg(P, 2)
    progress("sparse leg")
    out["sparse"] = sparse_leg(P, 3)
    with affinity_kept():
        out["cpu_path_n20"] = cpu_leg(P, args.cpu_threads)
    if not args.no_mixed:
        if args.batch_count > 0:
            progress("batched leg")
            out["batched"] = batched_leg(P, args.batch_count, 5)
        if args.serve_count > 0 and args.serve_mixes != "small":
            progress("served leg (decay 4)")
            out["served"] = served_leg(P, args.serve_count, args.serve_load, 6)
        if args.serve_count > 0 and args.serve_mixes != "heavy":
            # the other reading of the configuration's size law, P(n) ~ 2^-(n-16):
            # mostly n = 16..18, per-request overhead dominates
            progress("served leg (decay 1)")
            out["served_small_n"] = served_leg(P, args.serve_count, args.serve_load, 7,
                                               decay=1.0)
    if not args.no_cpu:
        progress("CPU baseline")
        with affinity_kept():
            out["cpu_baseline"] = cpu_baseline(mat, args.cpu_sample_log2, args.cpu_threads)
    progress("done")
    print(json.dumps(out), flush=True)


if __name__ == "__main__":
    main()
