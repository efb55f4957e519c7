"""Autotuner of the launch shapes: pair sums per size bucket and the BF16
GEMM.

Pair sums: for each (kernel, precision) and each tuned problem size
(n_targets, n_sources) of a grid of powers of two, it times f3d_pairsum (there
and at three quarters of it) over the launch shapes -- targets per lane K in
{1, 2, 4} and the wavefront count the source split aims for -- and keeps the
fastest.  FP32C sums depend on their shape at the 1e-8 level (K groups the
targets of the near/far test, the split the compensated partial sums), so their
shapes are tuned on powers of four only, over fewer wavefront counts, and the
sizes in between (the entries without a rate) take the nearest of those: a finer
grid would change sums of those sizes.  apply() installs the
fastest shape of the nearest tuned size (in log2 n_targets + log2 n_sources)
into every size bucket of the library (f3d_pairsum_set_launch_bucket), and
the 65536 x 65536 shape as the (kernel, precision) default.  The large
fiber -> fiber Oseen sum (262144 nodes, exclusion ranges) is tuned on its
own layout, bucket 18/18.

BF16 GEMM (f3d_gemm_set_stream): resident-weight, streaming or tiled kernel for
the per-node layers (N = 128, 256).  Batched LU (f3d_lu_set_launch): a table's
entry is checked and passed on, but no launch depends on it, and none is tuned.

The table lives in fiber3d_amd/tuning.json; the kernels module calls apply()
at import when it exists.  validate() checks a table's shape and ranges.
"""
import json
import os
import time

import numpy as np

from . import _lib as L

HERE = os.path.dirname(os.path.abspath(__file__))
CACHE = os.path.join(HERE, "tuning.json")
KERNELS = {"oseen": L.OSEEN, "rotlet": L.ROTLET, "stresslet": L.STRESSLET}
PRECS = {"f64": L.F64, "f32c": L.F32C}
LG_MIN, LG_MAX = 8, 22          # size buckets of the library (log2 sizes)
KS = (1, 2, 4)
WAVES = {"f64": (2048, 4096, 8192, 12288, 16384, 24576, 32768, 65536),
         "f32c": (2048, 4096, 8192, 16384, 32768)}
GRID_NT = (4096, 8192, 16384, 32768, 65536, 262144)
GRID_NS = (1024, 2048, 4096, 8192, 16384, 32768, 65536)
# the sizes of the grid whose shapes are timed
TUNED = {"f64": (GRID_NT, GRID_NS),
         "f32c": ((4096, 16384, 65536), (1024, 4096, 16384, 65536))}
LU_LAUNCH = {"f64": {"factor_waves_per_cu": 4, "solve_staged": 0},
             "f32c": {"factor_waves_per_cu": 8, "solve_staged": 0}}


def set_launch(kernel, precision, k, waves):
    rc = L.load().f3d_pairsum_set_launch(KERNELS[kernel], PRECS[precision], int(k), int(waves))
    L.check(rc, "f3d_pairsum_set_launch")


def set_launch_bucket(kernel, precision, lg_nt, lg_ns, k, waves):
    rc = L.load().f3d_pairsum_set_launch_bucket(KERNELS[kernel], PRECS[precision], int(lg_nt),
                                                int(lg_ns), int(k), int(waves))
    L.check(rc, "f3d_pairsum_set_launch_bucket")


def plan(kernel, precision, ns, nt):
    """(K, chunks, sources per chunk) f3d_pairsum would use."""
    import ctypes
    out = (ctypes.c_int32 * 3)()
    rc = L.load().f3d_pairsum_plan(KERNELS[kernel], PRECS[precision], int(ns), int(nt),
                                   ctypes.addressof(out))
    L.check(rc, "f3d_pairsum_plan")
    return tuple(out)


def lg(n):
    """ceil(log2 n) for n >= 1 (the library's bucket index before clamping)."""
    return int(max(0, int(n) - 1).bit_length())


def _nearest(points, a, b):
    return min(points, key=lambda p: (abs(p[0] - a) + abs(p[1] - b), p))


def expand_buckets(tuned):
    """{(lg_nt, lg_ns): entry} over the library's whole bucket range, each
    from the nearest tuned size."""
    pts = sorted(tuned)
    return {(a, b): tuned[_nearest(pts, a, b)]
            for a in range(LG_MIN, LG_MAX + 1) for b in range(LG_MIN, LG_MAX + 1)}


def fill_grid(rated):
    """The entries of every size of the grid: the timed ones ({"16/12": entry}),
    and in between the shape of the nearest of them."""
    pts = {tuple(int(s) for s in size.split("/")): v for size, v in rated.items()}
    near = {}
    for nt in GRID_NT:
        for ns in GRID_NS:
            v = pts[_nearest(sorted(pts), lg(nt), lg(ns))]
            near[f"{lg(nt)}/{lg(ns)}"] = {"k": v["k"], "waves": v["waves"]}
    return {**near, **rated}


def validate(table):
    """Raise ValueError unless `table` is a well-formed tuning table whose
    every shape the library accepts."""
    if not isinstance(table, dict):
        raise ValueError("table must be a JSON object")
    for key, v in table.get("pairsum", {}).items():
        kernel, precision = key.split("/")
        if kernel not in KERNELS or precision not in PRECS:
            raise ValueError(f"unknown pairsum entry {key}")
        if v["k"] not in KS or not (64 <= v["waves"] <= 1 << 20):
            raise ValueError(f"bad pairsum shape {key}: {v}")
    for key, buckets in table.get("pairsum_buckets", {}).items():
        kernel, precision = key.split("/")
        if kernel not in KERNELS or precision not in PRECS:
            raise ValueError(f"unknown pairsum bucket entry {key}")
        for size, v in buckets.items():
            a, b = (int(s) for s in size.split("/"))
            if not (LG_MIN <= a <= LG_MAX and LG_MIN <= b <= LG_MAX):
                raise ValueError(f"bucket {key} {size} outside [{LG_MIN}, {LG_MAX}]")
            if v["k"] not in KS or not (64 <= v["waves"] <= 1 << 20):
                raise ValueError(f"bad bucket shape {key} {size}: {v}")
    for prec, v in table.get("lu", {}).items():
        if prec not in PRECS:
            raise ValueError(f"unknown LU precision {prec}")
        cap = 4 if prec == "f64" else 8
        if not (1 <= v["factor_waves_per_cu"] <= cap) or v["solve_staged"] not in (0, 1):
            raise ValueError(f"bad LU launch {prec}: {v}")
    for n, v in table.get("gemm", {}).items():
        if n not in ("128", "256") or v["stream"] not in (0, 1, 2):
            raise ValueError(f"bad GEMM entry {n}: {v}")
    return table


def apply(path=CACHE, table=None):
    """Install a tuning table (the saved one by default); returns it (empty
    if there is none)."""
    if table is None:
        if not os.path.exists(path):
            return {}
        with open(path) as fh:
            table = json.load(fh)
    validate(table)
    lib = L.load()
    for key, v in table.get("pairsum", {}).items():
        kernel, precision = key.split("/")
        set_launch(kernel, precision, v["k"], v["waves"])
    for key, buckets in table.get("pairsum_buckets", {}).items():
        kernel, precision = key.split("/")
        tuned = {tuple(int(s) for s in size.split("/")): v for size, v in buckets.items()}
        for (a, b), v in expand_buckets(tuned).items():
            set_launch_bucket(kernel, precision, a, b, v["k"], v["waves"])
    for prec, v in table.get("lu", {}).items():
        L.check(lib.f3d_lu_set_launch(PRECS[prec], int(v["factor_waves_per_cu"]),
                                      int(v["solve_staged"])), "f3d_lu_set_launch")
    for n, v in table.get("gemm", {}).items():
        L.check(lib.f3d_gemm_set_stream(int(n), int(v["stream"])), "f3d_gemm_set_stream")
    return table


def _time_queued(fn, reps, replays=3):
    """Seconds per call of fn on the device: `reps` calls in one recorded graph,
    the fastest of `replays` (host work does not count, nor do the launches
    of calls that follow each other)."""
    import torch
    from .kernels import recording_stream
    stream = recording_stream()
    with torch.cuda.stream(stream):
        fn()
        recording_stream()  # (its recorded work's workspace)
        stream.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=stream):
            for _ in range(reps):
                fn()
    g.replay()
    a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
    best = None
    for _ in range(replays):
        a.record()
        g.replay()
        b.record()
        b.synchronize()
        t = a.elapsed_time(b) * 1e-3 / reps
        best = t if best is None else min(best, t)
    return best


def _time(fn, min_s=0.02, max_reps=200):
    """Seconds per call: one untimed call, then enough calls for ~min_s."""
    import torch
    fn()
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    fn()
    torch.cuda.synchronize()
    one = max(time.perf_counter() - t0, 1e-6)
    reps = int(min(max_reps, max(3, min_s / one)))
    t0 = time.perf_counter()
    for _ in range(reps):
        fn()
    torch.cuda.synchronize()
    return (time.perf_counter() - t0) / reps


def tune_pairsum(kernels=("oseen", "stresslet", "rotlet"), precisions=("f32c", "f64"),
                 ks=KS, seed=0, log=None):
    """Fastest (K, waves) per (kernel, precision) and tuned size, the grid's other
    sizes filled from them; the 65536 x 65536 entry is also the (kernel,
    precision) default."""
    import torch
    from .kernels import pairsum

    rng = np.random.default_rng(seed)
    nmax = max(GRID_NT + GRID_NS)
    direct = os.environ.get("F3D_PAIRSUM_DIRECT")
    # (the shapes are the general path's, also at sizes that the direct kernel takes)
    os.environ["F3D_PAIRSUM_DIRECT"] = "0"
    try:
        return _tune_pairsum(torch, pairsum, rng, nmax, kernels, precisions, ks, log)
    finally:
        if direct is None:
            del os.environ["F3D_PAIRSUM_DIRECT"]
        else:
            os.environ["F3D_PAIRSUM_DIRECT"] = direct


def _tune_pairsum(torch, pairsum, rng, nmax, kernels, precisions, ks, log):
    X = torch.from_numpy(rng.uniform(0, 1, (nmax, 3))).cuda()
    F = torch.from_numpy(rng.normal(size=(nmax, 3))).cuda()
    NR = torch.nn.functional.normalize(torch.from_numpy(rng.normal(size=(nmax, 3))), dim=1).cuda()
    out = torch.empty((nmax, 3), dtype=torch.float64, device="cuda")
    defaults, buckets = {}, {}
    for kernel in kernels:
        for precision in precisions:
            key = f"{kernel}/{precision}"
            buckets[key] = {}
            grid_nt, grid_ns = TUNED[precision]
            for nt in grid_nt:
                for ns in grid_ns:
                    best = None
                    for k in ks:
                        for w in WAVES[precision]:
                            set_launch_bucket(kernel, precision, lg(nt), lg(ns), k, w)
                            t = pairs = 0.0
                            # the bucket's largest sizes and three quarters of them
                            for t_, s_ in ((nt, ns), (3 * nt // 4, 3 * ns // 4)):
                                kw = dict(src_nrm=NR[:s_] if kernel == "stresslet" else None,
                                          precision=precision, out=out[:t_])
                                reps = max(1, min(10, int(2e9 / (t_ * s_))))
                                t += _time_queued(
                                    lambda: pairsum(kernel, X[:s_], F[:s_], X[:t_], **kw), reps)
                                pairs += t_ * s_
                            rate = pairs / t / 1e9
                            if best is None or rate > best[0]:
                                best = (rate, k, w)
                    set_launch_bucket(kernel, precision, lg(nt), lg(ns), best[1], best[2])
                    ent = {"k": best[1], "waves": best[2], "gpairs_s": round(best[0], 1)}
                    buckets[key][f"{lg(nt)}/{lg(ns)}"] = ent
                    if log:
                        log(f"{key} nt={nt} ns={ns}: {ent}")
                    if nt == ns == 65536:
                        defaults[key] = dict(ent)
            buckets[key] = fill_grid(buckets[key])
    return defaults, buckets


def tune_pairsum_fibers(precisions=("f32c", "f64"), ks=KS, log=None):
    """The fiber -> fiber Oseen sum of the large workload (4096 fibers x 64
    nodes in a ball of radius 14, each fiber's own nodes excluded): its
    spatially compact tiles and exclusion ranges (the given order is kept)
    make the best shape differ from the unit cube's; tuned at 262144 x
    262144, bucket 18/18."""
    import torch
    from . import configs
    from .kernels import pairsum

    cfg = configs.config(4)
    fibers = configs.make_fibers(cfg.fibers, cfg.seed)
    x = np.concatenate(fibers)
    lens = np.array([len(f) for f in fibers])
    lo = np.repeat(np.cumsum(lens) - lens, lens).astype(np.int32)
    hi = (lo + np.repeat(lens, lens)).astype(np.int32)
    X = torch.from_numpy(x).cuda()
    F = torch.from_numpy(np.random.default_rng(1).normal(size=x.shape)).cuda()
    excl = (torch.from_numpy(lo).cuda(), torch.from_numpy(hi).cuda())
    out = torch.empty_like(X)
    n = x.shape[0]
    res = {}
    for precision in precisions:
        best = None
        for k in ks:
            for w in WAVES[precision]:
                set_launch_bucket("oseen", precision, lg(n), lg(n), k, w)
                t = _time(lambda: pairsum("oseen", X, F, X, excl=excl, precision=precision,
                                          out=out), min_s=0.05, max_reps=5)
                rate = n * n / t / 1e9
                if best is None or rate > best[0]:
                    best = (rate, k, w)
        set_launch_bucket("oseen", precision, lg(n), lg(n), best[1], best[2])
        ent = {"k": best[1], "waves": best[2], "gpairs_s": round(best[0], 1)}
        res[f"oseen/{precision}"] = {f"{lg(n)}/{lg(n)}": ent}
        if log:
            log(f"oseen/{precision} fibers n={n}: {ent}")
    return res


def tune_gemm(M=262144, K=256, log=None):
    import torch
    from . import learned

    res = {}
    g = torch.Generator().manual_seed(0)
    for N in (128, 256):
        A = torch.randn(M, K, generator=g).cuda()
        B = (torch.randn(K, N, generator=g) / 16).cuda()
        bias = torch.randn(N, generator=g).cuda()
        C = torch.empty(M, N, device="cuda")
        t = {}
        for mode in (2, 1, 0):
            L.check(L.load().f3d_gemm_set_stream(N, mode), "f3d_gemm_set_stream")
            t[mode] = _time(lambda: learned.gemm(A, B, C, epi=learned.EPI_BIAS_RELU, bias=bias))
        best = min(t, key=t.get)
        L.check(L.load().f3d_gemm_set_stream(N, best), "f3d_gemm_set_stream")
        res[str(N)] = {"stream": best, "ms_resident": round(t[2] * 1e3, 4),
                       "ms_stream": round(t[1] * 1e3, 4), "ms_tiled": round(t[0] * 1e3, 4),
                       "shape": [M, K, N]}
        if log:
            log(f"gemm N={N}: {res[str(N)]}")
    return res


PARTS = ("pairsum", "fibers", "gemm")


PROBLEM = (f"pair sums: unit-cube points, n_targets x n_sources over {list(GRID_NT)} x "
           f"{list(GRID_NS)} (FP64) and {list(TUNED['f32c'][0])} x {list(TUNED['f32c'][1])} "
           "(FP32C, other sizes from the nearest), and the 262144-node fiber -> fiber Oseen sum "
           "with exclusion ranges (bucket 18/18); GEMM: 262144 x 256 x N")


def tune_all(path=CACHE, log=print, parts=PARTS, base=None):
    """Tune `parts` and save the table; parts not re-tuned are kept from
    `base` (a table, e.g. the saved one)."""
    import torch
    table = dict(base or {})
    if "pairsum" in parts:
        defaults, buckets = tune_pairsum(log=log)
        table["pairsum"] = defaults
        old_fib = {k: {s: v for s, v in b.items() if s == "18/18"}
                   for k, b in table.get("pairsum_buckets", {}).items()}
        table["pairsum_buckets"] = buckets
        for k, b in old_fib.items():
            table["pairsum_buckets"].setdefault(k, {}).update(b)
    if "fibers" in parts:
        for k, b in tune_pairsum_fibers(log=log).items():
            table.setdefault("pairsum_buckets", {}).setdefault(k, {}).update(b)
    table["lu"] = {p: dict(v) for p, v in LU_LAUNCH.items()}
    if "gemm" in parts:
        table["gemm"] = tune_gemm(log=log)
    table["device"] = torch.cuda.get_device_name(0)
    table["problem"] = PROBLEM
    validate(table)
    if path:
        with open(path, "w") as fh:
            json.dump(table, fh, indent=1)
    return table


if __name__ == "__main__":
    import argparse
    ap = argparse.ArgumentParser(description="tune launch shapes; writes a tuning table")
    ap.add_argument("path", nargs="?", default=CACHE)
    ap.add_argument("--only", nargs="+", choices=PARTS, default=list(PARTS),
                    help="re-tune these parts, keeping the others from the saved table")
    a = ap.parse_args()
    base = None
    if os.path.exists(CACHE):
        with open(CACHE) as fh:
            base = json.load(fh)
    tune_all(path=a.path, parts=tuple(a.only), base=base)
