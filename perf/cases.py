"""The work a program using fiber3d_amd has it do, as a list of cases.

Each case is one call (or one time step) through the package's public entry
points on inputs made from a seed: the pair sums of a step, the shell
operator, a whole matvec, the per-step assembly, the batched fiber LU and its
solves, a small whole time step and a training step of the per-node net.
Sizes are those of the package's own workloads (32 fibers x 32 nodes with a
1024-node shell; 1000 x 32 with 8000; 4096 x 64; 2048 fibers of 16 to 64
nodes; 65536 points; batches of 8192 samples); draw() spreads over the ranges
between and below them, odd sizes included.
"""
import math

import numpy as np
import torch

from fiber3d_amd.dense import BatchedLU, BlockSet
from fiber3d_amd.kernels import pairsum, periphery_apply
from fiber3d_amd.learned import MLP
from fiber3d_amd.system import FiberSystem, Shell
from fiber3d_amd.tstep import TimeStepper

ETA, REG, EPS = 1.0, 5e-3, 1e-5
DT, E, EPSILON, PENALTY, END_FORCE, NFD = 1e-3, 0.01, 1e-3, 500.0, 1.0, 4
C0 = -math.log(math.e * EPSILON ** 2) / (8.0 * math.pi * ETA)
C1 = 2.0 / (8.0 * math.pi * ETA)
FLOPS = {"oseen": 28.0, "rotlet": 26.0, "stresslet": 30.0}
N_IN, N_OUT, WIDTH = 23, 4, 256


# ---------------------------------------------------------------------------
# the cases

def listed():
    return [
        # the plus-end forces' flow on every node of a small system, once per
        # step and per right-hand side: the smallest pair sum, all latency
        {"name": "end_flow_small", "kind": "pair", "what": "ends", "kernel": "oseen",
         "precision": "f64", "fibers": 32, "nodes": "32", "points": 0},
        # fiber -> fiber flow of the time series in FP64 (the product that
        # anchors every step's residual), same-fiber pairs excluded
        {"name": "fiber_flow_f64", "kind": "pair", "what": "fibers", "kernel": "oseen",
         "precision": "f64", "fibers": 1000, "nodes": "32", "points": 0},
        # the raw kernel sweep of the headline benchmark
        {"name": "point_sweep_f32c", "kind": "pair", "what": "cloud", "kernel": "oseen",
         "precision": "f32c", "fibers": 0, "nodes": "", "points": 65536},
        # the periphery's double layer, once per matvec
        {"name": "shell_apply_f64", "kind": "shell", "precision": "f64", "points": 8000},
        # one Krylov product of the time series: block products and pair sums
        {"name": "matvec_f32c", "kind": "matvec", "precision": "f32c", "fibers": 1000,
         "nodes": "32", "points": 8000},
        # the assembly of the large workload's fibers after every step
        {"name": "assemble_large", "kind": "assemble", "fibers": 4096, "nodes": "64"},
        # the fiber blocks' LU: mixed fiber sizes in FP64 (plain steps), the
        # large workload in FP32 (fast steps)
        {"name": "factor_f64_mixed", "kind": "factor", "precision": "f64", "fibers": 2048,
         "nodes": "16,24,32,48,64"},
        {"name": "factor_f32_large", "kind": "factor", "precision": "f32c", "fibers": 4096,
         "nodes": "64"},
        # the preconditioner's solves, once per Krylov step: FP64 factors of
        # mixed sizes, FP32 factors of the time series without refinement
        {"name": "solve_f64_mixed", "kind": "solve", "precision": "f64", "refine": 0,
         "fibers": 2048, "nodes": "16,24,32,48,64"},
        {"name": "solve_f32_series", "kind": "solve", "precision": "f32c", "refine": 0,
         "fibers": 1000, "nodes": "32"},
        # a whole implicit time step of the small workload
        {"name": "step_small", "kind": "step", "mode": "plain", "fibers": 32, "nodes": "32",
         "points": 1024},
        # one optimiser step of the learned initial guess
        {"name": "train_step", "kind": "train", "batch": 8192},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _nodes(rng):
    """One node count (odd ones too) or a mix of two to five."""
    if rng.random() < 0.5:
        return str(rng.randint(9, 64))
    return ",".join(str(n) for n in sorted(rng.sample(range(9, 65), rng.randint(2, 5))))


def draw(rng):
    kind = rng.choice(["pair", "pair", "pair", "shell", "matvec", "assemble", "factor", "factor",
                       "solve", "solve", "step", "train"])
    prec = rng.choice(["f64", "f32c"])
    if kind == "pair":
        what = rng.choice(["ends", "fibers", "cloud", "surface"])
        c = {"kind": kind, "what": what, "precision": prec}
        if what == "cloud":
            c.update(kernel=rng.choice(["oseen", "rotlet", "stresslet"]), fibers=0, nodes="",
                     points=_log(rng, 100, 65536))
        else:
            c.update(kernel="stresslet" if what == "surface" else "oseen",
                     fibers=_log(rng, 1, 1000), nodes=_nodes(rng),
                     points=_log(rng, 100, 4800) if what == "surface" else 0)
        return c
    if kind == "shell":
        return {"kind": kind, "precision": prec, "points": _log(rng, 200, 8000)}
    if kind == "matvec":
        return {"kind": kind, "precision": prec, "fibers": _log(rng, 4, 600),
                "nodes": _nodes(rng), "points": _log(rng, 200, 8000)}
    if kind == "assemble":
        return {"kind": kind, "fibers": _log(rng, 16, 3000), "nodes": _nodes(rng)}
    if kind == "factor":
        return {"kind": kind, "precision": prec, "fibers": _log(rng, 4, 3000),
                "nodes": _nodes(rng)}
    if kind == "solve":
        return {"kind": kind, "precision": prec, "refine": 0 if prec == "f64" else
                rng.choice([0, 6]), "fibers": _log(rng, 4, 3000), "nodes": _nodes(rng)}
    if kind == "step":
        return {"kind": kind, "mode": rng.choice(["plain", "fast"]), "fibers": _log(rng, 8, 64),
                "nodes": _nodes(rng), "points": _log(rng, 200, 1024)}
    return {"kind": kind, "batch": _log(rng, 300, 32768)}


# ---------------------------------------------------------------------------
# inputs

def _sizes(case):
    """Node count of every fiber: a fixed mix of the case's counts."""
    counts = [int(n) for n in case["nodes"].split(",")]
    return np.random.default_rng(1).choice(counts, case["fibers"])


def _fibers(case, seed, radius=None):
    """Gently bent fibers of unit length (1.5 at 64 nodes or more) in a ball:
    list of (N, 3) arrays and the lengths."""
    sizes = _sizes(case)
    nf = len(sizes)
    rng = np.random.default_rng([seed, 2])
    length = 1.5 if sizes.max() >= 64 else 1.0
    radius = radius or 1.2 * max(1.0, nf ** (1.0 / 3.0))
    t, h, b = (rng.normal(size=(nf, 3)) for _ in range(3))
    t /= np.linalg.norm(t, axis=1, keepdims=True)
    b -= (b * t).sum(1, keepdims=True) * t
    b /= np.linalg.norm(b, axis=1, keepdims=True)
    c = radius * rng.uniform(size=(nf, 1)) ** (1.0 / 3.0) * h / np.linalg.norm(h, axis=1,
                                                                             keepdims=True)
    bend = rng.uniform(0.05, 0.3, size=nf)  # curvature radius 1 / bend
    out = []
    for k, n in enumerate(sizes):
        s = np.linspace(-0.5, 0.5, n)[:, None] * length
        out.append(c[k] + t[k] * np.sin(bend[k] * s) / bend[k]
                   + b[k] * (1.0 - np.cos(bend[k] * s)) / bend[k])
    return out, np.full(nf, length)


def _sphere(n, radius):
    """Fibonacci sphere: nodes, inward normals, equal weights."""
    i = np.arange(n)
    z = 1.0 - (2.0 * i + 1.0) / n
    phi = i * math.pi * (3.0 - math.sqrt(5.0))
    rho = np.sqrt(1.0 - z * z)
    u = np.stack([rho * np.cos(phi), rho * np.sin(phi), z], axis=1)
    return radius * u, -u, np.full(n, 4.0 * math.pi * radius ** 2 / n)


def _randn(seed, tag, *shape):
    return torch.from_numpy(np.random.default_rng([seed, tag]).normal(size=shape)).cuda()


def _cuda(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _pair_inputs(case, seed):
    """Keyword arguments of the pair sum."""
    if case["what"] == "cloud":
        n = case["points"]
        x = _cuda(np.random.default_rng([seed, 3]).uniform(size=(n, 3)))
        kw = dict(src_pos=x, src_den=_randn(seed, 4, n, 3), trg_pos=x, exclude_self=True)
        if case["kernel"] == "stresslet":
            nrm = _randn(seed, 5, n, 3)
            kw["src_nrm"] = nrm / nrm.norm(dim=1, keepdim=True)
        return kw
    fibers, lengths = _fibers(case, seed)
    sizes = np.array([len(f) for f in fibers])
    offs = np.concatenate([[0], np.cumsum(sizes)])
    X = _cuda(np.concatenate(fibers))
    if case["what"] == "surface":
        # the density of a rigid body or a shell, its flow on the fibers
        R = 1.0 + np.abs(np.concatenate(fibers)).max() * math.sqrt(3.0)
        pos, nrm, _ = _sphere(case["points"], R)
        return dict(src_pos=_cuda(pos), src_den=_randn(seed, 4, case["points"], 3), trg_pos=X,
                    src_nrm=_cuda(nrm))
    w = np.concatenate([_trapezoid(n) * L / 2.0 for n, L in zip(sizes, lengths)])
    fid = np.repeat(np.arange(len(sizes)), sizes)
    if case["what"] == "ends":
        last = offs[1:] - 1
        return dict(src_pos=X[_cuda(last)], src_den=_randn(seed, 4, len(sizes), 3), trg_pos=X,
                    src_w=_cuda(w[last]), excl=(_cuda(fid.astype(np.int32)),
                                                _cuda((fid + 1).astype(np.int32))))
    # forces and velocities in component order, as the force operator writes them
    npts = int(offs[-1])
    return dict(src_pos=X, src_den=_randn(seed, 4, 3, npts).t(), trg_pos=X, src_w=_cuda(w),
                excl=(_cuda(offs[fid].astype(np.int32)), _cuda(offs[fid + 1].astype(np.int32))),
                out=torch.zeros((3, npts), dtype=torch.float64, device="cuda").t())


def _shell_inputs(n, seed):
    pos, nrm, w = (_cuda(a) for a in _sphere(n, 10.0))
    q = _randn(seed, 6, n, 3)
    add = _randn(seed, 7, n, 3)
    return pos, nrm, w, q, add


def _radius(case):
    """Shell radius around the fibers of a case."""
    return 1.2 * max(1.0, case["fibers"] ** (1.0 / 3.0)) + 1.5


def _system_kw(lengths):
    return dict(eta=ETA, dt=DT, E=E, epsilon=EPSILON, penalty=PENALTY, nfd=NFD,
                end_force=END_FORCE, lengths=lengths)


def _packed_blocks(case, seed):
    """(sizes, A): the fibers' square blocks, column-major, back to back."""
    fibers, lengths = _fibers(case, seed)
    sizes = np.array([len(f) for f in fibers])
    off = np.concatenate([[0], np.cumsum(16 * sizes ** 2)])
    buf = torch.empty(int(off[-1]), dtype=torch.float64, device="cuda")
    for n in sorted(set(sizes.tolist())):
        ids = np.flatnonzero(sizes == n)
        for part in np.array_split(ids, max(1, len(ids) * n * n // 2_000_000)):
            A = _assembled(_cuda(np.stack([fibers[k] for k in part])), lengths[part], want="A")["A"]
            A = A.transpose(1, 2).reshape(len(part), -1)
            at = _cuda(off[part])[:, None] + torch.arange(A.shape[1], device="cuda")[None, :]
            buf[at.reshape(-1)] = A.reshape(-1)
    return sizes, buf


def _net_tensors(seed):
    """Weights, biases and Adam moments of a net in mid-training."""
    rng = np.random.default_rng([seed, 8])
    f = lambda a: torch.from_numpy(a.astype(np.float32)).cuda()
    dims = [(N_IN, WIDTH), (WIDTH, WIDTH), (WIDTH, N_OUT)]
    W = [f(rng.normal(size=d) * math.sqrt(2.0 / d[0])) for d in dims]
    b = [f(0.05 * rng.normal(size=d[1])) for d in dims]
    m = [f(1e-3 * rng.normal(size=tuple(p.shape))) for p in W + b]
    v = [f((5e-3 * rng.uniform(0.5, 2.0, size=tuple(p.shape))) ** 2) for p in W + b]
    return W + b, m, v


def _batch(case, seed):
    X = _randn(seed, 9, case["batch"], N_IN).float().contiguous()
    Y = (0.3 * _randn(seed, 10, case["batch"], N_OUT)).float().contiguous()
    return X, Y


def prepare(case, seed):
    kind = case["kind"]
    if kind == "pair":
        return dict(kind=kind, kernel=case["kernel"],
                    kw=dict(_pair_inputs(case, seed), eta=ETA, reg=REG, eps=EPS,
                            precision=case["precision"]))
    if kind == "shell":
        pos, nrm, w, q, add = _shell_inputs(case["points"], seed)
        e = []  # the singularity-subtraction vectors, fixed by the geometry
        for c in range(3):
            den = torch.zeros_like(pos)
            den[:, c] = w
            e.append(pairsum("stresslet", pos, den, pos, src_nrm=nrm, eta=ETA, reg=REG, eps=EPS,
                             exclude_self=True))
        return dict(kind=kind, args=(pos, nrm, w, *e, q, add), precision=case["precision"])
    if kind == "matvec":
        fibers, lengths = _fibers(case, seed)
        shell = Shell(*_sphere(case["points"], _radius(case)), eta=ETA, pc="block")
        sys = FiberSystem(fibers, shell, lu_precision="f32c", lu_refine=0, **_system_kw(lengths))
        return dict(kind=kind, sys=sys, x=_unknowns(sys, seed), precision=case["precision"],
                    out=torch.empty(sys.size, dtype=torch.float64, device="cuda"))
    if kind == "assemble":
        fibers, lengths = _fibers(case, seed)
        return dict(kind=kind, sys=FiberSystem(fibers, None, lu_precision="f32c", lu_refine=0,
                                               **_system_kw(lengths)))
    if kind in ("factor", "solve"):
        sizes, A = _packed_blocks(case, seed)
        blocks = BlockSet(4 * sizes)
        lu = BatchedLU(blocks, A, precision=case["precision"], refine=case.get("refine", 0))
        x = _randn(seed, 11, blocks.nrows)
        return dict(kind=kind, lu=lu, x=x, out=torch.empty_like(x))
    if kind == "step":
        fibers, lengths = _fibers(case, seed)
        shell = Shell(*_sphere(case["points"], _radius(case)), eta=ETA)
        return dict(kind=kind, stepper=TimeStepper(fibers, shell, mode=case["mode"], graph=True,
                                                   **_system_kw(lengths)))
    net = MLP(N_IN, N_OUT, width=WIDTH, seed=0)
    for mine, given in zip((net.params, net.m, net.v), _net_tensors(seed)):
        for p, g in zip(mine, given):
            p.copy_(g)
    net.t = 100
    return dict(kind=kind, net=net, batch=_batch(case, seed))


def _unknowns(sys, seed):
    """An unknown vector of the matvec: shell density, then X, Y, Z and the
    tension of every fiber, the positions close to the assembled ones (a
    Krylov vector after the preconditioner is as smooth)."""
    x = torch.zeros(sys.size, dtype=torch.float64, device="cuda")
    x[:sys.fib0] = _randn(seed, 12, sys.fib0)
    X = sys.X.cpu().numpy()
    rng = np.random.default_rng([seed, 13])
    parts = []
    for k in range(sys.nfib):
        p = X[sys.offs[k]:sys.offs[k + 1]]
        s = np.linspace(-1.0, 1.0, len(p))
        wave = np.stack([np.cos(a * s + rng.uniform(0, 6)) for a in (1.0, 2.0, 3.0)], axis=1)
        parts += [(p + 0.01 * wave).T.ravel(), rng.normal() + np.cos(2.0 * s)]
    x[sys.fib0:] = _cuda(np.concatenate(parts))
    return x


def run(state):
    kind = state["kind"]
    if kind == "pair":
        return pairsum(state["kernel"], **state["kw"])
    if kind == "shell":
        pos, nrm, w, ex, ey, ez, q, add = state["args"]
        return periphery_apply(pos, nrm, w, ex, ey, ez, q, add=add, eta=ETA, reg=REG, eps=EPS,
                               precision=state["precision"])
    if kind == "matvec":
        return state["sys"].matvec(state["x"], out=state["out"], precision=state["precision"])
    if kind == "assemble":
        S = state["sys"]
        S.prepare(refactor=False)
        return {"A": S.A_buf, "F": S.F_buf, "Q": list(S.Q_buf), "xs": S.xs, "xss": S.xss,
                "weights": S.weights, "rhs": S.rhs}
    if kind == "factor":
        lu = state["lu"]
        lu.factor()
        out = {"lu": lu.lu64 if lu.lu64 is not None else lu.lu32, "piv": lu.piv, "perm": lu.perm,
               "info": lu.info}
        if lu.rs is not None:
            out.update(rs=lu.rs, cs=lu.cs)
        return out
    if kind == "solve":
        return state["lu"].solve(state["x"], out=state["out"])
    if kind == "step":
        ts = state["stepper"]
        ts.step()
        return {"X": ts.sys.X, "tension": ts.tension, "shell_density": ts.shell_density}
    net = state["net"]
    loss = net.train_step(*state["batch"])
    return {"loss": loss, "params": list(net.params)}


# ---------------------------------------------------------------------------
# what a pass cannot do without

def _block_numbers(sizes):
    n = sizes.astype(np.float64)
    return dict(npts=n.sum(), A=(16 * n * n).sum(), F=(12 * n * n).sum(),
                Q=(3 * (4 * n - 14) * n).sum(), lu=(2.0 / 3.0 * (4 * n) ** 3).sum())


def work(case):
    kind = case["kind"]
    if kind == "train":
        m, weights = case["batch"], N_IN * WIDTH + WIDTH * WIDTH + WIDTH * N_OUT
        return {"bytes": 4.0 * (m * (N_IN + N_OUT) + 6 * weights), "flops": 6.0 * m * weights}
    if kind == "shell":
        n = float(case["points"])
        return {"bytes": 8 * n * (3 * 8 + 1), "flops": FLOPS["stresslet"] * n * n}
    if kind == "pair" and case["what"] == "cloud":
        n = float(case["points"])
        return {"bytes": 8 * n * (12 if case["kernel"] == "stresslet" else 9),
                "flops": FLOPS[case["kernel"]] * n * n}
    b = _block_numbers(_sizes(case))
    npts = b["npts"]
    if kind == "pair":
        ns = {"ends": case["fibers"], "fibers": npts, "surface": case["points"]}[case["what"]]
        return {"bytes": 8.0 * (ns * 9 + npts * 6), "flops": FLOPS[case["kernel"]] * ns * npts}
    if kind == "assemble":
        return {"bytes": 8.0 * (b["A"] + b["F"] + b["Q"] + 17 * npts),
                "flops": FLOPS["oseen"] * case["fibers"] * npts}
    if kind == "factor":
        return {"bytes": b["A"] * (16 if case["precision"] == "f64" else 12), "flops": b["lu"]}
    if kind == "solve":
        per = 8 if case["precision"] == "f64" else 4
        sweeps = 1 if case["refine"] else 0
        return {"bytes": b["A"] * (per * (1 + sweeps) + 8 * sweeps) + 64 * npts,
                "flops": 2 * b["A"] * (1 + 2 * sweeps)}
    ns = float(case["points"])
    pairs = FLOPS["oseen"] * npts * (npts + ns) + FLOPS["stresslet"] * ns * (npts + ns)
    blocks = b["A"] + b["F"] + b["Q"]
    if kind == "matvec":
        return {"bytes": 8.0 * (blocks + 28 * ns + 14 * npts),
                "flops": pairs + 2.0 * blocks}
    # a step: assembly, factorisation, about five products and solves
    return {"bytes": 8.0 * (blocks * 6 + b["A"] * 6 + 45 * ns * ns),
            "flops": 5 * (pairs + 2.0 * blocks) + b["lu"]}


# ---------------------------------------------------------------------------
# the same results in plain torch and numpy, 64 bits

def _trapezoid(n):
    w = np.full(n, 2.0 / (n - 1))
    w[0] = w[-1] = 1.0 / (n - 1)
    return w


def _fd(n, k, npts):
    """k-th derivative on n uniform nodes of [-1, 1], npts-point stencils:
    coefficients of the stencils' Lagrange polynomials, in integers."""
    half = (npts - 1) // 2
    D = np.zeros((n, n))
    for i in range(n):
        lo = 0 if i < half else n - npts if i > n - half - 2 else i - half
        offs = [lo - i + j for j in range(npts)]
        for j, o in enumerate(offs):
            poly, den = [1], 1
            for p in offs[:j] + offs[j + 1:]:
                poly = [a - p * b for a, b in zip([0] + poly, poly + [0])]
                den *= o - p
            D[i, lo + j] = math.factorial(k) * poly[k] / den
    return D * (0.5 * (n - 1)) ** k


def _resample(n, m):
    """Barycentric resampling from n uniform nodes to m uniform midpoints."""
    x, y = np.linspace(-1.0, 1.0, n), -1.0 + (2.0 * np.arange(m) + 1.0) / m
    w = (-1.0) ** np.arange(n)
    w[[0, -1]] *= 0.5
    d = y[:, None] - x[None, :]
    at = d == 0.0
    t = w / np.where(at, 1.0, d)
    P = t / t.sum(1, keepdims=True)
    hit = at.any(1)
    P[hit] = at[hit]
    return P


_matrices = {}


def _fiber_matrices(n):
    if n not in _matrices:
        _matrices[n] = ([_fd(n, k, NFD + k) for k in (1, 2, 3, 4)], _resample(n, n - 4),
                        _resample(n, n - 2))
    return _matrices[n]


def _assembled(X, lengths, want="AFQ"):
    """Square blocks A (B, 4N, 4N), force rows F (B, 3, N, 4N), tension
    projections Q (B, 3, 4N - 14, N) and derivatives of B fibers of N nodes."""
    B, N, _ = X.shape
    D0, PX, PT = _fiber_matrices(N)
    PX, PT = _cuda(PX), _cuda(PT)
    sc = _cuda(2.0 / np.asarray(lengths))[:, None, None]
    D1, D2, D3, D4 = (_cuda(D)[None] * sc ** (k + 1) for k, D in enumerate(D0))
    xs, xss, xsss = D1 @ X, D2 @ X, D3 @ X
    got = {"xs": xs, "xss": xss, "D1": D1, "PX": PX, "PT": PT}
    eye = torch.eye(N, dtype=torch.float64, device="cuda")
    rows = lambda v, M: v[:, :, None] * M  # diag(v) M
    if "F" in want:
        F = torch.zeros((B, 3, N, 4 * N), dtype=torch.float64, device="cuda")
        for a in range(3):
            F[:, a, :, a * N:(a + 1) * N] = -E * D4
            F[:, a, :, 3 * N:] = rows(xss[..., a], eye) + rows(xs[..., a], D1)
        got["F"] = F
    if "Q" in want:
        Q = torch.zeros((B, 3, 4 * N - 14, N), dtype=torch.float64, device="cuda")
        for a in range(3):
            Q[:, a, a * (N - 4):(a + 1) * (N - 4)] = PX
            Q[:, a, 3 * (N - 4):] = PT @ rows(xs[..., a], D1)
        got["Q"] = Q
    if "A" in want:
        A = torch.zeros((B, 4 * N, 4 * N), dtype=torch.float64, device="cuda")
        for a in range(3):
            r = slice(a * (N - 4), (a + 1) * (N - 4))
            for b in range(3):
                g = (C0 - C1) * xs[..., a] * xs[..., b] + (C0 + C1 if a == b else 0.0)
                A[:, r, b * N:(b + 1) * N] = PX @ (E * rows(g, D4) + (eye / DT if a == b else 0.0))
            A[:, r, 3 * N:] = PX @ (-2.0 * C0 * rows(xs[..., a], D1)
                                    - (C0 + C1) * rows(xss[..., a], eye))
            A[:, 3 * (N - 4):-14, a * N:(a + 1) * N] = PT @ (
                -(C1 + 7.0 * C0) * E * rows(xss[..., a], D4)
                - 6.0 * C0 * E * rows(xsss[..., a], D3) - PENALTY * rows(xs[..., a], D1))
        A[:, 3 * (N - 4):-14, 3 * N:] = PT @ (-2.0 * C0 * D2
                                             + (C0 + C1) * rows((xss ** 2).sum(-1), eye))
        # free ends: force, its tangential part with the tension, curvature
        for end, r, sign in ((0, 4 * N - 14, 1.0), (N - 1, 4 * N - 7, -1.0)):
            for a in range(3):
                c = slice(a * N, (a + 1) * N)
                A[:, r + a, c] = sign * E * D3[:, end]
                A[:, r + a, 3 * N + end] = -sign * xs[:, end, a]
                A[:, r + 3, c] = -sign * E * D2[:, end] * xss[:, end, a, None]
                A[:, r + 4 + a, c] = D2[:, end]
            A[:, r + 3, 3 * N + end] = -sign
        got["A"] = A
    return got


def _pair_exact(kernel, src_pos, src_den, trg_pos, src_nrm=None, src_w=None, excl=None,
                exclude_self=False, out=None):
    """The pair sum over chunks of targets."""
    ns, nt = src_pos.shape[0], trg_pos.shape[0]
    den = src_den if src_w is None else src_den * src_w[:, None]
    j = torch.arange(ns, device="cuda")
    res = torch.empty((nt, 3), dtype=torch.float64, device="cuda")
    step = max(1, (1 << 25) // max(ns, 1))
    for i0 in range(0, nt, step):
        i1 = min(nt, i0 + step)
        d = [trg_pos[i0:i1, a, None] - src_pos[None, :, a] for a in range(3)]
        r2 = d[0] * d[0] + d[1] * d[1] + d[2] * d[2]
        r2 = torch.where(r2 < EPS * EPS, r2 + REG * REG, r2)
        ri = r2.rsqrt()
        if excl is not None:
            ri[(j >= excl[0][i0:i1, None]) & (j < excl[1][i0:i1, None])] = 0.0
        if exclude_self:
            ri[j == torch.arange(i0, i1, device="cuda")[:, None]] = 0.0
        dot = lambda v: d[0] * v[:, 0] + d[1] * v[:, 1] + d[2] * v[:, 2]
        if kernel == "rotlet":
            c = ri ** 3
            part = [(c * (den[:, (a + 1) % 3] * d[(a + 2) % 3]
                          - den[:, (a + 2) % 3] * d[(a + 1) % 3])).sum(1) for a in range(3)]
        elif kernel == "oseen":
            c = dot(den) * ri ** 3
            part = [ri @ den[:, a] + (c * d[a]).sum(1) for a in range(3)]
        else:
            c = -6.0 * dot(den) * dot(src_nrm) * ri ** 5
            part = [(c * d[a]).sum(1) for a in range(3)]
        res[i0:i1] = torch.stack(part, dim=1)
    return res / (8.0 * math.pi * ETA)


def _shell_exact(pos, nrm, w, q, add):
    out = _pair_exact("stresslet", pos, q, pos, src_nrm=nrm, exclude_self=True)
    for c in range(3):
        den = torch.zeros_like(pos)
        den[:, c] = w
        e = _pair_exact("stresslet", pos, den, pos, src_nrm=nrm, exclude_self=True)
        out -= (q[:, c] / w)[:, None] * e
    return out - q / w[:, None] + nrm * (nrm * q).sum() + add


class _Exact:
    """The fiber system of fiber3d_amd.system in plain torch."""

    def __init__(self, fibers, lengths, shell=None):
        self.sizes = np.array([len(f) for f in fibers])
        self.offs = np.concatenate([[0], np.cumsum(self.sizes)])
        self.X = _cuda(np.concatenate(fibers))
        self.fib0 = 0 if shell is None else 3 * len(shell[0])
        self.shell = None if shell is None else tuple(_cuda(a) for a in shell)
        fid = np.repeat(np.arange(len(fibers)), self.sizes)
        self.excl = _cuda(self.offs[fid]), _cuda(self.offs[fid + 1])
        self.fid = _cuda(fid)
        self.w = _cuda(np.concatenate([_trapezoid(n) * L / 2.0
                                       for n, L in zip(self.sizes, lengths)]))
        self.groups = []
        for n in sorted(set(self.sizes.tolist())):
            ids = np.flatnonzero(self.sizes == n)
            got = _assembled(_cuda(np.stack([fibers[k] for k in ids])), lengths[ids])
            got["ids"] = ids
            got["node"] = _cuda(self.offs[ids])[:, None] + torch.arange(int(n), device="cuda")
            got["row"] = (self.fib0 + 4 * _cuda(self.offs[ids])[:, None]
                          + torch.arange(4 * int(n), device="cuda"))
            self.groups.append(got)
        self.size = self.fib0 + 4 * int(self.offs[-1])

    def nodal(self, name):
        out = torch.empty_like(self.X)
        for g in self.groups:
            out[g["node"]] = g[name]
        return out

    def rhs(self):
        """The right-hand side with the plus ends' forces along the tangent."""
        xs, last = self.nodal("xs"), _cuda(self.offs[1:] - 1)
        f = torch.zeros_like(xs)
        f[last] = END_FORCE * xs[last]
        src = dict(src_pos=self.X[last], src_den=f[last], src_w=self.w[last])
        v = _pair_exact("oseen", trg_pos=self.X, excl=(self.fid, self.fid + 1), **src)
        out = torch.zeros(self.size, dtype=torch.float64, device="cuda")
        if self.shell is not None:
            out[:self.fib0] = -_pair_exact("oseen", trg_pos=self.shell[0], **src).reshape(-1)
        for g in self.groups:
            n = g["node"].shape[1]
            t, fk, vk = g["xs"], f[g["node"]], v[g["node"]]
            along = (t * fk).sum(-1, keepdim=True) * t
            R = self.X[g["node"]] / DT + vk + C0 * (fk + along) + C1 * (fk - along)
            T = -PENALTY + (t * (g["D1"] @ vk)).sum(-1) + 2.0 * C0 * (t * (g["D1"] @ fk)).sum(-1) \
                + (C0 - C1) * (g["xss"] * fk).sum(-1)
            sq = torch.zeros((len(g["ids"]), 4 * n), dtype=torch.float64, device="cuda")
            for a in range(3):
                sq[:, a * (n - 4):(a + 1) * (n - 4)] = R[..., a] @ g["PX"].t()
            sq[:, 3 * (n - 4):-14] = T @ g["PT"].t()
            sq[:, -7:-4] = fk[:, -1]
            sq[:, -4] = (fk[:, -1] * t[:, -1]).sum(-1)
            out[g["row"]] = sq
        return out

    def matvec(self, x):
        f = torch.empty_like(self.X)
        for g in self.groups:
            f[g["node"]] = (g["F"] @ x[g["row"]][:, None, :, None])[..., 0].transpose(1, 2)
        src = dict(src_pos=self.X, src_den=f, src_w=self.w)
        v = _pair_exact("oseen", trg_pos=self.X, excl=self.excl, **src)
        out = torch.empty_like(x)
        if self.shell is not None:
            pos, nrm, w = self.shell
            q = x[:self.fib0].view(-1, 3)
            v += _pair_exact("stresslet", pos, q, self.X, src_nrm=nrm)
            flow = _pair_exact("oseen", trg_pos=pos, **src)
            out[:self.fib0] = _shell_exact(pos, nrm, w, q, flow).reshape(-1)
        for g in self.groups:
            y = (g["A"] @ x[g["row"]][:, :, None])[..., 0]
            y[:, :-14] -= (g["Q"] @ v[g["node"]].transpose(1, 2)[..., None])[..., 0].sum(1)
            out[g["row"]] = y
        return out

    def precond(self, x):
        out = x.clone()
        if self.shell is not None:
            out[:self.fib0] *= -self.shell[2].repeat_interleave(3) / (4.0 * math.pi)
        for g in self.groups:
            if "lu" not in g:
                g["lu"] = torch.linalg.lu_factor(g["A"].cpu())
            out[g["row"]] = torch.linalg.lu_solve(*g["lu"], x[g["row"]].cpu()[..., None])[..., 0].cuda()
        return out

    def solve(self, steps=70, tol=1e-13):
        """GMRES far below the step's own tolerance."""
        b = self.rhs()
        V, H, beta = [b / b.norm()], np.zeros((steps + 1, steps)), float(b.norm())
        for j in range(steps):
            w = self.matvec(self.precond(V[j]))
            for _ in range(2):
                for i, u in enumerate(V):
                    h = torch.dot(u, w)
                    H[i, j] += float(h)
                    w -= h * u
            H[j + 1, j] = float(w.norm())
            V.append(w / w.norm())
            e = np.zeros(j + 2)
            e[0] = beta
            y = np.linalg.lstsq(H[:j + 2, :j + 1], e, rcond=None)[0]
            if np.linalg.norm(H[:j + 2, :j + 1] @ y - e) < tol * beta:
                break
        return self.precond(sum(c * u for c, u in zip(y.tolist(), V)))


def _block_list(sizes, A):
    """Host blocks, grouped by order: (ids, (B, n, n) tensor)."""
    off = np.concatenate([[0], np.cumsum(16 * sizes ** 2)])
    A = A.cpu()
    for n in sorted(set(sizes.tolist())):
        ids = np.flatnonzero(sizes == n)
        yield ids, off, torch.stack([A[off[k]:off[k + 1]].view(4 * n, 4 * n).t() for k in ids])


def exact(case, seed):
    kind = case["kind"]
    if kind == "pair":
        return _pair_exact(case["kernel"], **_pair_inputs(case, seed))
    if kind == "shell":
        return _shell_exact(*_shell_inputs(case["points"], seed))
    if kind == "matvec":
        fibers, lengths = _fibers(case, seed)
        S = _Exact(fibers, lengths, _sphere(case["points"], _radius(case)))
        S.nfib = len(fibers)
        return S.matvec(_unknowns(S, seed))
    if kind == "assemble":
        fibers, lengths = _fibers(case, seed)
        S = _Exact(fibers, lengths)
        flat = {}
        for name, per in (("A", 16), ("F", 12), ("Q0", 0), ("Q1", 0), ("Q2", 0)):
            count = (4 * S.sizes - 14) * S.sizes if name[0] == "Q" else per * S.sizes ** 2
            off = np.concatenate([[0], np.cumsum(count)])
            buf = torch.empty(int(off[-1]), dtype=torch.float64, device="cuda")
            for g in S.groups:
                M = g["Q"][:, int(name[1])] if name[0] == "Q" else g[name]
                M = M.transpose(-1, -2)
                for k, m in zip(g["ids"], M):
                    buf[off[k]:off[k + 1]] = m.reshape(-1)
            flat[name] = buf
        return {"A": flat["A"], "F": flat["F"], "Q": [flat["Q%d" % c] for c in range(3)],
                "xs": S.nodal("xs"), "xss": S.nodal("xss"), "weights": S.w, "rhs": S.rhs()}
    if kind == "factor":
        # the rounding of an FP32 factorisation's pivots and factors has no
        # 64-bit counterpart
        if case["precision"] != "f64":
            return None
        sizes, A = _packed_blocks(case, seed)
        out = torch.empty(A.numel(), dtype=torch.float64)
        for ids, off, M in _block_list(sizes, A):
            LU, _ = torch.linalg.lu_factor(M)
            for k, m in zip(ids, LU):
                out[off[k]:off[k + 1]] = m.t().reshape(-1)
        return {"lu": out, "piv": None, "perm": None, "info": None}
    if kind == "solve":
        sizes, A = _packed_blocks(case, seed)
        rows = np.concatenate([[0], np.cumsum(4 * sizes)])
        x = _randn(seed, 11, int(rows[-1])).cpu()
        y = torch.empty_like(x)
        for ids, _, M in _block_list(sizes, A):
            b = torch.stack([x[rows[k]:rows[k + 1]] for k in ids])
            for k, s in zip(ids, torch.linalg.solve(M, b)):
                y[rows[k]:rows[k + 1]] = s
        return y
    if kind == "step":
        fibers, lengths = _fibers(case, seed)
        S = _Exact(fibers, lengths, _sphere(case["points"], _radius(case)))
        x = S.solve()
        X, T = torch.empty_like(S.X), torch.empty_like(S.w)
        for g in S.groups:
            n = g["node"].shape[1]
            part = x[g["row"]].view(len(g["ids"]), 4, n)
            X[g["node"]] = part[:, :3].transpose(1, 2)
            T[g["node"]] = part[:, 3]
        return {"X": X, "tension": T, "shell_density": x[:S.fib0]}
    P, m, v = ([t.double() for t in ts] for ts in _net_tensors(seed))
    X, Y = (t.double() for t in _batch(case, seed))
    for p in P:
        p.requires_grad_()
    h = torch.relu(X @ P[0] + P[3])
    h = torch.relu(h @ P[1] + P[4])
    loss = ((h @ P[2] + P[5] - Y) ** 2).mean()
    loss.backward()
    new = []
    for p, mk, vk in zip(P, m, v):
        g = p.grad
        mh = (0.9 * mk + 0.1 * g) / (1 - 0.9 ** 101)
        vh = (0.999 * vk + 0.001 * g * g) / (1 - 0.999 ** 101)
        new.append(p.detach() - 1e-3 * mh / (vh.sqrt() + 1e-8))
    return {"loss": float(loss), "params": new}
