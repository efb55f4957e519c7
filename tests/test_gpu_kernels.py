"""GPU parity of the pair-sum and periphery kernels against the FP64 oracle.

Bars: FP64 path relative 2-norm <= 1e-10, FP32-compensated path <= 1e-6.
"""
import numpy as np
import pytest
import torch

from conftest import rel2
from fiber3d_amd import kernels as FK
from fiber3d_amd.geometry import shape_gallery_sphere
from oracle import kernels as K
from oracle import periphery as P

pytestmark = pytest.mark.gpu

TOL = {"f64": 1e-10, "f32c": 1e-6}
ORACLE = {
    "oseen": lambda s, t, d, n, **kw: K.oseen_kernel_source_target(s, t, d, **kw),
    "rotlet": lambda s, t, d, n, **kw: K.rotlet_kernel_source_target(s, t, d, **kw),
    "stresslet": lambda s, t, d, n, **kw: K.stresslet_kernel_source_target(s, t, n, d, **kw),
}


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a, dtype=np.float64)).cuda()


def _problem(seed, ns, nt, coincident=5, near=True):
    rng = np.random.default_rng(seed)
    s = rng.uniform(-1, 1, size=(ns, 3))
    t = rng.uniform(-1, 1, size=(nt, 3))
    k = min(coincident, ns, nt)
    t[:k] = s[:k]  # exact coincident pairs exercise the regularisation
    if near:
        # 0 < r < eps: regularised, d kept.  Only for FP64: with FP32
        # coordinates of size ~1 such a d = t - s carries ~1e-2 relative error
        # (a limit of the FP32 path, stated in its documentation).
        t[k:2 * k] = s[:k] + 3e-6
    d = rng.normal(size=(ns, 3))
    n = rng.normal(size=(ns, 3))
    n /= np.linalg.norm(n, axis=1, keepdims=True)
    return s, t, d, n


@pytest.mark.parametrize("kernel", ["oseen", "rotlet", "stresslet"])
@pytest.mark.parametrize("precision", ["f64", "f32c"])
@pytest.mark.parametrize("ns,nt", [(1500, 1300), (1, 7), (65, 1), (333, 2049)])
def test_pairsum_matches_oracle(kernel, precision, ns, nt):
    print(f"case pairsum {kernel} {precision} ns={ns} nt={nt}", flush=True)
    s, t, d, n = _problem(ns * 7 + nt, ns, nt, near=(precision == "f64"))
    eta = 0.8
    ref = ORACLE[kernel](s, t, d, n, eta=eta)
    got = FK.pairsum(kernel, _dev(s), _dev(d), _dev(t), src_nrm=_dev(n), eta=eta,
                     precision=precision)
    torch.cuda.synchronize()
    assert rel2(got.cpu().numpy(), ref) < TOL[precision]


@pytest.mark.parametrize("precision", ["f64", "f32c"])
def test_pairsum_soa_weights_exclusion_accumulate(precision):
    print(f"case pairsum soa/excl {precision}", flush=True)
    rng = np.random.default_rng(3)
    nfib, N = 40, 32
    s = rng.uniform(-2, 2, size=(nfib * N, 3))
    f = rng.normal(size=(nfib * N, 3))
    w = rng.uniform(0.5, 1.5, size=nfib * N)
    lo = np.repeat(np.arange(nfib) * N, N).astype(np.int32)
    hi = lo + N
    ref = K.oseen_kernel_source_target(s, s, f * w[:, None], exclude=(lo, hi))
    # SoA buffers (3, N) passed as their (N, 3) transposes; output SoA too
    S = _dev(s.T.copy()).T
    F = _dev(f.T.copy()).T
    out = torch.full((3, nfib * N), 1.5, dtype=torch.float64, device="cuda").T
    FK.pairsum("oseen", S, F, S, src_w=_dev(w), excl=(torch.from_numpy(lo).cuda(),
               torch.from_numpy(hi).cuda()), precision=precision, out=out, accumulate=True)
    torch.cuda.synchronize()
    assert rel2(out.cpu().numpy().ravel() - 1.5, ref) < TOL[precision]


def test_pairsum_empty_sources_and_targets():
    t = _dev(np.ones((5, 3)))
    out = FK.pairsum("oseen", _dev(np.zeros((0, 3))), _dev(np.zeros((0, 3))), t)
    assert torch.count_nonzero(out).item() == 0
    out2 = FK.pairsum("oseen", t, t, _dev(np.zeros((0, 3))))
    assert out2.shape == (0, 3)


def test_dropin_names_match_oracle():
    print("case dropin names", flush=True)
    s, t, d, n = _problem(5, 700, 500)
    np.testing.assert_allclose(FK.oseen_kernel_source_target_numba(s.ravel(), t.ravel(), d.ravel()),
                               K.oseen_kernel_source_target(s, t, d), rtol=1e-9, atol=1e-12)
    np.testing.assert_allclose(FK.rotlet_kernel_source_target_numba(s, t, d, eta=2.0),
                               K.rotlet_kernel_source_target(s, t, d, eta=2.0), rtol=1e-9,
                               atol=1e-12)
    np.testing.assert_allclose(FK.stresslet_kernel_source_target_numba(s, t, n, d),
                               K.stresslet_kernel_source_target(s, t, n, d), rtol=1e-9,
                               atol=1e-12)
    np.testing.assert_allclose(FK.stresslet_kernel_times_normal_times_density_numba(s, n, d),
                               K.stresslet_kernel_times_normal_times_density(s, n, d), rtol=1e-9,
                               atol=1e-12)
    np.testing.assert_allclose(FK.complementary_kernel_times_density_numba(s, n, d),
                               K.complementary_kernel_times_density(s, n, d), rtol=1e-12)


@pytest.mark.parametrize("precision", ["f64", "f32c"])
def test_periphery_apply_matches_dense_operator(precision):
    print(f"case periphery {precision}", flush=True)
    N, R = 800, 5.0
    x, nout = shape_gallery_sphere(N, R)
    nrm = -nout
    w = np.full(N, 4 * np.pi * R * R / N)
    ex, ey, ez = P.singularity_subtraction_vectors(x, nrm, w)
    rng = np.random.default_rng(8)
    q = rng.normal(size=(N, 3))
    add = rng.normal(size=(N, 3))
    M = P.shell_matrix(x, nrm, w, ex, ey, ez)
    ref = M @ q.ravel() + add.ravel()
    got = FK.periphery_apply(_dev(x), _dev(nrm), _dev(w), _dev(ex), _dev(ey), _dev(ez), _dev(q),
                             add=_dev(add), precision=precision)
    torch.cuda.synchronize()
    assert rel2(got.cpu().numpy(), ref) < TOL[precision]


def test_large_oseen_f32c_against_f64_and_oracle_rows():
    # Full raw-sweep size: 65536 points in the unit cube, self term excluded.
    print("case large oseen 65536", flush=True)
    rng = np.random.default_rng(1)
    N = 65536
    x = rng.uniform(0, 1, size=(N, 3))
    f = rng.normal(size=(N, 3))
    X, F = _dev(x), _dev(f)
    idx = torch.arange(N, dtype=torch.int32, device="cuda")
    excl = (idx, idx + 1)
    u64 = FK.pairsum("oseen", X, F, X, excl=excl, precision="f64")
    u32 = FK.pairsum("oseen", X, F, X, excl=excl, precision="f32c")
    torch.cuda.synchronize()
    assert rel2(u32.cpu().numpy(), u64.cpu().numpy()) < 1e-6
    # oracle on a sample of 96 targets against all sources
    rows = rng.choice(N, size=96, replace=False)
    ref = K.oseen_kernel_source_target(x, x[rows], f, exclude=(rows, rows + 1))
    assert rel2(u64.cpu().numpy()[rows], ref.reshape(-1, 3)) < 1e-10
    # linearity
    u2 = FK.pairsum("oseen", X, 2.0 * F - F, X, excl=excl, precision="f64")
    torch.cuda.synchronize()
    assert rel2(u2.cpu().numpy(), u64.cpu().numpy()) < 1e-13


@pytest.mark.parametrize("kernel", ["oseen", "rotlet", "stresslet"])
@pytest.mark.parametrize("precision", ["f64", "f32c"])
def test_padding_sources_are_masked_without_regularisation(kernel, precision):
    """With eps = reg = 0 nothing is regularised.  100 sources leave 28
    zero-density padding records in the last 64-source tile, placed at the
    origin (FP64) or at the bounding box's minimum corner (FP32C, quantised
    0); a target sits exactly there.  The reference's sum over the real
    sources is finite at that target, and so must ours be."""
    print(f"case padding {kernel} {precision}", flush=True)
    rng = np.random.default_rng(21)
    s = rng.uniform(0.1, 1.0, size=(100, 3))
    t = np.vstack([np.zeros((1, 3)), rng.uniform(0.1, 1.0, size=(40, 3))])
    d = rng.normal(size=(100, 3))
    n = rng.normal(size=(100, 3))
    n /= np.linalg.norm(n, axis=1, keepdims=True)
    ref = ORACLE[kernel](s, t, d, n, reg=0.0, epsilon_distance=0.0)
    assert np.isfinite(ref).all()
    got = FK.pairsum(kernel, _dev(s), _dev(d), _dev(t), src_nrm=_dev(n), reg=0.0, eps=0.0,
                     precision=precision).cpu().numpy().ravel()
    assert np.isfinite(got).all()
    assert rel2(got, ref) < TOL[precision]


@pytest.mark.parametrize("precision", ["f64", "f32c"])
def test_self_sum_drops_the_diagonal_without_regularisation(precision):
    """The stresslet self-sum (j != i) with eps = reg = 0: the i == j pair is
    dropped by the self-pair flag rather than relying on a regularised
    r = 0 term."""
    rng = np.random.default_rng(22)
    x = rng.uniform(-1, 1, size=(300, 3))
    n = rng.normal(size=(300, 3))
    n /= np.linalg.norm(n, axis=1, keepdims=True)
    q = rng.normal(size=(300, 3))
    ref = K.stresslet_kernel_times_normal_times_density(x, n, q, reg=0.0, epsilon_distance=0.0)
    assert np.isfinite(ref).all()
    X = _dev(x)
    got = FK.pairsum("stresslet", X, _dev(q), X, src_nrm=_dev(n), reg=0.0, eps=0.0,
                     precision=precision, exclude_self=True).cpu().numpy().ravel()
    assert rel2(got, ref) < TOL[precision]


@pytest.mark.parametrize("kernel", ["oseen", "rotlet", "stresslet"])
@pytest.mark.parametrize("ns,nt", [(1, 1), (32, 1024), (511, 255), (512, 257), (513, 513),
                                   (1025, 2048), (700, 2049), (4096, 260), (3, 70001)])
def test_one_launch_sums_match_the_general_path(kernel, ns, nt, monkeypatch):
    """Small FP64 calls run in one launch; an explicit launch shape keeps them
    on the general path.  Both over every form a call can take: weights,
    exclusion ranges (empty, partial, whole), the self flag, accumulation, AoS,
    SoA and reversed strides, near and coincident pairs, output over an input.

    Each pair carries a few 1e-15 in both; sums of up to 4096 random terms
    cancel by at most their root (64): 64 x 1e-14."""
    print(f"case one-launch {kernel} ns={ns} nt={nt}", flush=True)
    tol = 64 * 1e-14
    s, t, d, n = (_dev(a) for a in _problem(ns + nt, ns, nt))
    rng = np.random.default_rng(nt)
    w = _dev(rng.uniform(0.5, 2.0, size=ns))
    lo = rng.integers(0, ns, size=nt)
    hi = np.minimum(lo + rng.integers(0, 40, size=nt), ns)
    hi[0], lo[0] = ns, 0  # a target without sources
    excl = tuple(torch.from_numpy(a.astype(np.int32)).cuda() for a in (lo, hi))
    soa = lambda a: a.t().contiguous().t()
    back = lambda a: torch.flip(a, (0,))
    base = _dev(rng.normal(size=(nt, 3)))
    kw = dict(src_nrm=n, eta=0.7)

    def call(form):
        if form == "plain":
            return FK.pairsum(kernel, s, d, t, **kw)
        if form == "weights, ranges, accumulate, SoA":
            out = soa(base.clone())
            return FK.pairsum(kernel, soa(s), soa(d), soa(t), src_nrm=soa(n), eta=0.7, src_w=w,
                              excl=excl, out=out, accumulate=True)
        if form == "mixed strides":
            return FK.pairsum(kernel, s, d, soa(t), out=torch.empty_like(back(t)), **kw)
        if form == "output over the densities":
            dd = torch.zeros((max(ns, nt), 3), dtype=torch.float64, device="cuda")
            dd[:ns] = d
            FK.pairsum(kernel, s, dd[:ns], t, out=dd[:nt], **kw)
            return dd[:nt].clone()
        m = min(ns, nt)
        return FK.pairsum(kernel, s[:m], d[:m], s[:m], src_nrm=n[:m], eta=0.7, reg=0.0, eps=0.0,
                          exclude_self=True)

    for form in ("plain", "weights, ranges, accumulate, SoA", "mixed strides",
                 "output over the densities", "self"):
        got = call(form).cpu().numpy()
        monkeypatch.setenv("F3D_PAIRSUM_K64", "1")
        ref = call(form).cpu().numpy()
        monkeypatch.delenv("F3D_PAIRSUM_K64")
        if form == "self" and min(ns, nt) == 1:
            assert not got.any() and not ref.any()
        else:
            assert rel2(got, ref) < tol, form


@pytest.mark.parametrize("kernel", ["oseen", "rotlet", "stresslet"])
@pytest.mark.parametrize("ns,nt,one", [(4096, 2048, True), (4096, 5000, False),
                                       (3000, 9000, False), (512, 40000, False),
                                       (128, 200000, True), (4097, 2048, False)])
def test_one_launch_sums_stop_where_their_last_turn_is_short(kernel, ns, nt, one, monkeypatch):
    """A second turn of the CUs for a few workgroups makes the one launch the
    slower path (4096 x 5000: 40 against 27 us): such a call takes the general
    path, bit for bit; the others agree with it (64 x 1e-14, as above).  The
    stresslet's line lies lower: 22.7 against 17.5 us at 4096 x 2000."""
    s, t, d, n = (_dev(a) for a in _problem(ns + nt, ns, nt))
    call = lambda: FK.pairsum(kernel, s, d, t, src_nrm=n, eta=0.7).cpu().numpy()
    got = call()
    monkeypatch.setenv("F3D_PAIRSUM_DIRECT", "0")
    ref = call()
    if (kernel, ns) == ("stresslet", 4096):
        one = False
    assert np.array_equal(got, ref) != one
    assert rel2(got, ref) < 64 * 1e-14


@pytest.mark.parametrize("n", [258, 1400])
def test_one_launch_shell_matches_the_general_path(n, monkeypatch):
    """The shell operator's epilogue (singularity subtraction, completion sum,
    added flow) on both paths."""
    from fiber3d_amd import configs
    from fiber3d_amd.system import Shell
    xs, ns_, ws_ = configs.make_periphery(n, 3.0)
    sh = Shell(xs, ns_, ws_)
    rng = np.random.default_rng(n)
    q, add = _dev(rng.normal(size=(len(xs), 3))), _dev(rng.normal(size=(len(xs), 3)))
    got = sh.apply(q, add=add).cpu().numpy()
    monkeypatch.setenv("F3D_PAIRSUM_K64", "1")
    ref = sh.apply(q, add=add).cpu().numpy()
    assert rel2(got, ref) < 64 * 1e-14


@pytest.mark.parametrize("precision,ns,nt", [("f64", 300, 70), ("f64", 5000, 3000),
                                             ("f32c", 300, 70)])
def test_densities_and_normals_in_their_own_layouts(precision, ns, nt):
    """Positions, normals and densities in different layouts (in both paths of
    FP64) give the bits of the same call on contiguous copies."""
    print(f"case layouts {precision} ns={ns}", flush=True)
    s, t, d, n = (_dev(a) for a in _problem(ns, ns, nt, near=False))
    soa = d.t().contiguous().t()
    every_other = torch.empty((2 * ns, 3), dtype=torch.float64, device="cuda")[::2].copy_(n)
    kw = dict(eta=0.8, precision=precision)
    a = FK.pairsum("stresslet", s, soa, t, src_nrm=every_other, **kw)
    b = FK.pairsum("stresslet", s, d, t, src_nrm=n, **kw)
    assert torch.equal(a, b)
    assert torch.equal(FK.pairsum("oseen", s, soa, t, **kw), FK.pairsum("oseen", s, d, t, **kw))


@pytest.mark.parametrize("prec", ["f64", "f32c"])
@pytest.mark.parametrize("ns", [1000, 4096, 4097])
@pytest.mark.parametrize("kind", ["oseen", "stresslet"])
def test_reversed_exclusion_ranges_are_empty(kind, ns, prec):
    """A range with hi < lo excludes nothing, whichever kernel takes the call
    and whatever the ranges of the targets beside it."""
    from fiber3d_amd.kernels import pairsum
    print(f"case reversed ranges {kind} {ns} {prec}", flush=True)
    rng = np.random.default_rng(ns)
    X, F, T = (torch.from_numpy(rng.normal(size=(n, 3))).cuda() for n in (ns, ns, 130))
    lo = torch.from_numpy(rng.integers(0, ns, 130).astype(np.int32)).cuda()
    empty, rev = lo.clone(), lo - 1 - torch.arange(130, dtype=torch.int32, device="cuda")
    empty[::3] += 40
    rev[::3] = empty[::3]
    kw = dict(src_nrm=F if kind == "stresslet" else None, precision=prec)
    want = pairsum(kind, X, F, T, excl=(lo, empty), **kw)
    assert torch.equal(pairsum(kind, X, F, T, excl=(lo, rev), **kw), want)
    none = pairsum(kind, X, F, T, excl=(lo, lo - 1), **kw)
    assert torch.equal(none, pairsum(kind, X, F, T, excl=(lo, lo), **kw))


def _sums(count, ns=20000, nt=3000):
    """Calls of pairsum (general path, several launches each) on data of their
    own, with the results of serial runs."""
    rng = np.random.default_rng(count)
    calls = []
    for k in range(count):
        X, F, T = (torch.from_numpy(rng.normal(size=(n, 3))).cuda() for n in (ns + k, ns + k, nt))
        kw = dict(src_nrm=F) if k % 2 else {}
        calls.append(lambda kind=("oseen", "stresslet")[k % 2], X=X, F=F, T=T, kw=kw:
                     FK.pairsum(kind, X, F, T, precision=("f64", "f32c")[k // 2 % 2], **kw))
    want = [c() for c in calls]
    torch.cuda.synchronize()
    return calls, want


def test_sums_on_several_streams_do_not_share_a_workspace():
    """Sums queued on different streams at once, and graphs recorded on one stream
    while it runs sums of its own, give what serial runs give."""
    print("case sums on several streams", flush=True)
    calls, want = _sums(4)
    streams = [torch.cuda.Stream() for _ in calls]
    for _ in range(5):
        got = [None] * len(calls)
        for s in streams:
            s.wait_stream(torch.cuda.current_stream())
        for k, (c, s) in enumerate(zip(calls, streams)):
            with torch.cuda.stream(s):
                got[k] = c()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(got, want))
    # recorded on streams[0], replayed on the current stream beside eager sums there
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=streams[0]):
        out = calls[1]()
    for _ in range(5):
        out.zero_()
        streams[0].wait_stream(torch.cuda.current_stream())
        graph.replay()
        with torch.cuda.stream(streams[0]):
            eager = calls[0]()
        torch.cuda.synchronize()
        assert torch.equal(out, want[1]) and torch.equal(eager, want[0])


def test_sums_from_several_threads_on_one_stream():
    """A sum's launches are queued together: those of another thread on the same
    stream come before or after."""
    print("case sums from several threads", flush=True)
    import threading
    calls, want = _sums(4, ns=6000, nt=1000)
    got = [[] for _ in calls]

    def work(k):
        for _ in range(20):
            got[k].append(calls[k]())
    threads = [threading.Thread(target=work, args=(k,)) for k in range(len(calls))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    for g, w in zip(got, want):
        assert len(g) == 20 and all(torch.equal(a, w) for a in g)


@pytest.mark.parametrize("ns", [100, 5000])
def test_densities_and_normals_in_host_memory_are_copied(ns):
    """Densities and normals on the host, in either layout, act as their
    copies on the positions' device."""
    print(f"case host densities {ns}", flush=True)
    rng = np.random.default_rng(ns)
    X, F, N = (torch.from_numpy(rng.normal(size=(ns, 3))) for _ in range(3))
    T = torch.from_numpy(rng.normal(size=(64, 3))).cuda()
    soa = lambda t: t.t().contiguous().t()
    want = FK.pairsum("stresslet", X.cuda(), F.cuda(), T, src_nrm=N.cuda())
    for f, n in ((soa(F), N.cuda()), (F, N), (F.cuda(), soa(N))):
        assert torch.equal(FK.pairsum("stresslet", X.cuda(), f, T, src_nrm=n), want)
