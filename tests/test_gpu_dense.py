"""GPU batched LU / solve / block GEMV against LAPACK (SciPy) on the host."""
import numpy as np
import pytest
import scipy.linalg as sla
import torch

from conftest import rel2
from fiber3d_amd.dense import BatchedLU, BlockGemv, BlockSet, DenseGemv

pytestmark = pytest.mark.gpu


def _mats(sizes, seed, cond_shift=4.0):
    rng = np.random.default_rng(seed)
    return [rng.normal(size=(n, n)) + cond_shift * np.eye(n) for n in sizes]


SIZES = [64, 96, 128, 192, 256, 37, 1, 100, 255, 17]


def test_lu_factor_f64_matches_lapack():
    print("case lu f64 factor", flush=True)
    mats = _mats(SIZES, 0)
    bs = BlockSet(SIZES)
    A = bs.pack(mats)
    lu = BatchedLU(bs, A, precision="f64")
    torch.cuda.synchronize()
    LU = bs.unpack(lu.lu64)
    piv = lu.piv.cpu().numpy()
    assert lu.info.cpu().numpy().tolist() == [0] * len(SIZES)
    for b, M in enumerate(mats):
        lu_ref, piv_ref = sla.lu_factor(M)
        o = bs.x_off_h[b]
        np.testing.assert_array_equal(piv[o:o + SIZES[b]], piv_ref)
        assert rel2(LU[b], lu_ref) < 1e-12


@pytest.mark.parametrize("n", [15, 16, 31, 32, 33, 48, 63, 65, 129, 161, 224, 241])
@pytest.mark.parametrize("precision", ["f64", "f32c"])
def test_lu_factor_strip_edges(precision, n):
    """Orders at the edges of the factorisation's panels, strips and waves:
    LAPACK's pivots and factors in FP64, P (Dr A Dc) = L U in FP32.  Beside
    each, a block of the same order whose columns are full of equal maxima (the
    first row must win), one with a zero column and one with a column of
    NaN."""
    print(f"case lu strip edges {precision} n={n}", flush=True)
    rng = np.random.default_rng(n)
    M = rng.normal(size=(n, n))
    # exact in either precision: entries of L and U in {-1, 0, 1}
    T = (np.tril(rng.integers(-1, 2, size=(n, n)), -1) + np.eye(n)) @ (
        np.triu(rng.integers(-1, 2, size=(n, n)), 1) + np.eye(n))
    Z = M.copy()
    Z[:, n // 2] = 0.0
    N = M.copy()
    N[:, n - 1] = np.nan
    bs = BlockSet([n] * 4)
    lu = BatchedLU(bs, bs.pack([M, T, Z, N]), precision=precision)
    torch.cuda.synchronize()
    LU = bs.unpack((lu.lu64 if precision == "f64" else lu.lu32).double())
    piv = lu.piv.cpu().numpy().reshape(4, n)
    assert lu.info.cpu().numpy().tolist()[:3] == [0, 0, n // 2 + 1]
    ref, piv_ref = sla.lu_factor(M)
    if precision == "f64":
        np.testing.assert_array_equal(piv[0], piv_ref)
        assert rel2(LU[0], ref) < 1e-12 * n
    for k in range(4):
        # the interchanges and the permutation agree, and rows stay in range
        p = np.arange(n)
        for j, q in enumerate(piv[k]):
            assert j <= q < n
            p[[j, q]] = p[[q, j]]
        np.testing.assert_array_equal(lu.perm.cpu().numpy()[k * n:(k + 1) * n], p)
    if precision == "f64":
        np.testing.assert_array_equal(piv[1], np.arange(n))
        np.testing.assert_array_equal(LU[1], sla.lu_factor(T)[0])
    As = M
    if precision == "f32c":
        As = lu.rs.cpu().numpy()[:n, None] * M * lu.cs.cpu().numpy()[None, :n]
    P = lu.perm.cpu().numpy()[:n]
    back = (np.tril(LU[0], -1) + np.eye(n)) @ np.triu(LU[0])
    # |L U - P A| <= 2 n eps |L| |U| element by element
    bound = (np.abs(np.tril(LU[0], -1)) + np.eye(n)) @ np.abs(np.triu(LU[0]))
    eps = 2.0 ** -53 if precision == "f64" else 2.0 ** -24
    assert (np.abs(back - As[P]) <= 2 * n * eps * bound + 1e-300).all()


@pytest.mark.parametrize("precision", ["f64", "f32c"])
def test_lu_solve_batched(precision):
    print(f"case lu solve {precision}", flush=True)
    mats = _mats(SIZES, 1)
    bs = BlockSet(SIZES)
    A = bs.pack(mats)
    lu = BatchedLU(bs, A, precision=precision, refine=10, tol=1e-14)
    rng = np.random.default_rng(2)
    xs = [rng.normal(size=n) for n in SIZES]
    b = np.concatenate([M @ x for M, x in zip(mats, xs)])
    y = lu.solve(torch.from_numpy(b).cuda())
    torch.cuda.synchronize()
    yh = y.cpu().numpy()
    tol = 1e-12
    for k, x in enumerate(xs):
        o = bs.x_off_h[k]
        assert rel2(yh[o:o + SIZES[k]], x) < tol, (k, SIZES[k])
    if precision == "f32c":
        it = lu.iters.cpu().numpy()
        assert it.max() >= 1 and it.max() < 10
    # in-place (y aliases x)
    bb = torch.from_numpy(b).cuda()
    lu.solve(bb, out=bb)
    torch.cuda.synchronize()
    assert rel2(bb.cpu().numpy(), np.concatenate(xs)) < tol


@pytest.mark.parametrize("precision", ["f64", "f32c"])
def test_lu_solve_segment_edges(precision):
    """One unrefined solve at the edges of the substitutions' 64-row segments
    and column chunks: the backward error of L U z = P (rs x), y = cs z with
    the kernel's own factors, element by element (3 n eps |L| |U| |z|)."""
    print(f"case lu solve segment edges {precision}", flush=True)
    sizes = [1, 2, 3, 5, 8, 63, 64, 65, 72, 80, 127, 128, 129, 135, 191, 192, 193, 200, 255, 256]
    mats = _mats(sizes, 11)
    bs = BlockSet(sizes)
    lu = BatchedLU(bs, bs.pack(mats), precision=precision, refine=0)
    x = np.random.default_rng(12).normal(size=bs.nrows)
    y = lu.solve(torch.from_numpy(x).cuda()).cpu().numpy()
    LU = bs.unpack((lu.lu64 if precision == "f64" else lu.lu32).double())
    perm = lu.perm.cpu().numpy()
    for k, n in enumerate(sizes):
        rows = slice(bs.x_off_h[k], bs.x_off_h[k] + n)
        rs, cs = (np.ones(n), np.ones(n)) if precision == "f64" else (
            lu.rs.cpu().numpy()[rows], lu.cs.cpu().numpy()[rows])
        Lo, U = np.tril(LU[k], -1) + np.eye(n), np.triu(LU[k])
        z = y[rows] / cs
        r = Lo @ (U @ z) - (rs * x[rows])[perm[rows]]
        bound = 3 * n * 2.0 ** -53 * (np.abs(Lo) @ (np.abs(U) @ np.abs(z)))
        assert (np.abs(r) <= bound).all(), n


def test_lu_solve_quotients_outside_the_safe_range():
    """Diagonal blocks whose pivots or right-hand sides lie where the
    reciprocal form of the quotient is not exact: the same numbers as a
    division, infinities and NaN included (the extreme pivots to 2 ulp)."""
    print("case lu solve quotients", flush=True)
    d = np.array([3.0, 7e200, 5e-201, 0.0, np.inf, 1.1e150, 3e-130, np.nan])
    x = np.array([1.0, 2.0, 3.0, 1.0, 2.0, 1e300, np.inf, 1.0])
    sizes = [1] * len(d)
    bs = BlockSet(sizes)
    lu = BatchedLU(bs, bs.pack([np.array([[v]]) for v in d]), precision="f64", refine=0)
    y = lu.solve(torch.from_numpy(x).cuda()).cpu().numpy()
    with np.errstate(divide="ignore", invalid="ignore"):
        ref = x / d
    fin = np.isfinite(ref)
    np.testing.assert_allclose(y[fin], ref[fin], rtol=2.0 ** -51, atol=0)
    np.testing.assert_array_equal(y[~fin], ref[~fin])


def test_lu_zero_pivot_info():
    M = np.eye(8)
    M[3, 3] = 0.0
    M[3, :] = 0.0
    bs = BlockSet([8, 8])
    lu = BatchedLU(bs, bs.pack([np.eye(8) * 2.0, M]), precision="f64")
    torch.cuda.synchronize()
    assert lu.info.cpu().numpy().tolist() == [0, 4]


def test_block_gemv():
    print("case block gemv", flush=True)
    rng = np.random.default_rng(4)
    ms = [12, 256, 64, 130]
    ks = [16, 200, 256, 3]
    mats = [rng.normal(size=(m, k)) for m, k in zip(ms, ks)]
    x_off = np.concatenate([[0], np.cumsum(ks)[:-1]])
    y_off = np.concatenate([[0], np.cumsum(ms)[:-1]])
    g = BlockGemv(ms, ks, x_off, y_off)
    M = g.pack(mats)
    x = rng.normal(size=sum(ks))
    y0 = rng.normal(size=sum(ms))
    y = torch.from_numpy(y0.copy()).cuda()
    g(M, torch.from_numpy(x).cuda(), y, alpha=2.0, beta=-0.5)
    torch.cuda.synchronize()
    ref = np.concatenate([2.0 * Mb @ x[xo:xo + k] for Mb, xo, k in zip(mats, x_off, ks)]) - 0.5 * y0
    assert rel2(y.cpu().numpy(), ref) < 1e-13


@pytest.mark.parametrize("beta", [0.0, 1.0])
def test_block_gemv_edges(beta):
    """Row counts at the edges of the segments and column counts at the edges
    of the waves' column groups (none, one, a group and one more, all waves).
    Sums of k <= 260 O(1) products: 260 eps of their absolute sum, here taken
    against |alpha| |M| |x| + |beta y|."""
    print(f"case block gemv edges beta={beta}", flush=True)
    rng = np.random.default_rng(11)
    ms, ks = zip(*[(m, k) for m in (1, 2, 31, 32, 33, 63, 64, 65, 127, 128, 129, 255, 256)
                   for k in (0, 1, 4, 7, 8, 9, 15, 16, 17, 31, 33, 64, 65, 127, 128, 129, 260)])
    mats = [rng.normal(size=(m, k)) for m, k in zip(ms, ks)]
    x_off = np.concatenate([[0], np.cumsum(ks)[:-1]])
    y_off = np.concatenate([[0], np.cumsum(ms)[:-1]])
    g = BlockGemv(ms, ks, x_off, y_off)
    x, y0 = rng.normal(size=sum(ks)), rng.normal(size=sum(ms))
    y = torch.from_numpy(y0.copy()).cuda()
    g(g.pack(mats), torch.from_numpy(x).cuda(), y, alpha=-1.5, beta=beta)
    got = y.cpu().numpy()
    for M, xo, yo in zip(mats, x_off, y_off):
        m, k = M.shape
        xb, yb = x[xo:xo + k], y0[yo:yo + m]
        ref = -1.5 * (M @ xb) + beta * yb
        scale = 1.5 * (np.abs(M) @ np.abs(xb)) + np.abs(beta * yb)
        assert (np.abs(got[yo:yo + m] - ref) <= 260 * 2.3e-16 * scale + 1e-300).all(), (m, k)


@pytest.mark.parametrize("beta", [0.0, -0.5])
def test_block_gemv_sum(beta):
    """Four products into the same rows, the later terms with fewer rows (none,
    up to a segment's edge, all) than the block; tolerance as above."""
    print(f"case block gemv sum beta={beta}", flush=True)
    rng = np.random.default_rng(12)
    ms = np.array([20, 32, 33, 64, 66, 128, 130, 256])
    rows = [ms, np.maximum(ms - 14, 1), np.minimum(ms, 32), np.minimum(ms, 64)]
    ks = [ms, np.array([5, 8, 8, 16, 17, 32, 33, 64]), ms, np.array([1, 0, 3, 260, 9, 15, 16, 7])]
    alphas = [1.0, -1.0, 0.5, 2.0]
    y_off = np.concatenate([[0], np.cumsum(ms)[:-1]])
    terms, host = [], []
    for m, k, a in zip(rows, ks, alphas):
        mats = [rng.normal(size=(mb, kb)) for mb, kb in zip(m, k)]
        x_off = np.concatenate([[0], np.cumsum(k)[:-1]])
        x = rng.normal(size=int(k.sum()))
        g = BlockGemv(m, k, x_off, y_off)
        terms.append((g, g.pack(mats), torch.from_numpy(x).cuda(), a))
        host.append((mats, x_off, x, a))
    y0 = rng.normal(size=int(ms.sum()))
    y = torch.from_numpy(y0.copy()).cuda()
    BlockGemv.sum(terms, y, beta=beta)
    got = y.cpu().numpy()
    for b, (m, yo) in enumerate(zip(ms, y_off)):
        ref, scale = beta * y0[yo:yo + m], np.abs(beta * y0[yo:yo + m])
        for mats, x_off, x, a in host:
            M = mats[b]
            xb = x[x_off[b]:x_off[b] + M.shape[1]]
            ref[:M.shape[0]] += a * (M @ xb)
            scale[:M.shape[0]] += np.abs(a) * (np.abs(M) @ np.abs(xb))
        assert (np.abs(got[yo:yo + m] - ref) <= 2 * 260 * 2.3e-16 * scale).all(), b


def test_batched_lu_on_real_fiber_blocks_config2_shape():
    """Workload 2 shape: fibers with N in {16, 24, 32, 48, 64} (n = 4N up to
    256), A_sq assembled from the fiber discretisation; FP32 LU + FP64
    refinement to 1e-12 against the FP64 LU in one batch."""
    print("case batched lu config2-like", flush=True)
    from fiber3d_amd import configs
    from fiber3d_amd.system import FiberSystem
    spec = configs.FiberSpec(160, [16, 24, 32, 48, 64], 1.0, 8.0)
    fibers = configs.make_fibers(spec, seed=2)
    S = FiberSystem(fibers, None, lu_precision="f32c", lu_refine=10, lu_tol=1e-14)
    rng = np.random.default_rng(5)
    xs = torch.from_numpy(rng.normal(size=S.bs.nrows)).cuda()
    b = torch.empty_like(xs)
    S.gA(S.A_buf, xs, b)          # b = A_sq x for every block
    y32 = S.lu.solve(b)
    lu64 = BatchedLU(S.bs, S.A_buf, precision="f64")
    y64 = lu64.solve(b)
    torch.cuda.synchronize()
    assert S.lu.info.cpu().numpy().max() == 0
    e32 = rel2(y32.cpu().numpy(), xs.cpu().numpy())
    e64 = rel2(y64.cpu().numpy(), xs.cpu().numpy())
    print(f"forward error f32+IR {e32:.2e}  f64 {e64:.2e}  max sweeps {int(S.lu.iters.max())}")
    # FP64 refinement drives every block's relative residual to 1e-12 or below
    Ay = torch.empty_like(b)
    S.gA(S.A_buf, y32, Ay)
    r = (b - Ay).cpu().numpy()
    bh = b.cpu().numpy()
    for k in range(S.bs.nb):
        o, n = S.bs.x_off_h[k], S.bs.sizes[k]
        assert np.linalg.norm(r[o:o + n]) <= 1e-12 * np.linalg.norm(bh[o:o + n]), k
    # forward error stays at the conditioning level of the FP64 factorisation
    assert e32 < max(1e4 * e64, 1e-9)


@pytest.mark.parametrize("kernel", ["mfma", "vector"])
def test_lu_factor_f32_is_a_factorisation(kernel, monkeypatch):
    """The equilibrated FP32 factors satisfy P (Dr A Dc) = L U to FP32
    accuracy, with ipiv and perm consistent (blocked MFMA kernel and the
    register-resident VALU kernel; orders not divisible by 32 included)."""
    print(f"case lu f32 factor {kernel}", flush=True)
    if kernel == "vector":
        monkeypatch.setenv("F3D_LU32_KERNEL", "vector")
    else:
        monkeypatch.delenv("F3D_LU32_KERNEL", raising=False)
    mats = _mats(SIZES, 7)
    bs = BlockSet(SIZES)
    lu = BatchedLU(bs, bs.pack(mats), precision="f32c")
    torch.cuda.synchronize()
    assert lu.info.cpu().numpy().tolist() == [0] * len(SIZES)
    LU = bs.unpack(lu.lu32.double())
    piv, perm = lu.piv.cpu().numpy(), lu.perm.cpu().numpy()
    rs, cs = lu.rs.cpu().numpy(), lu.cs.cpu().numpy()
    for b, M in enumerate(mats):
        n, o = SIZES[b], bs.x_off_h[b]
        As = rs[o:o + n, None] * M * cs[None, o:o + n]
        p = perm[o:o + n]
        ref = np.arange(n)
        for j in range(n):
            q = piv[o + j]
            assert j <= q < n
            ref[[j, q]] = ref[[q, j]]
        np.testing.assert_array_equal(p, ref)
        L = np.tril(LU[b], -1) + np.eye(n)
        U = np.triu(LU[b])
        assert np.abs(L).max() <= 1.0 + 1e-6          # partial pivoting
        err = np.abs(As[p] - L @ U).max() / np.abs(As).max()
        assert err < 2e-5, (n, err)


@pytest.mark.parametrize("count,m,offset", [(1, 3072, 0), (3, 1806, 0), (2, 7, 0), (2, 130, 1),
                                            (1, 1, 0)])
def test_dense_gemv_batched(count, m, offset):
    """Row-per-wave dense GEMV against NumPy in FP64: even and odd sizes, and
    an x that is not 16-byte aligned (the one-double-per-lane path)."""
    print(f"case dense gemv count={count} m={m} offset={offset}", flush=True)
    rng = np.random.default_rng(m + count)
    M = rng.normal(size=(count, m, m))
    x = rng.normal(size=count * m)
    g = DenseGemv(torch.from_numpy(M).cuda())
    xbuf = torch.zeros(count * m + offset, dtype=torch.float64, device="cuda")
    xbuf[offset:] = torch.from_numpy(x)
    y = torch.full((count * m,), float("nan"), dtype=torch.float64, device="cuda")
    g(xbuf[offset:], y)
    torch.cuda.synchronize()
    ref = np.einsum("bij,bj->bi", M, x.reshape(count, m)).ravel()
    assert rel2(y.cpu().numpy(), ref) < 1e-13


@pytest.mark.parametrize("count,m,offset", [(1, 3072, 0), (3, 1806, 0), (2, 7, 0), (2, 132, 1),
                                            (1, 1, 0)])
def test_dense_gemv_batched_f32_entries(count, m, offset):
    """FP32 matrix entries, FP64 vector and arithmetic: equal to the FP64
    product of the FP32-rounded matrix to FP64 rounding, on the four-floats-
    per-lane path (m a multiple of 4, aligned), odd sizes and an x that is not
    16-byte aligned (one entry per lane)."""
    print(f"case dense gemv f32 count={count} m={m} offset={offset}", flush=True)
    rng = np.random.default_rng(m + count + 1)
    M32 = rng.normal(size=(count, m, m)).astype(np.float32)
    x = rng.normal(size=count * m)
    g = DenseGemv(torch.from_numpy(M32).cuda())
    xbuf = torch.zeros(count * m + offset, dtype=torch.float64, device="cuda")
    xbuf[offset:] = torch.from_numpy(x)
    y = torch.full((count * m,), float("nan"), dtype=torch.float64, device="cuda")
    g(xbuf[offset:], y)
    torch.cuda.synchronize()
    ref = np.einsum("bij,bj->bi", M32.astype(np.float64), x.reshape(count, m)).ravel()
    assert rel2(y.cpu().numpy(), ref) < 1e-13


@pytest.mark.parametrize("n", [1, 64, 65, 130, 256])
def test_lu_solve_divides_by_pivots_beyond_the_reciprocal(n):
    """Upper triangular factors with pivots whose reciprocal over- or
    underflows, or whose quotients are the subnormal numbers: every entry is the
    correctly rounded quotient of its right-hand side (the rest of the factor is
    zero, so that nothing else rounds), in every segment of the rows."""
    print(f"case lu solve quotients at the ends of the range n={n}", flush=True)
    # (the oracle's C library, built for speed, leaves the host thread flushing
    # subnormal numbers to zero)
    torch.set_flush_denormal(False)
    rng = np.random.default_rng(n)
    d = np.ldexp(rng.uniform(1.0, 2.0, n) * rng.choice([-1.0, 1.0], n),
                 rng.choice([-1070, -1030, -1022, -700, -401, -3, 0, 401, 1000, 1023], n))
    q = np.ldexp(rng.uniform(1.0, 2.0, n), rng.integers(-30, 30, n))
    with np.errstate(over="ignore", under="ignore"):
        x = np.clip(d * q, -1e308, 1e308)
        ref = x / d
    bs = BlockSet([n])
    lu = BatchedLU(bs, bs.pack([np.eye(n)]), precision="f64", refine=0)
    lu.lu64.copy_(torch.from_numpy(np.diag(d).ravel()))
    y = lu.solve(torch.from_numpy(x).cuda()).cpu().numpy()
    np.testing.assert_array_equal(y, ref)


@pytest.mark.parametrize("mmax,nb,said", [(32, 40, 32), (64, 40, 64), (64, 2051, 64), (128, 2051, 128),
                                          (256, 2051, 256), (200, 40, 64), (200, 2051, 64),
                                          (200, 2051, 100)])
def test_block_gemv_of_many_blocks(mmax, nb, said):
    """Few and many blocks of each size class, with rows and columns at the edges of
    the waves' shares, and blocks taller than the call's mmax says; 260 eps of
    the absolute sums."""
    print(f"case block gemv many mmax={mmax} nb={nb} said={said}", flush=True)
    rng = np.random.default_rng(nb + mmax + said)
    ms = rng.choice([m for m in (1, 2, 31, 32, 33, 50, 63, 64, 65, 100, 127, 128, 129, 200, 256)
                     if m <= mmax], nb)
    ms[-1] = mmax
    ks = rng.choice([0, 1, 7, 8, 9, 15, 16, 17, 31, 32, 33, 64, 65, 129], nb)
    x_off, y_off = np.cumsum(ks) - ks, np.cumsum(ms) - ms
    mats = [rng.normal(size=(m, k)) for m, k in zip(ms, ks)]
    g = BlockGemv(ms, ks, x_off, y_off)
    g.mmax = said
    x, y0 = rng.normal(size=int(ks.sum()) + 1), rng.normal(size=int(ms.sum()))
    y = torch.from_numpy(y0.copy()).cuda()
    g(g.pack(mats), torch.from_numpy(x).cuda(), y, alpha=0.75, beta=-0.5)
    got = y.cpu().numpy()
    for M, xo, yo in zip(mats, x_off, y_off):
        m, k = M.shape
        xb, yb = x[xo:xo + k], y0[yo:yo + m]
        scale = 0.75 * (np.abs(M) @ np.abs(xb)) + 0.5 * np.abs(yb)
        assert (np.abs(got[yo:yo + m] - (0.75 * (M @ xb) - 0.5 * yb)) <= 260 * 2.3e-16 * scale).all()


def test_lu_factor_of_many_small_blocks():
    """Many blocks of order up to 64 take strips of 64 rows: the same factors,
    interchanges and zero pivots as in small batches, to the bit, with ties, zero
    columns, NaN and every order mixed."""
    print("case lu many small blocks", flush=True)
    rng = np.random.default_rng(77)
    sizes = [int(n) for n in rng.integers(1, 65, 1100)]
    sizes[:8] = [1, 15, 16, 17, 32, 33, 63, 64]
    mats = []
    for k, n in enumerate(sizes):
        M = rng.normal(size=(n, n))
        if k % 5 == 1:
            M = rng.integers(-1, 2, size=(n, n)).astype(float)  # ties, some singular
        elif k % 5 == 2:
            M[:, n // 2] = 0.0
        elif k % 50 == 3:
            M[n // 3, n // 2] = np.nan
        mats.append(M)
    bs = BlockSet(sizes)
    lu = BatchedLU(bs, bs.pack(mats), precision="f64", refine=0)
    LU, piv = bs.unpack(lu.lu64), lu.piv.cpu().numpy()
    perm, info = lu.perm.cpu().numpy(), lu.info.cpu().numpy()
    for k0 in range(0, len(sizes), 400):
        part = slice(k0, k0 + 400)
        b2 = BlockSet(sizes[part])
        l2 = BatchedLU(b2, b2.pack(mats[part]), precision="f64", refine=0)
        rows = slice(int(bs.x_off_h[k0]), int(bs.x_off_h[k0]) + b2.nrows)
        for a, b in zip(LU[part], b2.unpack(l2.lu64)):
            np.testing.assert_array_equal(a, b)
        np.testing.assert_array_equal(piv[rows], l2.piv.cpu().numpy())
        np.testing.assert_array_equal(perm[rows], l2.perm.cpu().numpy())
        np.testing.assert_array_equal(info[part], l2.info.cpu().numpy())


@pytest.mark.parametrize("nb", [3, 300, 2100])
def test_block_gemv_forms_agree_to_the_bit(nb):
    """A block's product is the same whatever the call's other blocks are: the
    forms for at most 64 and 128 rows keep the order of the one for all."""
    print(f"case block gemv forms nb={nb}", flush=True)
    rng = np.random.default_rng(nb)
    ms = rng.choice([1, 14, 31, 32, 33, 50, 63, 64], nb)
    ks = rng.choice([1, 7, 8, 9, 15, 16, 17, 33, 64, 65, 130], nb)
    mats = [rng.normal(size=(m, k)) for m, k in zip(ms, ks)]
    got = []
    for tall in (64, 100, 256):
        m, k = np.append(ms, tall), np.append(ks, 40)
        rest = np.random.default_rng(1)
        g = BlockGemv(m, k, np.cumsum(k) - k, np.cumsum(m) - m)
        x = np.append(np.random.default_rng(2).normal(size=int(ks.sum())), rest.normal(size=40))
        y = torch.ones(int(m.sum()), dtype=torch.float64, device="cuda")
        M = g.pack(mats + [rest.normal(size=(tall, 40))])
        g(M, torch.from_numpy(x).cuda(), y, alpha=0.7, beta=0.3)
        got.append(y.cpu().numpy()[:int(ms.sum())])
    np.testing.assert_array_equal(got[0], got[2])
    np.testing.assert_array_equal(got[1], got[2])
