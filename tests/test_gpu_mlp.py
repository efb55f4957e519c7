"""MFMA BF16 GEMM and the MLP forward/backward against FP64 references."""
import numpy as np
import pytest
import torch

from conftest import rel2
from fiber3d_amd import learned as LG
from oracle import mlp as OM

pytestmark = pytest.mark.gpu


def _bf16(a):
    return torch.from_numpy(np.asarray(a, np.float32)).bfloat16().float().double().numpy()


@pytest.mark.parametrize("M,N,K", [(64, 64, 16), (100, 70, 37), (1000, 256, 256), (3, 5, 7)])
def test_gemm_bf16_matches_fp64_of_rounded_inputs(M, N, K):
    print(f"case gemm {M}x{N}x{K}", flush=True)
    rng = np.random.default_rng(M + N + K)
    A = rng.normal(size=(M, K)).astype(np.float32)
    B = rng.normal(size=(K, N)).astype(np.float32)
    ref = _bf16(A) @ _bf16(B)
    C = torch.empty((M, N), device="cuda")
    LG.gemm(torch.from_numpy(A).cuda(), torch.from_numpy(B).cuda(), C)
    torch.cuda.synchronize()
    assert rel2(C.cpu().numpy(), ref) < 1e-6  # FP32 accumulation of exact BF16 products
    # transposed operands and split-K atomic accumulation
    At = torch.from_numpy(A.T.copy()).cuda()
    C2 = torch.zeros((M, N), device="cuda")
    LG.gemm(At, torch.from_numpy(B).cuda(), C2, LG.EPI_ATOMIC, transA=True, ksplit=3)
    torch.cuda.synchronize()
    assert rel2(C2.cpu().numpy(), ref) < 1e-6


def test_mlp_forward_backward_against_oracle():
    print("case mlp fwd/bwd", flush=True)
    torch.manual_seed(0)
    net = LG.MLP(8, 3, width=256, seed=3)
    rng = np.random.default_rng(1)
    X = rng.normal(size=(2000, 8)).astype(np.float32)
    T = rng.normal(size=(2000, 3)).astype(np.float32)
    Xd = torch.from_numpy(X).cuda()
    Y = net.forward(Xd, keep=True)
    dY = (2.0 / Y.numel()) * (Y - torch.from_numpy(T).cuda())
    g = net.backward(dY.contiguous())
    torch.cuda.synchronize()
    params = [p.double().cpu().numpy() for p in net.params]
    Yr, _ = OM.forward(params, X.astype(np.float64))
    gr = OM.grads(params, X.astype(np.float64), T.astype(np.float64))
    # BF16 operands (8-bit mantissa): a few 1e-3 relative on products of
    # width-256 layers
    assert rel2(Y.cpu().numpy(), Yr) < 2e-2
    for a, b in zip(g, gr):
        assert rel2(a.cpu().numpy(), b) < 5e-2


def test_mlp_training_reduces_loss():
    print("case mlp train", flush=True)
    rng = np.random.default_rng(2)
    X = rng.normal(size=(4096, 6)).astype(np.float32)
    T = (np.sin(X[:, :1]) + 0.5 * X[:, 1:2] * X[:, 2:3]).astype(np.float32)
    net = LG.MLP(6, 1, seed=0)
    Xd, Td = torch.from_numpy(X).cuda(), torch.from_numpy(T).cuda()
    first = net.train_step(Xd, Td, lr=1e-3)
    for _ in range(300):
        last = net.train_step(Xd, Td, lr=1e-3)
    assert last < 0.1 * first


@pytest.mark.parametrize("N", [128, 256])
@pytest.mark.parametrize("M,K", [(4099, 256), (1000, 48), (257, 160), (4096, 256), (32832, 64)])
@pytest.mark.parametrize("epi", ["store", "bias_relu", "bias", "relu_grad"])
def test_per_node_layer_kernels_agree(N, M, K, epi):
    """The per-node layer kernels (resident-weight, streaming, tiled; chosen
    per N through f3d_gemm_set_stream) on one problem with each epilogue,
    partial last row blocks included, and whole row blocks only (M = 4096:
    fewer row blocks than workgroups; M = 32832: 1026 or 513 row blocks, an
    odd count for some workgroups): each meets the FP64 product of the
    BF16-rounded inputs, and the Z output of the bias + ReLU epilogue holds
    the pre-activation."""
    from fiber3d_amd import _lib as L
    print(f"case layer kernels {M}x{N}x{K} {epi}", flush=True)
    rng = np.random.default_rng(M * 7 + N + K)
    A = rng.normal(size=(M, K)).astype(np.float32)
    B = rng.normal(size=(K, N)).astype(np.float32)
    bias = rng.normal(size=N).astype(np.float32)
    zin = rng.normal(size=(M, N)).astype(np.float32)
    pre = _bf16(A) @ _bf16(B)
    code = {"store": LG.EPI_STORE, "bias_relu": LG.EPI_BIAS_RELU, "bias": LG.EPI_BIAS,
            "relu_grad": LG.EPI_RELU_GRAD}[epi]
    if epi == "store":
        ref = pre
    elif epi == "bias":
        ref = pre + bias
    elif epi == "bias_relu":
        ref = np.maximum(pre + bias, 0.0)
    else:
        ref = np.where(zin > 0, pre, 0.0)
    lib = L.load()
    try:
        for mode in (2, 1, 0):
            L.check(lib.f3d_gemm_set_stream(N, mode), "f3d_gemm_set_stream")
            C = torch.full((M, N), 7.0, device="cuda")
            Z = torch.full((M, N), 7.0, device="cuda") if epi == "bias_relu" else None
            LG.gemm(torch.from_numpy(A).cuda(), torch.from_numpy(B).cuda(), C, code,
                    bias=torch.from_numpy(bias).cuda() if epi in ("bias", "bias_relu") else None,
                    Z=Z, Zin=torch.from_numpy(zin).cuda() if epi == "relu_grad" else None)
            torch.cuda.synchronize()
            assert rel2(C.cpu().numpy(), ref) < 1e-6, mode
            if Z is not None:
                assert rel2(Z.cpu().numpy(), pre + bias) < 1e-6, mode
    finally:
        from fiber3d_amd import autotune
        autotune.apply()


@pytest.mark.parametrize("M,n_in,n_out,width", [(1, 1, 1, 256), (63, 5, 2, 64), (64, 23, 4, 256),
                                               (257, 23, 4, 256), (1000, 7, 65, 130),
                                               (20000, 23, 4, 256)])
def test_mlp_passes_against_fp64(M, n_in, n_out, width):
    """The net's forward and backward passes at the edges of the products'
    tiles and sample slices, for a strided input and output gradient, against
    FP64 products of the same BF16-rounded operands: FP32 accumulation over K
    terms (2 K eps of the absolute products, element by element)."""
    print(f"case mlp passes M={M} {n_in}-{width}-{n_out}", flush=True)
    rng = np.random.default_rng(M + width)
    net = LG.MLP(n_in, n_out, width=width, seed=1)
    X = torch.from_numpy(rng.normal(size=(n_in + 1, M)).astype(np.float32)).cuda().t()[:, :n_in]
    dY = torch.from_numpy(rng.normal(size=(n_out, M)).astype(np.float32)).cuda().t()
    Y = net.forward(X, keep=True)
    _, H1, H2 = net._cache
    g = [t.cpu().double().numpy() for t in net.backward(dY)]
    h = lambda t: t.detach().cpu().double().numpy()
    W, b = [h(t) for t in net.W], [h(t) for t in net.b]

    def check(got, A, B, add=0.0, mask=None):
        A, B = _bf16(A), _bf16(B)
        ref, mag = A @ B + add, np.abs(A) @ np.abs(B) + np.abs(add)
        if mask is not None:
            ref, mag = ref * mask, mag * mask
        assert (np.abs(got - ref) <= 2 * (A.shape[1] + 2) * 2.0 ** -24 * mag).all()
        return ref
    pre = check(h(H1), h(X), W[0], b[0], mask=h(H1) > 0)
    assert (pre[h(H1) > 0] > -1e-3).all()
    check(h(H2), h(H1), W[1], b[1], mask=h(H2) > 0)
    check(h(Y), h(H2), W[2], b[2])
    # the gradients' inner factors are not returned: FP64 from the same masks
    # and BF16 operands, to the rounding of one BF16 operand of each product
    d2 = (_bf16(h(dY)) @ _bf16(W[2]).T) * (h(H2) > 0)
    d1 = (_bf16(d2) @ _bf16(W[1]).T) * (h(H1) > 0)
    for got, A, B in ((g[2], h(H2).T, h(dY)), (g[1], h(H1).T, d2), (g[0], h(X).T, d1)):
        mag = np.abs(_bf16(A)) @ np.abs(_bf16(B))
        assert (np.abs(got - _bf16(A) @ _bf16(B)) <= 2.0 ** -7 * mag + 1e-30).all()
    for got, B in ((g[5], h(dY)), (g[4], d2), (g[3], d1)):
        assert (np.abs(got - B.sum(0)) <= 2.0 ** -7 * np.abs(B).sum(0) + 1e-30).all()


@pytest.mark.parametrize("N", [128, 256])
@pytest.mark.parametrize("M,K", [(49152, 32), (49153, 48), (65599, 256)])
def test_per_node_layer_kernels_of_many_rows(N, M, K):
    """The streaming and resident kernels from the row count at which they
    take over, whole and partial last blocks."""
    from fiber3d_amd import _lib as L
    print(f"case layer kernels of many rows {M}x{N}x{K}", flush=True)
    rng = np.random.default_rng(M + N + K)
    A = rng.normal(size=(M, K)).astype(np.float32)
    B = rng.normal(size=(K, N)).astype(np.float32)
    bias = rng.normal(size=N).astype(np.float32)
    ref = np.maximum(_bf16(A) @ _bf16(B) + bias, 0.0)
    try:
        for mode in (2, 1):
            L.check(L.load().f3d_gemm_set_stream(N, mode), "f3d_gemm_set_stream")
            C = torch.full((M, N), 7.0, device="cuda")
            LG.gemm(torch.from_numpy(A).cuda(), torch.from_numpy(B).cuda(), C, LG.EPI_BIAS_RELU,
                    bias=torch.from_numpy(bias).cuda())
            assert rel2(C.cpu().numpy(), ref) < 1e-6, mode
    finally:
        from fiber3d_amd import autotune
        autotune.apply()


def test_adam_and_mse_against_fp64():
    """Three fused optimiser steps and the loss's gradient against FP64."""
    print("case adam mse", flush=True)
    rng = np.random.default_rng(4)
    net = LG.MLP(3, 2, seed=2)
    P = [p.cpu().double().numpy() for p in net.params]
    m, v = [np.zeros_like(p) for p in P], [np.zeros_like(p) for p in P]
    for t in range(1, 4):
        G = [rng.normal(size=p.shape).astype(np.float32) for p in P]
        net.adam([torch.from_numpy(q).cuda() for q in G], lr=1e-2)
        for k, q in enumerate(G):
            q = q.astype(np.float64)
            m[k] = 0.9 * m[k] + 0.1 * q
            v[k] = 0.999 * v[k] + 0.001 * q * q
            P[k] -= 1e-2 * (m[k] / (1 - 0.9 ** t)) / (np.sqrt(v[k] / (1 - 0.999 ** t)) + 1e-8)
    for p, r in zip(net.params, P):
        np.testing.assert_allclose(p.cpu().double().numpy(), r, rtol=0, atol=3e-6)
    X = torch.from_numpy(rng.normal(size=(777, 3)).astype(np.float32)).cuda()
    T = torch.from_numpy(rng.normal(size=(777, 2)).astype(np.float32)).cuda()
    Y = net.forward(X)
    loss = net.train_step(X, T, lr=0.0)
    assert abs(loss - float(((Y.double() - T.double()) ** 2).mean())) <= 1e-6 * loss


def test_mlp_passes_take_any_layout_and_check_types():
    """A strided weight (and bias) acts as the dense copy of its values, in the
    forward and the backward pass, also when the process's default type is
    FP64; a layer without a bias adds none; a weight of another type or shape
    is refused."""
    print("case mlp layouts", flush=True)
    rng = np.random.default_rng(8)
    X = torch.from_numpy(rng.normal(size=(300, 5)).astype(np.float32)).cuda()
    dY = torch.from_numpy(rng.normal(size=(300, 2)).astype(np.float32)).cuda()

    def passes(net):
        return [net.forward(X, keep=True)] + net.backward(dY)
    net, dense = LG.MLP(5, 2, seed=6), LG.MLP(5, 2, seed=6)
    for k in range(3):
        w = torch.from_numpy(rng.normal(size=net.W[k].shape).astype(np.float32)).cuda() / 16
        b = torch.from_numpy(rng.normal(size=net.b[k].shape).astype(np.float32)).cuda()
        dense.W[k], dense.b[k] = w, b
        net.W[k] = w.t().contiguous().t()
        net.b[k] = torch.stack([b, -b], 1)[:, 0]
    want = passes(dense)
    assert all(torch.equal(a, b) for a, b in zip(passes(net), want))
    torch.set_default_dtype(torch.float64)
    try:
        assert all(torch.equal(a, b) for a, b in zip(passes(net), want))
    finally:
        torch.set_default_dtype(torch.float32)
    net.b[1], dense.b[1] = None, torch.zeros_like(dense.b[1])
    assert torch.equal(net.forward(X), dense.forward(X))
    for k in range(3):
        for bad in (dense.W[k].double(), dense.W[k][:-1], dense.W[k].cpu()):
            net.W[k] = bad
            with pytest.raises(AssertionError):
                net.forward(X)
            if k:
                with pytest.raises(AssertionError):
                    net.backward(dY)
        net.W[k] = dense.W[k]


def _adam_ref(p, g, m, v, t, lr):
    g = g.astype(np.float64)
    m = 0.9 * m + 0.1 * g
    v = 0.999 * v + 0.001 * g * g
    return p - lr * (m / (1 - 0.9 ** t)) / (np.sqrt(v / (1 - 0.999 ** t)) + 1e-8), m, v


@pytest.mark.parametrize("odd", ["f64_grad", "strided_param", "strided_moment", "row_grad"])
def test_adam_on_tensors_of_any_layout(odd):
    """Gradients of another type or a broadcast shape, and parameters or
    moments that are views, take the same step as dense ones, and what lies
    beside a view stays as it is."""
    print(f"case adam {odd}", flush=True)
    rng = np.random.default_rng(14)
    net = LG.MLP(4, 3, width=32, seed=3)
    room = torch.full((32, 64), 5.0, device="cuda")
    if odd == "strided_param":
        room[:, ::2] = net.params[1]
        net.params[1] = room[:, ::2]
    if odd == "strided_moment":
        net.m[1] = room[:, ::2].zero_()
    P = [p.cpu().double().numpy() for p in net.params]
    m, v = [np.zeros_like(p) for p in P], [np.zeros_like(p) for p in P]
    for t in (1, 2):
        G = [rng.normal(size=p.shape).astype(np.float32) for p in P]
        if odd == "row_grad":
            G[1] = G[1][:1]
        g = [torch.from_numpy(q).cuda() for q in G]
        if odd == "f64_grad":
            g = [q.double() for q in g]
        net.adam(g, lr=1e-2)
        for k, q in enumerate(G):
            P[k], m[k], v[k] = _adam_ref(P[k], np.broadcast_to(q, P[k].shape), m[k], v[k], t, 1e-2)
    for p, r in zip(net.params, P):
        np.testing.assert_allclose(p.cpu().double().numpy(), r, rtol=0, atol=3e-6)
    assert bool((room[:, 1::2] == 5.0).all())


def test_adam_refuses_tensors_it_cannot_use():
    """A gradient of the wrong shape or in host memory is an error."""
    print("case adam refused", flush=True)
    for bad in (lambda g: g[:-1], lambda g: g.cpu()):
        net = LG.MLP(4, 3, width=32, seed=3)
        g = [torch.ones_like(p) for p in net.params]
        g[1] = bad(g[1])
        with pytest.raises(RuntimeError):
            net.adam(g)


def test_train_step_takes_the_targets_that_torch_subtracts():
    """Targets that broadcast, of another type, one number or one value in host
    memory train as the full FP32 tensor does; those that torch cannot subtract
    from the output are refused."""
    print("case train_step targets", flush=True)
    rng = np.random.default_rng(21)
    X = torch.from_numpy(rng.normal(size=(70, 3)).astype(np.float32)).cuda()
    row = torch.tensor([1.5, -0.25], device="cuda")
    full = row.expand(70, 2)

    def params(target):
        net = LG.MLP(3, 2, width=32, seed=4)
        loss = net.train_step(X, target, lr=1e-2)
        return loss, [p.cpu() for p in net.params]
    for target, same in ((row, full), (full.half(), full), (full.t().contiguous().t(), full),
                         (2.0, torch.full((70, 2), 2.0, device="cuda")),
                         (torch.tensor(2.0), torch.full((70, 2), 2.0, device="cuda"))):
        (la, pa), (lb, pb) = params(target), params(same.contiguous())
        assert abs(la - lb) <= 1e-6 * lb
        for a, b in zip(pa, pb):
            torch.testing.assert_close(a, b, rtol=0, atol=2e-6)
    for bad in (full.cpu(), full > 0):
        with pytest.raises(RuntimeError):
            params(bad)
    with pytest.raises(AssertionError):
        params(full.double())


def test_mlp_passes_of_no_samples():
    """An empty batch has an empty output and zero gradients."""
    print("case mlp no samples", flush=True)
    net = LG.MLP(5, 2, width=64, seed=6)
    Y = net.forward(torch.empty((0, 5), device="cuda"), keep=True)
    assert Y.shape == (0, 2)
    for g, p in zip(net.backward(torch.empty((0, 2), device="cuda")), net.params):
        assert g.shape == p.shape and not bool(g.any())


@pytest.mark.parametrize("n", [1, 3, 2 ** 24 + 1])
def test_mse_gradient_factor_is_rounded_once(n):
    """dy = fl(2 / n) (y - t), also where n itself is not an FP32 number."""
    from fiber3d_amd import _lib as L
    from fiber3d_amd.kernels import _stream
    print(f"case mse factor n={n}", flush=True)
    y, t = torch.rand(n, device="cuda"), torch.rand(n, device="cuda")
    dy, loss = torch.empty_like(y), torch.empty((), device="cuda")
    ws = torch.empty(L.load().f3d_mse_workspace_size(), dtype=torch.uint8, device="cuda")
    L.check(L.load().f3d_mse(n, L.ptr(y), L.ptr(t), L.ptr(dy), L.ptr(loss), L.ptr(ws), ws.numel(),
                             _stream()), "f3d_mse")
    assert torch.equal(dy, (2.0 / n) * (y - t))
    ref = float(((y - t).double() ** 2).mean())
    assert abs(float(loss) - ref) <= 1e-6 * ref


def _layer(M, N, K, epi, form, seed, mode, in_place=False):
    """One gemm call in a mode of f3d_gemm_set_stream; its results against FP64
    products of the BF16-rounded operands, element by element: FP32
    accumulation over K terms (2 K eps of the absolute products)."""
    from fiber3d_amd import _lib as L
    from fiber3d_amd import autotune
    g = torch.Generator(device="cuda").manual_seed(seed)
    rnd = lambda *s: torch.randn(*s, device="cuda", generator=g)
    A = rnd(M, K + 3)[:, :K] if form == "strided" else rnd(M, K)
    B, bias, zin = rnd(K, N), rnd(N), rnd(M, N)
    b16 = lambda t: t.bfloat16().double()
    pre, mag = b16(A) @ b16(B), b16(A).abs() @ b16(B).abs()
    code = {"store": LG.EPI_STORE, "bias_relu": LG.EPI_BIAS_RELU, "bias": LG.EPI_BIAS,
            "relu_grad": LG.EPI_RELU_GRAD}[epi]
    if epi.startswith("bias"):
        pre, mag = pre + bias.double(), mag + bias.double().abs()
    want = pre.clamp(min=0) if epi == "bias_relu" else (
        pre * (zin > 0) if epi == "relu_grad" else pre)
    C = A if in_place else torch.full((M, N), 7.0, device="cuda")
    Z = torch.full((M, N), 7.0, device="cuda") if epi == "bias_relu" and not in_place else None
    L.check(L.load().f3d_gemm_set_stream(N, mode), "f3d_gemm_set_stream")
    try:
        LG.gemm(A, B.t().contiguous() if form == "transB" else B, C, code, transB=form == "transB",
                bias=bias if epi.startswith("bias") else None, Z=Z,
                Zin=zin if epi == "relu_grad" else None)
        torch.cuda.synchronize()
    finally:
        autotune.apply()
    bound = 2 * (K + 2) * 2.0 ** -24 * mag
    assert bool(((C.double() - want).abs() <= bound).all()), mode
    if Z is not None:
        assert bool(((Z.double() - pre).abs() <= bound).all()), mode


@pytest.mark.parametrize("N", [128, 256])
@pytest.mark.parametrize("epi", ["store", "bias_relu", "bias", "relu_grad"])
@pytest.mark.parametrize("M,K,form", [(4097, 16, "dense"), (4159, 32, "transB"), (12289, 96, "dense"),
                                      (49153, 23, "dense"), (49280, 50, "transB"),
                                      (49153, 48, "strided"), (49159, 64, "transB"),
                                      (32768, 100, "dense"), (32767, 250, "transB")])
def test_row_block_kernels_with_every_epilogue(M, K, form, epi, N):
    """The resident and streaming kernels where the dispatch takes them (a K
    that is not a multiple of 16 or of 4, or rows that are not aligned, goes to
    the streaming kernel in both modes), with every epilogue, the
    pre-activations, transposed weights and partial last row blocks."""
    print(f"case row blocks {M}x{N}x{K} {form} {epi}", flush=True)
    for mode in (2, 1):
        _layer(M, N, K, epi, form, M + K, mode)


@pytest.mark.parametrize("N", [128, 256])
@pytest.mark.parametrize("M", [128, 1000, 4096])
def test_layers_in_place(M, N):
    """An N x N layer whose output is its input's storage."""
    print(f"case layer in place {M}x{N}", flush=True)
    for mode in (2, 1):
        _layer(M, N, N, "bias_relu", "dense", M + N, mode, in_place=True)


def test_more_rows_than_the_tiled_grid_has():
    """A short K, which the tiled kernel takes, with more row tiles than a grid's y
    extent: the rows go to a row-block kernel."""
    print("case rows beyond the tiled grid", flush=True)
    M, N, K = 64 * 65536 + 1, 128, 4
    A, B = torch.randn(M, K, device="cuda"), torch.randn(K, N, device="cuda")
    C = torch.full((M, N), 7.0, device="cuda")
    LG.gemm(A, B, C)
    for rows in (slice(0, 1000), slice(M // 2, M // 2 + 1000), slice(M - 1000, M)):
        want = A[rows].bfloat16().double() @ B.bfloat16().double()
        assert rel2(C[rows].cpu().numpy(), want.cpu().numpy()) < 1e-6


def test_adam_on_shared_parameters():
    """A parameter listed twice takes both of its steps, one after the other."""
    print("case adam shared", flush=True)
    rng = np.random.default_rng(5)
    net = LG.MLP(4, 3, width=4096, seed=3)
    net.params[4] = net.params[3]
    G = [rng.normal(size=p.shape).astype(np.float32) for p in net.params]
    net.adam([torch.from_numpy(q).cuda() for q in G], lr=1e-2)
    want = np.zeros(4096)
    for q in (G[3], G[4]):
        want = _adam_ref(want, q, np.zeros(4096), np.zeros(4096), 1, 1e-2)[0]
    np.testing.assert_allclose(net.params[3].cpu().double().numpy(), want, rtol=0, atol=3e-6)
