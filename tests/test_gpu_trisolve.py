"""Triangular solves through inverted 512 x 512 diagonal blocks, at the sizes
where the tiling can go wrong: one row, the edges of the 16 x 16 tiles, of the
256 and 512 blocks and of the group of 32 blocks, and column counts at the
edges of 16, 32, 64 and 1024.

Factors L = I + strict, U = (2 .. 3) I + strict with entries below 1 / n: every
product has a condition number of a few units, so FP64 sums in any order agree
to a small multiple of n 2^-53 (2e-12 at 16500 at the very worst); the
tolerance is the 1e-12 of the existing triangular-solve tests."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _factor(n, lda, seed):
    import torch
    g = torch.Generator(device="cuda").manual_seed(seed)
    F = (torch.rand(n, lda, generator=g, device="cuda") - 0.5) / n      # F[col, row]
    F[:, :n].diagonal().copy_(2.0 + torch.rand(n, generator=g, device="cuda"))
    return F, g


def _tri(F, n):
    import torch
    M = F[:, :n].t().double()
    return M.tril(-1) + torch.eye(n, device="cuda", dtype=torch.float64), M.triu()


@pytest.mark.parametrize("n", [1, 15, 17, 255, 257, 511, 512, 513, 769, 1025, 2600])
@pytest.mark.parametrize("nrhs,pad", [(1, 0), (16, 1), (17, 0), (33, 3), (65, 0)])
@pytest.mark.parametrize("trans", [False, True])
def test_lu_solve_tiles(ctx, n, nrhs, pad, trans):
    import torch
    F, g = _factor(n, n + pad, n)
    X = torch.rand(nrhs, n + 2 * pad, generator=g, device="cuda", dtype=torch.float64) - 0.5
    X0 = X.clone()
    ctx.lu_solve(n, nrhs, min(n, 512), F, n + pad, X, n + 2 * pad, trans=trans)
    L, U = _tri(F, n)
    A = (L @ U).t() if trans else L @ U
    ref = torch.linalg.solve(A, X0[:, :n].t())
    assert torch.equal(X[:, n:], X0[:, n:])
    assert ((X[:, :n].t() - ref).abs().max() / ref.abs().max()).item() < 1e-12


@pytest.mark.parametrize("n,nrhs,trans", [(600, 1025, False), (600, 1090, True), (16500, 2, False), (16500, 1, True)])
def test_lu_solve_past_one_pass(ctx, n, nrhs, trans):
    """More columns than one pass takes; more blocks than are inverted at a time."""
    import torch
    F, g = _factor(n, n, 3)
    X = torch.rand(nrhs, n, generator=g, device="cuda", dtype=torch.float64) - 0.5
    B = X.t().clone()
    ctx.lu_solve(n, nrhs, 512, F, n, X, n, trans=trans)
    L, U = _tri(F, n)
    # A x against b: the factors are within a few units of the identity
    R = U.t() @ (L.t() @ X.t()) if trans else L @ (U @ X.t())
    assert ((R - B).abs().max() / B.abs().max()).item() < 1e-12


@pytest.mark.parametrize("bad", [np.nan, np.inf])
def test_rows_before_a_nonfinite_entry_stay(ctx, bad):
    """Row 300 of one column: L^-1 leaves the rows before it and the other
    columns alone, U^-1 the rows after it."""
    import torch
    n, i = 700, 300
    F, g = _factor(n, n, 9)
    X = torch.rand(n, generator=g, device="cuda", dtype=torch.float64)
    good = X.clone()
    X[i] = bad
    for solve, keep, gone in ((ctx.trsv_lower, slice(0, i), slice(i, n)), (ctx.trsv_upper, slice(i + 1, n), slice(0, i + 1))):
        x, y = X.clone(), good.clone()
        solve(n, 512, F, n, x)
        solve(n, 512, F, n, y)
        assert ((x[keep] - y[keep]).abs().max() / y.abs().max()).item() < 1e-12
        assert not torch.isfinite(x[gone]).any()


def test_captured_and_replayed(ctx):
    import torch
    n, nrhs = 1300, 5
    F, g = _factor(n, n, 4)
    X = torch.zeros(nrhs, n, device="cuda", dtype=torch.float64)
    B = torch.rand(3, nrhs, n, generator=g, device="cuda", dtype=torch.float64)
    want = B.clone()
    for k in range(3):
        ctx.lu_solve(n, nrhs, 512, F, n, want[k], n)
        ctx.trsv_lower(n, 512, F, n, want[k, 1])
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        ctx.lu_solve(n, nrhs, 512, F, n, X, n)
        ctx.trsv_lower(n, 512, F, n, X[1])
    for k in range(3):
        X.copy_(B[k])
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(X, want[k])


def _hard(n, kind, rng):
    """Triangles far from the identity: T (lower, unit) in FP32 values."""
    T = np.tril(rng.standard_normal((n, n)) * 0.3, -1) if kind == "normal" else np.tril(np.full((n, n), -0.02), -1)
    if kind == "first":
        T = np.tril(rng.uniform(-0.5, 0.5, (n, n)) / n, -1)
        T[:400, :400] = np.tril(rng.standard_normal((400, 400)) * 0.3, -1)
    return (T + np.eye(n)).astype(np.float32).astype(np.float64)


@pytest.mark.parametrize("n", [120, 512, 900, 1600])
@pytest.mark.parametrize("kind", ["normal", "constant", "first"])
@pytest.mark.parametrize("upper,trans", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("nrhs", [1, 18])
def test_ill_conditioned_triangles(ctx, n, kind, upper, trans, nrhs):
    """Blocks whose inverse would cost accuracy.  Substitution in any order has
    |b - T x| <= gamma |T| |x| entry by entry with gamma = (n + 2) u / (1 - (n +
    2) u), u = 2^-53 (one more rounding for the reciprocal diagonal); b = T x0
    with a small x0, the right-hand side for which a product with the inverse is
    1e3 and more above that."""
    import torch
    if kind == "first" and n < 400:
        pytest.skip("smaller than its hard block")
    rng = np.random.default_rng(n)
    T = _hard(n, kind, rng)
    if upper:
        T = np.ascontiguousarray(T[::-1, ::-1])          # unit upper
        T = (T * rng.uniform(0.5, 2.0, n)[:, None]).astype(np.float32).astype(np.float64)
    M = T + 0.0
    opT = T.T if trans else T
    X0 = rng.standard_normal((n, nrhs))
    B = (opT.astype(np.longdouble) @ X0.astype(np.longdouble)).astype(np.float64)
    # the other triangle is the identity's: L = I has no stored diagonal, U = I does
    LU = np.triu(M) if upper else np.tril(M, -1) + np.eye(n)
    F = torch.from_numpy(np.ascontiguousarray(LU.T.astype(np.float32))).cuda()
    Xc = torch.from_numpy(np.ascontiguousarray(B.T)).cuda()
    if nrhs == 1 and not trans:
        (ctx.trsv_upper if upper else ctx.trsv_lower)(n, 512, F, n, Xc)
    else:
        ctx.lu_solve(n, nrhs, 512, F, n, Xc, n, trans=trans)
    X = Xc.cpu().numpy().T.astype(np.longdouble)
    R = np.abs(B.astype(np.longdouble) - opT.astype(np.longdouble) @ X)
    u = 2.0 ** -53
    gamma = (n + 2) * u / (1 - (n + 2) * u)
    assert np.isfinite(X).all()
    assert (R <= gamma * (np.abs(opT) @ np.abs(X))).all(), float((R / (np.abs(opT) @ np.abs(X))).max() / gamma)
