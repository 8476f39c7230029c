"""Diagonal-block LU (128-column sub-blocks on several workgroups) and the
panel TRSMs at the sizes where its tiling can go wrong: one row, the edges of
the 32 x 32 steps and of the 128-column sub-blocks, orders that are no
multiple of either, the largest, and a leading dimension that leaves the
columns unaligned.  Against the oracle with the relative 2e-5 of the existing
getrf and TRSM tests (FP32 with another order of the sums)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
SEED = 42


def _dev(a):
    import torch
    return torch.from_numpy(a).cuda()


def _factored(oracle, b, n):
    D = oracle.gen_block(n, 0, 0, b, b, SEED)
    ref = D.copy()
    oracle.lib().orc_getrf_nopiv_f32(b, oracle._ptr(ref), b)
    return D, ref


@pytest.mark.parametrize("b", [1, 31, 33, 97, 127, 129, 160, 257, 384, 500, 513, 777, 1000])
@pytest.mark.parametrize("pad", [0, 3])
def test_getrf_tiles(ctx, oracle, b, pad):
    import torch
    D, ref = _factored(oracle, b, 4 * b + 4)
    buf = np.full((b, b + pad), 7.0, dtype=np.float32)      # buf[col, row]
    buf[:, :b] = D
    g = _dev(buf)
    info = torch.full((1,), 5, dtype=torch.int32, device="cuda")
    ctx.getrf(b, g, b + pad, info)
    got = g.cpu().numpy()
    assert int(info.cpu()[0]) == 0
    assert np.all(got[:, b:] == 7.0)
    assert np.max(np.abs(got[:, :b] - ref)) / np.max(np.abs(ref)) < 2e-5


@pytest.mark.parametrize("b,z", [(96, 95), (300, 0), (300, 130), (512, 511), (1000, 900)])
@pytest.mark.parametrize("bad", [0.0, np.inf])
def test_getrf_first_bad_pivot_of_any_sub_block(ctx, b, z, bad):
    import torch
    A = np.eye(b, dtype=np.float32)
    A[z, z] = bad
    if z + 40 < b:
        A[z + 40, z + 40] = 0.0                              # a later one is not reported
    info = torch.zeros(1, dtype=torch.int32, device="cuda")
    ctx.getrf(b, _dev(A), b, info)
    assert int(info.cpu()[0]) == z + 1


@pytest.mark.parametrize("scale", [2.0 ** 104, 2.0 ** -109])
def test_getrf_pivots_past_the_fast_reciprocal(ctx, oracle, scale):
    """A scaled by a power of two s: L stays, U scales with it.  Pivots are
    about 2^7 s, so both s leave the range of the Newton reciprocal
    (2^-100 .. 2^100), while every quantity formed on the way stays a normal
    FP32 number: the smallest inverse entry about 2^-15 / s, the smallest
    update term 2^-10 s.  The runs differ in how each pivot's reciprocal is
    rounded, one FP32 ulp (1.2e-7) of every l and of the updates built on it:
    2e-6 allows sixteen of them."""
    b = 160
    D, _ = _factored(oracle, b, 4 * b)
    g, s = _dev(D), _dev((D * np.float32(scale)).astype(np.float32))
    ctx.getrf(b, g, b)
    ctx.getrf(b, s, b)
    ref, got = g.cpu().numpy(), s.cpu().numpy()
    lower = np.tril(np.ones((b, b), dtype=bool), -1).T       # [col, row] with row > col
    want = np.where(lower, ref, ref * np.float32(scale))
    assert np.max(np.abs(got - want)[lower]) / np.max(np.abs(want[lower])) < 2e-6
    assert np.max(np.abs(got - want)[~lower]) / np.max(np.abs(want[~lower])) < 2e-6


@pytest.mark.parametrize("b", [1, 33, 100, 257, 513, 777, 1000, 1024])
@pytest.mark.parametrize("m", [1, 45])
def test_trsm_tiles(ctx, oracle, b, m):
    n = m + b
    _, ref = _factored(oracle, b, n + 4)
    L = oracle.gen_block(n + 4, b, 0, m, b, SEED)
    U = oracle.gen_block(n + 4, 0, b, b, m, SEED)
    gF, gL, gU = _dev(ref), _dev(L), _dev(U)
    ctx.trsm_lpanel(m, b, gF, b, gL, m)
    ctx.trsm_upanel(b, m, gF, b, gU, b)
    oracle.lib().orc_trsm_runn_f32(m, b, oracle._ptr(ref), b, oracle._ptr(L), m)
    oracle.lib().orc_trsm_llnu_f32(b, m, oracle._ptr(ref), b, oracle._ptr(U), b)
    assert np.max(np.abs(gL.cpu().numpy() - L)) / np.max(np.abs(L)) < 2e-5
    assert np.max(np.abs(gU.cpu().numpy() - U)) / np.max(np.abs(U)) < 2e-5


def test_getrf_captured(ctx, oracle):
    """Captured on the caller's stream and replayed, with eager work between."""
    import torch
    b = 320
    D, _ = _factored(oracle, b, 4 * b)
    src = _dev(D)
    want = src.clone()
    ctx.getrf(b, want, b)
    buf = torch.empty_like(src)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        buf.copy_(src)
        ctx.getrf(b, buf, b)
    for _ in range(3):
        buf.fill_(3.0)
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(buf, want)


@pytest.mark.parametrize("b", [160, 257, 384, 500, 650, 1000])
def test_inverses_grown_with_the_factorization(ctx, oracle, b):
    """Two diagonal blocks: the panels beside the first are products with the
    inverses that grow by a 128-column sub-block at a time.  L21 U11 = A21 and
    L11 U12 = A12 in FP64, within the 2e-5 of the TRSM tests."""
    import torch
    n = 2 * b
    A = oracle.gen_block(2 * n, 0, 0, n, n, SEED)             # A[col, row]
    F = _dev(A)
    ctx.factor(n, b, F, n, fmt="f16")
    A, F = torch.from_numpy(A).t().double(), F.cpu().t().double()
    L = F[:b, :b].tril(-1) + torch.eye(b, dtype=torch.float64)
    U = F[:b, :b].triu()
    for got, want in ((F[b:, :b] @ U, A[b:, :b]), (L @ F[:b, b:], A[:b, b:])):
        assert ((got - want).abs().max() / want.abs().max()).item() < 2e-5


@pytest.mark.parametrize("b", [1, 31, 60, 128, 200, 512])
@pytest.mark.parametrize("m", [1, 15, 17, 4096, 4097])
def test_trsm_strip_widths(ctx, oracle, b, m):
    """16-wide strips up to 4096, 32-wide ones past it, unaligned panels;
    L U11 = A21 and L11 U = A12 in FP64, within the 2e-5 above."""
    import torch
    D, ref = _factored(oracle, b, 4 * b + 4)
    F = _dev(ref)                                             # F[col, row]
    g = torch.Generator(device="cuda").manual_seed(m)
    L = torch.rand(b, m + 1, generator=g, device="cuda") - 0.5
    U = torch.rand(m, b + 1, generator=g, device="cuda") - 0.5
    L0, U0 = L.clone(), U.clone()
    ctx.trsm_lpanel(m, b, F, b, L, m + 1)
    ctx.trsm_upanel(b, m, F, b, U, b + 1)
    assert torch.equal(L[:, m:], L0[:, m:]) and torch.equal(U[:, b:], U0[:, b:])
    T = F.t().double()
    low = T.tril(-1) + torch.eye(b, device="cuda", dtype=torch.float64)
    for got, want in ((L[:, :m].t().double() @ T.triu(), L0[:, :m].t().double()),
                      (low @ U[:, :b].t().double(), U0[:, :b].t().double())):
        assert ((got - want).abs().max() / want.abs().max()).item() < 2e-5


@pytest.mark.parametrize("b", [60, 128, 512])
def test_narrow_strips_add_the_diagonal_last(ctx, oracle, b):
    """U12 of a diagonally dominant block is A12 minus sums of small products:
    one rounding of the large term (rms 2^-25 of it) when the unit diagonal's
    term is the last one added, and two or more otherwise.  Both strip widths
    on the same columns, each within 1.5 of that one rounding."""
    import torch
    D, ref = _factored(oracle, b, 4 * b + 4)
    F = _dev(ref)
    g = torch.Generator(device="cuda").manual_seed(b)
    wide = torch.rand(6000, b, generator=g, device="cuda") - 0.5      # U[col, row]
    narrow = wide[:2000].clone()
    low = F.t().double().tril(-1) + torch.eye(b, device="cuda", dtype=torch.float64)
    want = torch.linalg.solve_triangular(low, wide.t().double(), upper=False, unitriangular=True).t()
    ctx.trsm_upanel(b, 6000, F, b, wide, b)
    ctx.trsm_upanel(b, 2000, F, b, narrow, b)
    for got, w in ((wide, want), (narrow, want[:2000])):
        assert ((got.double() - w).norm() / w.norm()).item() < 1.5 * 2.0 ** -25


def _hard_triangle(b, rng):
    """Unit lower, 32 x 32 diagonal blocks near the identity, condition 1e6 and more as a whole."""
    T = rng.standard_normal((b, b)) * (0.2 if b > 500 else 1.0)
    for i in range(0, b, 32):
        T[i:i + 32, i:i + 32] = rng.uniform(-0.5, 0.5, T[i:i + 32, i:i + 32].shape) / 32
    return (np.tril(T, -1) + np.eye(b)).astype(np.float32)


@pytest.mark.parametrize("b", [60, 100, 257, 500, 513, 640, 777, 1000, 1024])
@pytest.mark.parametrize("m,pad", [(1, 0), (33, 1), (700, 4)])
def test_trsm_ill_conditioned(ctx, b, m, pad):
    """The entrywise bound of substitution in 32-blocks: |B - T X| <= g |T| |X|
    with g = 2 (b + 64) u, u = 2^-24.  b + 32 roundings of the products and the
    subtractions; 32 more and the factor 2 for the 32 x 32 inverses, whose
    |D^-1| |D| is below 2."""
    import torch
    rng = np.random.default_rng(b + m)
    L = _hard_triangle(b, rng)
    D = rng.uniform(0.5, 2.0, b).astype(np.float32)
    U = (np.ascontiguousarray(L.T) * D[None, :]).astype(np.float32)          # upper, columns scaled
    u = 2.0 ** -24
    X0 = rng.standard_normal((b, m))
    for up in (True, False):
        T = L.astype(np.float64) if up else U.T.astype(np.float64)           # op on a b x m panel of columns
        B = (T @ X0).astype(np.float32)
        M = L if up else U
        F = torch.from_numpy(np.ascontiguousarray(np.pad(M.T, ((0, 0), (0, pad))))).cuda()
        # U panel: column j at P[j]; L panel: row i of the panel is column i here, P[k, i]
        P = torch.from_numpy(np.ascontiguousarray(np.pad(B.T if up else B, ((0, 0), (0, pad))))).cuda()
        before = P.clone()
        if up:
            ctx.trsm_upanel(b, m, F, b + pad, P, b + pad)
            X = P.cpu().numpy()[:, :b].T.astype(np.float64)
            assert torch.equal(P[:, b:], before[:, b:])
        else:
            ctx.trsm_lpanel(m, b, F, b + pad, P, m + pad)
            X = P.cpu().numpy()[:, :m].astype(np.float64)
            assert torch.equal(P[:, m:], before[:, m:])
        R = np.abs(B.astype(np.float64) - T @ X)
        bound = 2 * (b + 64) * u * (np.abs(T) @ np.abs(X))
        assert np.isfinite(X).all()
        assert (R <= bound).all(), (up, float((R / bound).max()))


@pytest.mark.parametrize("b", [100, 600])
@pytest.mark.parametrize("bad", [np.nan, np.inf])
def test_trsm_entries_before_a_nonfinite_one_stay(ctx, b, bad):
    """Entry k of one row or column: what the triangle solves before it, and the
    other rows or columns, are not touched."""
    import torch
    rng = np.random.default_rng(b)
    m, k, j = 40, b - 45, 7
    T = torch.from_numpy((rng.uniform(-0.5, 0.5, (b, b)) / b + 2 * np.eye(b)).astype(np.float32)).cuda()
    P = torch.from_numpy(rng.uniform(-0.5, 0.5, (m, b)).astype(np.float32)).cuda()
    for up in (True, False):
        good = P.clone() if up else P.t().contiguous()
        got = good.clone()
        (got if up else got.t())[j, k] = bad
        for Q in (good, got):
            if up:
                ctx.trsm_upanel(b, m, T, b, Q, b)
            else:
                ctx.trsm_lpanel(m, b, T, b, Q, m)
        a, w = (got, good) if up else (got.t(), good.t())
        keep = torch.ones_like(w, dtype=torch.bool)
        keep[j, k:] = False
        assert not torch.isfinite(a[j, k])
        assert ((a - w)[keep].abs().max() / w.abs().max()).item() < 1e-6


def test_trsm_of_more_lines_than_one_launch_takes(ctx):
    """2^28 + 70 rows or columns of two entries: the launch would have 2^32
    threads and more."""
    import torch
    m, b = (1 << 28) + 70, 2
    T = torch.tensor([[2.0, 0.5], [0.25, 4.0]], device="cuda")        # column-major: L = [1, .5], U = [2 .25; 0 4]
    P = torch.ones(m * b, device="cuda")
    ctx.trsm_lpanel(m, b, T, b, P, m)
    # x0 = 1 / 2, x1 = (1 - .25 x0) / 4, exact in FP32
    assert bool((P[:m] == 0.5).all()) and bool((P[m:] == 0.21875).all())
    P.fill_(1.0)
    ctx.trsm_upanel(b, m, T, b, P, b)
    assert bool((P[0::2] == 1.0).all()) and bool((P[1::2] == 0.5).all())


@pytest.mark.parametrize("n,pad", [(33, 0), (60, 0), (64, 3), (128, 0), (129, 1), (200, 0), (300, 0), (512, 0), (515, 1),
                                   (777, 0), (1024, 0)])
@pytest.mark.parametrize("diag", [0.3, 1.0, 3.0])
def test_getrf_far_from_dominance(ctx, n, pad, diag):
    """Elimination has |A - L U| <= g |L| |U| entry by entry whatever the growth:
    n roundings of the sums, 64 more and the factor 2 for the 32 x 32 inverses,
    which are taken only where |D^-1| |D| is below 16 (their products add at most
    16 roundings' worth of the 32-block's own |L| |U|): g = 2 (n + 64 + 16) u."""
    import torch
    rng = np.random.default_rng(n)
    A = (rng.uniform(-0.5, 0.5, (n, n)) * (1.0 - np.eye(n)) + np.eye(n) * diag * rng.choice([-1.0, 1.0], n)).astype(np.float32)
    F = torch.from_numpy(np.ascontiguousarray(np.pad(A.T, ((0, 0), (0, pad))))).cuda()
    info = torch.full((1,), 7, dtype=torch.int32, device="cuda")
    ctx.getrf(n, F, n + pad, info)
    assert info.item() == 0
    M = F[:, :n].t().cpu().numpy().astype(np.float64)
    L, U = np.tril(M, -1) + np.eye(n), np.triu(M)
    assert np.isfinite(M).all()
    u = 2.0 ** -24
    bound = 2 * (n + 80) * u * (np.abs(L) @ np.abs(U))
    R = np.abs(A.astype(np.float64) - L @ U)
    assert (R <= bound).all(), float((R / bound).max())


@pytest.mark.parametrize("n,pad", [(129, 0), (160, 4), (256, 0), (300, 0), (512, 0), (777, 3), (1024, 0)])
@pytest.mark.parametrize("diag", [0.3, 1.0, 3.0, 6.0, 400.0])
def test_factor_of_one_block_far_from_dominance(ctx, n, pad, diag):
    """The solve's own LU of a single block, whose factors stay FP32: the bound
    above with 16 more roundings for the strips through inverses of 128 x 128
    sub-blocks, which too are taken only where |D^-1| |D| is below 16."""
    import torch
    rng = np.random.default_rng(n)
    A = (rng.uniform(-0.5, 0.5, (n, n)) * (1.0 - np.eye(n)) + np.eye(n) * diag * rng.choice([-1.0, 1.0], n)).astype(np.float32)
    F = torch.from_numpy(np.ascontiguousarray(np.pad(A.T, ((0, 0), (0, pad))))).cuda()
    ctx.factor(n, n, F, n + pad)
    M = F[:, :n].t().cpu().numpy().astype(np.float64)
    L, U = np.tril(M, -1) + np.eye(n), np.triu(M)
    assert np.isfinite(M).all()
    bound = 2 * (n + 96) * 2.0 ** -24 * (np.abs(L) @ np.abs(U))
    R = np.abs(A.astype(np.float64) - L @ U)
    assert (R <= bound).all(), float((R / bound).max())
