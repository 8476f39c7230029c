"""The diagonal sums and the matrix-free residual at the edges of their tiling:
fewer columns than a chunk, one more than a chunk, row ranges that start and
end inside a workgroup's rows, the smallest orders.  The diagonal is bit-exact
against the oracle (FP64, j ascending); the residual is within the 1e-13 of
the existing GEMV test (FP64 sums in another order)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
SEED = 42


@pytest.mark.parametrize("n,i0,cnt", [(1, 0, 1), (2, 0, 2), (55, 3, 40), (57, 0, 57), (64, 63, 1), (113, 0, 113),
                                      (1000, 900, 100), (4097, 65, 130)])
def test_gen_diag_ranges(ctx, oracle, n, i0, cnt):
    import torch
    d = torch.full((cnt + 1,), 7.0, dtype=torch.float64, device="cuda")
    ctx.gen_diag(n, SEED, i0, cnt, d)
    got = d.cpu().numpy()
    assert np.array_equal(got[:cnt].view(np.uint64), oracle.gen_diag(n, SEED)[i0:i0 + cnt].view(np.uint64))
    assert got[cnt] == 7.0


@pytest.mark.parametrize("n", [1, 7, 63, 65, 257, 300, 2049, 4500])
def test_otf_gemv_edges(ctx, oracle, n):
    import torch
    rng = np.random.default_rng(n)
    d = oracle.gen_diag(n, SEED)
    x, y = rng.standard_normal(n), rng.standard_normal(n)
    gy = torch.from_numpy(y.copy()).cuda()
    ctx.otf_gemv(n, SEED, torch.from_numpy(d).cuda(), -1.0, torch.from_numpy(x).cuda(), gy)
    ref = oracle.otf_gemv(n, d, -1.0, x, y, SEED)
    scale = np.max(np.abs(y)) + np.max(np.abs(d)) * 2 * np.max(np.abs(x))
    assert np.max(np.abs(gy.cpu().numpy() - ref)) / scale < 1e-13


@pytest.mark.parametrize("n,i0,j0,m,k", [(1, 0, 0, 1, 1), (300, 0, 0, 300, 300), (700, 250, 200, 13, 71),
                                         (700, 0, 255, 257, 65), (700, 256, 64, 256, 64), (2000, 1999, 0, 1, 2000),
                                         (2000, 0, 1999, 2000, 1), (900, 100, 107, 600, 9)])
@pytest.mark.parametrize("diag", [False, True])
def test_gen_matrix_blocks(ctx, oracle, n, i0, j0, m, k, diag):
    """Bit-exact blocks at the edges of 256 rows, 64 columns and groups of 8,
    with and without the diagonal, nothing written outside."""
    import torch
    d = oracle.gen_diag(n, SEED)
    A = torch.full((k + 1, m + 3), 7.0, device="cuda")
    ctx.gen_matrix(n, SEED, i0, j0, m, k, torch.from_numpy(d).cuda() if diag else None, A, m + 3)
    got = A.cpu().numpy()
    want = oracle.gen_block(n, i0, j0, m, k, SEED)           # [col, row], diagonal entries d
    if not diag:
        for c in range(k):
            r = j0 + c - i0
            if 0 <= r < m:
                want[c, r] = got[c, r]
                assert abs(got[c, r]) <= 0.5
    assert np.array_equal(got[:k, :m].view(np.uint32), want.view(np.uint32))
    assert (got[k:] == 7.0).all() and (got[:, m:] == 7.0).all()
