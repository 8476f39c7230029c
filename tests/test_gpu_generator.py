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
