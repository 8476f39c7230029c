"""The passes over a dense FP64 matrix: the transposed FP32 copy (each entry the
rounding of one number, so exact) and the infinity norms, at the edges of the 64
x 64 tiles, of the 512-column and 128-row chunks, with a leading dimension.  A
sum of n terms in any order is within n 2^-53 of the exact one."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 127, 129, 511, 513, 1200, 2049])
@pytest.mark.parametrize("pad", [0, 3])
def test_copy_and_norms(ctx, n, pad):
    import torch
    g = torch.Generator(device="cuda").manual_seed(n)
    A = torch.randn(n, n + pad, generator=g, device="cuda", dtype=torch.float64)
    A[:, n:] = float("nan")                                   # never read
    V = A[:, :n]
    F = torch.full((n, n + pad), 7.0, device="cuda")
    ctx.narrow_transpose(n, A, n + pad, F, n + pad)
    assert torch.equal(F[:, :n], V.t().float()) and (F[:, n:] == 7.0).all()
    out = torch.empty((), dtype=torch.float64, device="cuda")
    for trans in (False, True):
        ctx.norm_abs(n, A, n + pad, out, trans=trans)
        want = V.abs().sum(0 if trans else 1).max()
        assert abs((out - want).item()) <= 2 * n * 2.0 ** -53 * want.item()
        B = A.clone()
        B[n // 2, n - 1] = float("nan")
        ctx.norm_abs(n, B, n + pad, out, trans=trans)
        assert torch.isnan(out)
