"""Overlapping the trailing update with the next panel only while the update is
long enough: the schedules differ, the factors must not.  7168 overlaps its
first steps only, 1536 none; with one inner block the rows below stay on the
panel's stream, with two they have their own."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,b,outer", [(7168, 512, 1), (7168, 512, 2), (7168, 256, 3), (1536, 128, 1), (1536, 128, 4)])
@pytest.mark.parametrize("fmt", ["f16", "e4m3"])
def test_factors_do_not_depend_on_the_overlap(ctx, n, b, outer, fmt):
    import torch
    g = torch.Generator(device="cuda").manual_seed(n + b)
    A = torch.rand(n, n, generator=g, device="cuda") - 0.5
    A.diagonal().copy_(n / 4 + 1 + torch.rand(n, generator=g, device="cuda"))
    out = []
    for lookahead in (False, True, 2):
        F = A.clone()
        ctx.factor(n, b, F, n, fmt=fmt, outer=outer, lookahead=lookahead)
        out.append(F)
    assert torch.isfinite(out[0]).all()
    assert torch.equal(out[0], out[1]) and torch.equal(out[0], out[2])
