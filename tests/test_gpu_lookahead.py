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


@pytest.mark.parametrize("n,b,outer", [(7200, 60, 1), (7200, 60, 4), (7200, 100, 1), (7200, 100, 4)])
def test_padded_slices_under_the_overlap(ctx, n, b, outer):
    """b = 60 and 100 fill 60 of 64 and 100 of 128 values of a slice: the TRSMs
    write the FP16 copies of the next panel, zeros up to whole 32-blocks, into the
    other buffer while the update reads this one."""
    test_factors_do_not_depend_on_the_overlap(ctx, n, b, outer, "f16")


@pytest.mark.parametrize("n,b,outer,split,trail16", [(7200, 60, 8, 3, 0), (7200, 100, 4, 0, 0), (7680, 128, 8, 3, 1),
                                                     (7680, 256, 4, 2, 2)])
def test_lazy_split_solves_under_the_overlap(ctx, n, b, outer, split, trail16):
    """Lazy initialisation, the two-part panel and the FP16 partial sums, whose
    streams meet only where the update is long enough to be overlapped: the
    first steps here."""
    import numpy as np
    out = []
    for lookahead in (0, 1, 2):
        r = ctx.solve(n, b, fmt="f16", outer=outer, lookahead=lookahead, lazy=True, split=split, trail16=trail16,
                      keep_factors=True)
        assert r["converged"]
        out.append((ctx.solution_factors(n), ctx.solution_x(n)))
        ctx.release()
    for F, x in out[1:]:
        assert np.array_equal(F.view(np.uint32), out[0][0].view(np.uint32))
        assert np.array_equal(x, out[0][1])
