"""Plain FP16 panels converted by the TRSMs that form them against the separate
conversion, which a profiled run keeps: the same bits, for panels past and below
the 16-wide strips, blocks that are no multiple of 32 and the packed layout."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,b,outer", [(1200, 60, 1), (1000, 100, 2), (1285, 257, 1), (999, 333, 1), (2048, 256, 2),
                                       (6144, 512, 2), (6400, 128, 4), (4800, 48, 1)])
def test_profiled_and_plain_runs_agree(ctx, n, b, outer):
    out = []
    for profile in (False, True):
        r = ctx.solve(n, b, fmt="f16", outer=outer, seed=5, profile=profile, keep_factors=True)
        assert r["converged"]
        out.append((r["residual"], ctx.solution_x(n), ctx.solution_factors(n)))
    assert out[0][0] == out[1][0]
    assert np.array_equal(out[0][1], out[1][1]) and np.array_equal(out[0][2], out[1][2])
