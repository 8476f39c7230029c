"""The batched LU at the edges of its 32-column blocks, of the 15 waves that
share a block column's tiles and of the two-panel groups of width 64: every
width converges, and the widths' solutions agree.

A harness below 16 bounds |b - A x| by 16 n 2^-53 (|A| |x| + |b|), so two such
solutions differ by at most 64 n 2^-53 cond(A) |x|: 4.3e-11 |x|, n cond(A) being
below 6000 for all of these.  (Order 2 is left out: its diagonal makes it
singular whenever the two other entries have one sign.)"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes", [range(3, 36), (63, 65, 95, 96, 97, 159, 161), (479, 480, 481, 511, 513, 543, 545),
                                   (575, 577, 991, 993, 1024)])
def test_batch_widths_agree(ctx, sizes):
    import hplai
    n = np.array(list(sizes), dtype=np.int32)
    nrhs = np.array([i % 4 + 1 for i in range(n.size)], dtype=np.int32)
    seeds = np.arange(n.size, dtype=np.uint64) * 11 + 3
    out = []
    for nb in (16, 32, 64):
        bt = hplai.Batch(ctx, n, nrhs, seeds)
        bt.set_nb((nb,) * 4)
        st = bt.run("persistent")
        assert st["failed"] == 0
        out.append([bt.solution(s).copy() for s in range(n.size)])
        bt.close()
    for a, b, c in zip(*out):
        assert np.array_equal(a, b)
        assert np.max(np.abs(b - c)) / np.max(np.abs(b)) < 1e-10
