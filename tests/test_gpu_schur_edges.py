"""Schur update of a C that is no whole number of tiles: one row, one column
and the neighbours of 32, 64 and 128, an odd leading dimension, nothing written
outside.  K = 64 products of FP16 values below 1/2, so every sum of magnitudes
is at most 16 and 64 FP32 roundings differ from the exact sum by at most
64 * 16 * 2^-24 = 6.2e-5."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [1, 31, 63, 64, 65, 129])
@pytest.mark.parametrize("n", [1, 31, 33, 64, 127, 130])
def test_schur_f16_edges(ctx, m, n):
    import torch
    rng = np.random.default_rng(m * 1000 + n)
    L = (rng.random((m, 64)) - 0.5).astype(np.float16)
    U = (rng.random((n, 64)) - 0.5).astype(np.float16)
    C = rng.random((n + 2, m + 5)).astype(np.float32)          # C[col, row]
    g = torch.from_numpy(C).cuda()
    ctx.schur_update(0, m, n, 1, 64, torch.from_numpy(L).cuda(), 64, None, 0, torch.from_numpy(U).cuda(), 64, None, 0,
                     0, g[1, 2:], m + 5)
    got = g.cpu().numpy()
    want = C.astype(np.float64)
    want[1:n + 1, 2:m + 2] -= U.astype(np.float64) @ L.astype(np.float64).T
    assert np.max(np.abs(got - want)) < 6.2e-5
    inside = np.zeros(C.shape, dtype=bool)
    inside[1:n + 1, 2:m + 2] = True
    assert np.array_equal(got[~inside], C[~inside])


@pytest.mark.parametrize("fmt", [0, 2])
@pytest.mark.parametrize("m,n", [(8192, 1024), (8391, 1000), (8448, 1024), (16384, 1024), (16640, 1024)])
def test_schur_tile_choice(ctx, fmt, m, n):
    """128, 132 and 256, 260 tiles of 256 x 256: the edges of the range below two
    tiles per CU that the larger tile takes, with ragged edges, K of 2 KB.  An
    FP32 sum of K products in any order is within K 2^-24 of the sum of their
    magnitudes."""
    import torch
    K = 1024 if fmt == 0 else 2048
    g = torch.Generator(device="cuda").manual_seed(m + n)
    dt = torch.float16 if fmt == 0 else torch.float8_e4m3fn
    L = (torch.rand(m, K, generator=g, device="cuda") - 0.5).to(dt)
    U = (torch.rand(n, K, generator=g, device="cuda") - 0.5).to(dt)
    ns = K // 512
    eL = torch.zeros(ns, (m + 511) // 512, dtype=torch.int32, device="cuda")
    eU = torch.zeros(ns, (n + 511) // 512, dtype=torch.int32, device="cuda")
    C = torch.rand(n, m, generator=g, device="cuda")
    C0 = C.clone()
    ctx.schur_update(fmt, m, n, ns, 512, L, K, eL, eL.shape[1], U, K, eU, eU.shape[1], 512, C, m)
    Ld, Ud = L.double(), U.double()
    want = C0.double() - Ud @ Ld.t()
    bound = (Ud.abs() @ Ld.abs().t() + C0.double()) * (K * 2.0 ** -24)
    assert ((C.double() - want).abs() <= bound).all()


@pytest.mark.parametrize("fmt,pad", [(0, 0), (2, 0), (2, 128)])
def test_schur_packed_first(ctx, fmt, pad):
    """A row-layout update large enough to be packed first, ragged in rows,
    columns and leading dimension, against the same update as two row blocks,
    which are not: the same sums in the same order, so the same bits."""
    import torch
    m, n, K, cut = 22311, 21903, 1024 if fmt == 0 else 2048, 11264
    g = torch.Generator(device="cuda").manual_seed(7)
    dt = torch.float16 if fmt == 0 else torch.float8_e4m3fn
    L = (torch.rand(m, K + pad, generator=g, device="cuda") - 0.5).to(dt)
    U = (torch.rand(n, K + pad, generator=g, device="cuda") - 0.5).to(dt)
    ns, tl, tu = K // 512, (m + 511) // 512, (n + 511) // 512
    eL = torch.randint(-2, 3, (ns, tl), generator=g, device="cuda", dtype=torch.int32)
    eU = torch.randint(-2, 3, (ns, tu), generator=g, device="cuda", dtype=torch.int32)
    C = torch.rand(n, m, generator=g, device="cuda")
    D = C.clone()
    ctx.schur_update(fmt, m, n, ns, 512, L, K + pad, eL, tl, U, K + pad, eU, tu, 512, C, m)
    for r0, r1 in ((0, cut), (cut, m)):
        ctx.schur_update(fmt, r1 - r0, n, ns, 512, L[r0:], K + pad, eL[0, r0 // 512:], tl, U, K + pad, eU, tu, 512,
                         D[0, r0:], m)
    assert torch.equal(C, D)


def test_gemmschur_of_more_entries_than_one_launch_takes(ctx):
    """B of (2^18 + 3) x 2^14 entries, staged by a thread each: past 2^32."""
    import torch
    n, m, k = 3, (1 << 18) + 3, 1 << 14
    a = torch.ones(k, n, dtype=torch.float16, device="cuda")
    b = torch.zeros(m, k, dtype=torch.float16, device="cuda")
    b[:, 0], b[:, -1] = 1.0, 0.5                       # two entries a column: exact
    b[-1, 7] = 3.0
    c = torch.full((m, n), 2.0, device="cuda")
    ctx.gemmschur_f16(n, m, k, a, n, b, k, c, n)
    assert bool((c[:-1] == 0.5).all()) and bool((c[-1] == -2.5).all())
