"""Tile exponents of hplai_quantize at the shapes where the tile scan can go
wrong: float4 and scalar columns, ragged last tiles, tiles split over several
workgroups, tiles narrower than a wave, a tile of zeros.  Bit-exact against
the oracle's exponent rule and conversions."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,k,tb,pad", [(300, 64, 128, 0),      # float4 scan, ragged last tile
                                        (301, 67, 128, 1),      # scalar scan, odd everything
                                        (1030, 1040, 512, 2),   # tiles past one workgroup's share
                                        (70, 2500, 512, 0),     # one short tile
                                        (45, 33, 7, 0), (5, 1, 1, 3)])
@pytest.mark.parametrize("side", [0, 1])
@pytest.mark.parametrize("fmt", ["e4m3", "f16t"])
def test_tile_exponents(ctx, oracle, m, k, tb, pad, side, fmt):
    import hplai
    import torch
    rng = np.random.default_rng(m * 1000 + k)
    nt = -(-m // tb)
    rows = (rng.standard_normal((m, k)) * 10.0 ** rng.integers(-6, 4, size=nt)[np.arange(m) // tb][:, None]).astype(
        np.float32)
    if nt > 1:
        rows[tb:2 * tb] = 0.0
    X = rows.T if side == 0 else rows                     # [column][entry]
    src = np.full((X.shape[0], X.shape[1] + pad), 1e30, dtype=np.float32)   # padding must not be read into a tile
    src[:, :X.shape[1]] = X
    es = 1 if fmt == "e4m3" else 2
    dst = torch.zeros(m * k * es, dtype=torch.uint8, device="cuda")
    exps = torch.full((nt,), 99, dtype=torch.int32, device="cuda")
    ctx.quantize(hplai.FMTS[fmt], side, m, k, tb, torch.from_numpy(src).cuda(), src.shape[1], dst, k, exps)
    e = np.array([oracle.tile_exp(2 if fmt == "e4m3" else 1, np.max(np.abs(rows[t * tb:(t + 1) * tb])))
                  for t in range(nt)])
    assert np.array_equal(exps.cpu().numpy(), e.astype(np.int32))
    scaled = np.ldexp(rows, e[np.arange(m) // tb][:, None]).astype(np.float32)
    got = dst.cpu().numpy()
    if fmt == "e4m3":
        assert np.array_equal(got.reshape(m, k), oracle.f32_to_e4m3_bits(scaled))
    else:
        assert np.array_equal(got.view(np.uint16).reshape(m, k), oracle.f32_to_f16_bits(scaled))


@pytest.mark.parametrize("m,k,tb,pad", [(300, 70, 1, 0), (301, 33, 3, 1), (64, 64, 15, 0), (1000, 600, 5, 2),
                                        (1, 1, 1, 0), (200, 17, 16, 0)])
@pytest.mark.parametrize("side", [0, 1])
@pytest.mark.parametrize("fmt", ["e4m3", "f16t"])
def test_short_tiles(ctx, oracle, m, k, tb, pad, side, fmt):
    """Tiles of a few lines, several of them in a workgroup's 64."""
    test_tile_exponents(ctx, oracle, m, k, tb, pad, side, fmt)


@pytest.mark.parametrize("tb", [1, 16])
@pytest.mark.parametrize("side", [0, 1])
def test_more_tiles_than_one_launch_takes(ctx, oracle, tb, side):
    import hplai
    import torch
    tiles, k = (1 << 22) + 5, 1
    m = tiles * tb
    values = (2.0 ** np.arange(-20, 12)).astype(np.float32) * np.float32(1.37)
    want = np.array([oracle.tile_exp(2, v) for v in values], dtype=np.int32)
    pick = torch.randint(0, len(values), (tiles,), generator=torch.Generator().manual_seed(1))
    # one line of a tile holds its maximum
    src = torch.zeros(m, device="cuda")
    src[torch.arange(tiles, device="cuda") * tb + tb // 2] = torch.from_numpy(values).cuda()[pick.cuda()]
    dst = torch.zeros(m, dtype=torch.uint8, device="cuda")
    exps = torch.full((tiles,), 99, dtype=torch.int32, device="cuda")
    ctx.quantize(hplai.FMT_E4M3, side, m, k, tb, src, m if side == 0 else k, dst, k, exps)
    assert np.array_equal(exps.cpu().numpy(), want[pick.numpy()])
    q = oracle.f32_to_e4m3_bits(np.ldexp(values, want).astype(np.float32))
    got = dst.cpu().numpy().reshape(tiles, tb)
    assert np.array_equal(got[:, tb // 2], q[pick.numpy()])
    assert (np.delete(got, tb // 2, axis=1) == 0).all()


@pytest.mark.parametrize("side", [0, 1])
def test_more_entries_than_threads_of_one_launch(ctx, side):
    """Side 0: 2^30 + 70 rows (64 of them a workgroup); side 1: 2^32 + 70 columns
    of one entry (a thread each)."""
    import hplai
    import torch
    m = (1 << 30) + 70 if side == 0 else (1 << 32) + 70
    src = torch.full((m,), 1.5, device="cuda")
    src[-1] = -2.0
    dst = torch.zeros(m, dtype=torch.float16, device="cuda")
    ctx.quantize(hplai.FMT_F16, side, m, 1, 1, src, m if side == 0 else 1, dst, 1)
    assert torch.equal(dst[:-1].min(), dst[:-1].max()) and dst[0].item() == 1.5 and dst[-1].item() == -2.0
