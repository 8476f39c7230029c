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
