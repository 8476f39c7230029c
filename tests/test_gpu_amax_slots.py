"""Tile exponents of hplai_quantize where a tile is scanned in four parts: the
largest entry in each part in turn, fewer columns than parts, ragged last
tiles, the smallest and largest tile of that range and the next one.
Bit-exact against the oracle's exponent rule and conversions."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,k,tb,pad", [(2560, 512, 512, 0),       # the smallest tile in parts
                                        (1541, 521, 512, 3),       # scalar scan, a last tile of 5
                                        (90000, 3, 90000, 0),      # side 0: three columns, an empty part
                                        (3, 90000, 7, 0),          # side 1 of the same
                                        (2100, 2048, 1024, 0),     # the largest tile with a slot a part
                                        (2100, 2049, 1024, 0)])    # its parts meet
@pytest.mark.parametrize("side", [0, 1])
@pytest.mark.parametrize("fmt", ["e4m3", "f16t"])
def test_tile_parts(ctx, oracle, m, k, tb, pad, side, fmt):
    import hplai
    import torch
    rng = np.random.default_rng(m + k)
    nt = -(-m // tb)
    rows = rng.uniform(-1.0, 1.0, size=(m, k)).astype(np.float32)
    for t in range(nt):                                   # the largest entry: in part t % 4
        h = min(tb, m - t * tb)
        span = k if side == 0 else h
        q = min(span - 1, (t % 4) * span // 4 + span // 8)
        if side == 0:
            rows[t * tb + h // 2, q] = 3.0 * 2.0 ** t
        else:
            rows[t * tb + q, k // 2] = 3.0 * 2.0 ** t
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
