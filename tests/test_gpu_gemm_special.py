"""The tiled GEMM's scale products (f32 outer products on the matrix cores) at the values where a multiplication could
differ from the vector unit's: infinite, NaN and subnormal scales.  Each output is its own row's and column's sum, so
special values stay in their row or column, and every output matches the terms f32(d_w * d_x) * dot added in f64."""

import numpy as np
import pytest
import torch

from comp_amd import _abi, host
from oracle import oracle as O
from tests.test_gpu_gemm import dev

pytestmark = pytest.mark.gpu

# (n, m): one to eight column tiles a workgroup (the scales' one product a tile, and four tiles at a time)
SHAPES = [(9000, 14), (300, 30), (12330, 24), (11000, 70), (28700, 200)]


def case(fmt, n, m, seed):
    """Planes on the device, the d_w (q4_k: and dmin) values and the exact dots of every block (q4_k: and the mins')."""
    k = 1536 if O.FORMATS[fmt]["block"] == 256 else 736
    rng = np.random.default_rng(seed)
    wq, ws = host.split(fmt, O.weights(fmt, rng, n, k), n, k)
    xq, xd = host.quantize(fmt, dev(O.activations(rng, k, m, block=O.ACT_BLOCK[O.FORMATS[fmt]["act"]])))
    return k, dev(wq), ws.copy(), xq, xd.clone()


def terms(fmt, ws, xd, s):
    """f64 [M][N][blocks] terms of Y with the scale products rounded to f32, and their magnitudes."""
    half = ws.view(torch.float16).float()
    if fmt != "q4_k":
        t = (xd[:, None, :] * half[None]).double() * s.double()
        return t, t.abs()
    half = half.view(ws.shape[0], -1, 8)
    a = (xd[:, None, :] * half[None, :, :, 0]).double() * s[..., 0].double()
    b = (xd[:, None, :] * half[None, :, :, 1]).double() * s[..., 1].double()
    return a - b, a.abs() + b.abs()


def run(fmt, n, m, special):
    k, wq, ws, xq, xd = case(fmt, n, m, 7 * n + m)
    ws = torch.from_numpy(ws).cuda()
    f = host.FORMATS[fmt]
    launch = _abi.gemm_launch(host.FMT_ID[fmt], m, n, k, k // f["block"] * f["qbytes"])
    assert launch[0], "the batched kernel multiplies its scales on the vector unit"
    print(f"special scales {fmt} n={n} k={k} m={m} {special.__name__} {launch}", flush=True)
    clean, s = host.gemm(fmt, wq, ws, xq, xd, n, k, store_s=True)
    rows, cols = special(fmt, ws, xd)
    y, s2 = host.gemm(fmt, wq, ws, xq, xd, n, k, store_s=True)
    plain, _ = host.gemm(fmt, wq, ws, xq, xd, n, k)
    assert torch.equal(s, s2)  # the dots know no scales
    assert bool(((y == plain) | (y.isnan() & plain.isnan())).all())
    return clean, plain, *terms(fmt, ws, xd, s), rows, cols


def infinite_and_nan(fmt, ws, xd):
    """An infinite d_w in row 5, a NaN one in row 18, an infinite d_x in column 3, a NaN one in column 9."""
    per = 8 if fmt == "q4_k" else 1
    ws[5, 2 * per], ws[18, 1 * per] = 0x7C00, 0x7E00
    if fmt == "q4_k":
        ws[33, 1] = 0x7C00  # an infinite dmin
    xd[3, 2], xd[9, -1] = float("inf"), float("nan")
    return [5, 18, 33] if fmt == "q4_k" else [5, 18], [3, 9]


def subnormal_products(fmt, ws, xd):
    """Every product f32(d_w * d_x) subnormal."""
    xd.mul_(2.0**-126)
    return [], []


@pytest.mark.parametrize("fmt", ["q4_0", "tq2_0", "q8_0", "iq4_nl", "q4_k"])
@pytest.mark.parametrize("n,m", SHAPES)
def test_infinite_and_nan_scales_stay_in_their_row_or_column(fmt, n, m):
    clean, y, t, _, rows, cols = run(fmt, n, m, infinite_and_nan)
    keep = torch.ones_like(y, dtype=torch.bool)
    keep[:, rows] = False
    keep[cols] = False
    assert torch.equal(y[keep], clean[keep])
    ref = t.sum(2)
    assert torch.equal(y.isnan(), ref.isnan()) and torch.equal(y.isinf(), ref.isinf())
    assert torch.equal(y[y.isinf()] > 0, ref[y.isinf()] > 0)
    assert not bool(y[:, rows].isfinite().any()) and not bool(y[cols].isfinite().any())


@pytest.mark.parametrize("fmt", ["q4_0", "tq2_0", "q8_0", "iq4_nl", "q4_k"])
@pytest.mark.parametrize("n,m", SHAPES)
def test_subnormal_scale_products_are_kept(fmt, n, m):
    _, y, t, mag, _, _ = run(fmt, n, m, subnormal_products)
    nb = t.shape[2]
    # as test_gpu_gemm_tile.py's bound, and half the smallest subnormal for each of a term's and a sum's roundings
    bound = (2 * nb + 16) * 2.0**-24 * mag.sum(2) + (4 * nb + 16) * 2.0**-150
    assert bool(((y.double() - t.sum(2)).abs() <= bound).all())
    assert float((y != 0).float().mean()) > 0.9
