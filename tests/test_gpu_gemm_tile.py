"""The tiled matrix-core GEMM (komp_*_gemm, rows of more than 4 K steps): S exact and Y within its bound against the oracle on
ragged shapes (rows, columns and blocks that leave partial tiles, steps and K groups; a few of few columns run the batched
kernel), and on shapes large enough for every plan, where the exact block dots are f64 matrix products of the oracle's decoded weights."""

import numpy as np
import pytest
import torch

from comp_amd import _abi, host
from oracle import oracle as O
from tests.test_gpu_gemm import check, dev

pytestmark = pytest.mark.gpu
FMTS = ["q4_0", "tq2_0", "q8_0", "iq4_nl", "q4_k"]

# (n, k of 32-value blocks, k of 256-value blocks, m)
RAGGED = [(1, 672, 1280, 5), (33, 4192, 2816, 9), (100, 544, 1280, 16), (70, 1056, 1536, 31), (1, 672, 1280, 65), (17, 1120, 2304, 70), (129, 1056, 1536, 97), (45, 4192, 2816, 129), (300, 736, 1792, 83)]


@pytest.mark.parametrize("fmt", FMTS)
@pytest.mark.parametrize("shape", range(len(RAGGED)))
@pytest.mark.parametrize("extreme", [False, True])
def test_ragged_shapes_match_oracle(fmt, shape, extreme):
    n, k32, k256, m = RAGGED[shape]
    check(fmt, n, k256 if O.FORMATS[fmt]["block"] == 256 else k32, m, 700 + shape, extreme)


@pytest.mark.parametrize("fmt", FMTS)
def test_unaligned_scales_and_padded_rows(fmt):
    k = 1536 if O.FORMATS[fmt]["block"] == 256 else 1120
    check(fmt, 45, k, 66, 21, ws_offset=8 if fmt == "q4_k" else 1, pad=48)


# (n, m) at 1536 or 736 values of K: with MORE and REST every plan of gemm_tile_plan on a 256-CU device, in every format
# (tests/test_gemm_launch.py holds the lists to that)
PLANS = [(64, 5), (4331, 5), (8400, 9), (1420, 33), (4331, 20), (8400, 20), (2340, 200), (5340, 49), (8400, 33), (670, 768),
         (8400, 66), (8400, 130), (11000, 130), (12330, 200), (11000, 260), (11000, 515)]


@pytest.mark.parametrize("fmt", FMTS)
@pytest.mark.parametrize("shape", range(len(PLANS)))
def test_every_plan(fmt, shape):
    n, m = PLANS[shape]
    check_large(fmt, n, 1536 if O.FORMATS[fmt]["block"] == 256 else 736, m, shape)


# plans that the shapes above do not take, on a 256-CU device
MORE = [("q4_0", 28700, 1056, 66), ("iq4_nl", 4099, 1056, 5), ("q4_0", 12330, 672, 17), ("q4_0", 16500, 672, 1100),
        ("tq2_0", 70, 2304, 9), ("tq2_0", 4099, 2304, 5), ("tq2_0", 28700, 1536, 260), ("tq2_0", 28700, 1536, 5),
        ("q8_0", 20000, 672, 768), ("q8_0", 12330, 672, 17), ("q4_k", 4099, 2304, 9), ("q4_k", 8211, 1792, 17)]


@pytest.mark.parametrize("fmt,n,k,m", MORE)
def test_more_plans(fmt, n, k, m):
    check_large(fmt, n, k, m, n + m)


# (format, n, k, m, the workgroup's K groups, row groups, row tiles and column tiles on a 256-CU device)
REST = [("q4_0", 4331, 1280, 5, (4, 1, 2, 1)), ("q4_0", 6912, 1280, 17, (4, 2, 1, 2)), ("iq4_nl", 28700, 1280, 130, (1, 4, 2, 4)),
        ("iq4_nl", 16500, 672, 1100, (1, 4, 2, 8)), ("iq4_nl", 6912, 1280, 17, (4, 2, 1, 2)),
        ("iq4_nl", 12330, 672, 17, (4, 2, 2, 2)), ("q4_k", 8400, 1280, 12, (4, 1, 2, 1))]  # fmt: skip


@pytest.mark.parametrize("fmt,n,k,m,plan", REST)
def test_remaining_plans(fmt, n, k, m, plan):
    f = host.FORMATS[fmt]
    launch = _abi.gemm_launch(host.FMT_ID[fmt], m, n, k, k // f["block"] * f["qbytes"])
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:
        assert launch[:5] == (True, *plan)
    check_large(fmt, n, k, m, n + m)


def check_large(fmt, n, k, m, seed):
    blk = O.FORMATS[fmt]["block"]
    nb = k // blk
    rng = np.random.default_rng(seed)
    W = O.weights(fmt, rng, n, k)
    wq, ws = host.split(fmt, W, n, k)
    x = O.activations(rng, k, m, block=O.ACT_BLOCK[O.FORMATS[fmt]["act"]])
    print(f"tile gemm {fmt} n={n} k={k} m={m} plan {host.gemm_plan(fmt, m, n, k)}", flush=True)
    xq, xd = host.quantize(fmt, dev(x))
    y, s = host.gemm(fmt, dev(wq), dev(ws), xq, xd, n, k, store_s=True)
    y_plain, _ = host.gemm(fmt, dev(wq), dev(ws), xq, xd, n, k)
    assert torch.equal(y, y_plain)
    v = dev(O.weight_values(fmt, wq, n, k).astype(np.float64)).view(n, nb, blk)
    q = xq.double().view(m, nb, blk)
    if fmt == "q4_k":
        sc, mn = (dev(a.astype(np.float64)) for a in O.q4_k_scales(ws.view(np.uint8).reshape(n, nb, 16)[:, :, 4:]))
        v = (v.view(n, nb, 8, 32) * sc[..., None]).reshape(n, nb, 256)
        qs = q.view(m, nb, 8, 32).sum(3)
        d = dev(O.f16_bits_to_f32(ws.reshape(n, nb, 8)[:, :, 0]).astype(np.float64))
        dmin = dev(O.f16_bits_to_f32(ws.reshape(n, nb, 8)[:, :, 1]).astype(np.float64))
    else:
        d = dev(O.f16_bits_to_f32(ws).astype(np.float64))
    ref = torch.zeros((m, n), dtype=torch.float64, device="cuda")
    mag = torch.zeros_like(ref)  # the terms' magnitudes
    for b in range(nb):
        dots = q[:, b] @ v[:, b].T.contiguous()  # exact: integers below 2^53
        scale = xd[:, b, None].double() * d[None, :, b]
        if fmt == "q4_k":
            mins = qs[:, b] @ mn[:, b].T.contiguous()
            assert torch.equal(s[:, :, b, 0].double(), dots) and torch.equal(s[:, :, b, 1].double(), mins)
            ms = xd[:, b, None].double() * dmin[None, :, b]
            ref += scale * dots - ms * mins
            mag += (scale * dots).abs() + (ms * mins).abs()
        else:
            assert torch.equal(s[:, :, b].double(), dots)
            ref += scale * dots
            mag += (scale * dots).abs()
    # each term takes at most 4 roundings of its own and nb (q4_k: 2 nb) in the running sum, plus the K groups' sums
    assert bool(((y.double() - ref).abs() <= (2 * nb + 16) * 2.0**-24 * mag).all())
    assert float((y.double() - ref).norm() / ref.norm()) <= 1e-6
