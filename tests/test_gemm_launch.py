"""Which matrix-core GEMM launch a call makes (the library's plan query; no GPU needed)."""

import os
import re

import pytest

from comp_amd import _abi, host
from tests import test_gpu_gemm_tile as tile_tests

FMTS = sorted(host.FMT_ID)


def launch(fmt, m, n, k, store_s=False):
    f = host.FORMATS[fmt]
    return _abi.gemm_launch(host.FMT_ID[fmt], m, n, k, k // f["block"] * f["qbytes"], store_s)


@pytest.mark.parametrize("fmt", FMTS)
def test_column_groups_fit_the_grid(fmt):
    """Whatever the plan's column tiles, and with S the smaller ones of the launch that writes it."""
    for m in (1, 16 * 65535, 1 << 20, 1 << 24):
        for n in (1, 100, 3000):
            for k in (1280, 2048, 4096, 8192):
                for store_s in (False, True):
                    _, _, _, _, col_tiles, col_groups = launch(fmt, m, n, k, store_s)
                    assert 1 <= col_groups <= 65535 and 16 * col_tiles * col_groups >= min(m, 16 * 65535)


@pytest.mark.parametrize("fmt", FMTS)
def test_s_keeps_the_k_split(fmt):
    """Y is the same bit for bit with and without S: both launches split K alike."""
    for m in (4, 20, 60, 300, 2000):
        for n in (64, 2000, 9000, 40000):
            for k in (1280, 4096, 14336):
                a, b = launch(fmt, m, n, k), launch(fmt, m, n, k, True)
                assert a[0] == b[0] and a[1] == b[1]


@pytest.mark.parametrize("fmt", FMTS)
@pytest.mark.parametrize("m", [65, 80, 96])
def test_one_round_of_workgroups_fits_every_xcd(fmt, m):
    """5200 rows by a few column groups: a row group's column groups share one of the 8 XCDs, so a plan of at most a
    workgroup a CU in all must not leave an XCD more of them than its 32 CUs (a second round there costs 45-65%)."""
    _, k_groups, row_groups, row_tiles, _, col_groups = launch(fmt, m, 5200, 8192)
    groups = -(-5200 // (16 * row_groups * row_tiles))
    assert groups * col_groups > 256 or -(-groups // 8) * col_groups <= 32


@pytest.mark.parametrize("m,n,k", [(16, 9216, 1536), (24, 9216, 1280), (16, 12288, 1280)])
def test_q4_k_short_rows_take_few_k_groups(m, n, k):
    """Rows of 5-6 blocks leave most of 8 K groups idle, and 16-row workgroups come three or more a CU: 8.2 us on 32 rows
    by 4 K groups against 12.2 (9216 x 1536 at 16 columns)."""
    tiled, k_groups, row_groups, row_tiles, *_ = launch("q4_k", m, n, k)
    assert tiled and k_groups <= 4 and row_groups * row_tiles >= 2


# (format, columns, rows, K, tiled) on 256 CUs, on both sides of each line: a quantizer and a GEMM on the tile, over the
# same on the batched kernel, with weights out of the caches (and left there by the replay before)
# fmt: off
MEASURED = [
    ("q4_0", 4, 4096, 2560, False),  # 1.12 (1.01)
    ("q4_0", 6, 4096, 2560, False),  # 1.11 (1.05)
    ("q4_0", 12, 4096, 2560, True),  # 1.03 (0.92)
    ("q4_0", 4, 3072, 1280, True),  # 1.07 (0.95)
    ("q4_0", 4, 4096, 4096, True),  # 1.05 (0.97)
    ("q4_0", 4, 4096, 14336, False),  # 1.07 (1.04)
    ("q4_0", 12, 4096, 14336, True),  # 0.95 (0.95)
    ("q4_0", 4, 6144, 6912, True),  # 1.01 (0.85)
    ("q4_0", 8, 14336, 6912, False),  # 1.04 (1.03)
    ("q4_0", 12, 14336, 6912, True),  # 1.01 (1.00)
    ("q4_0", 4, 10240, 6912, True),  # 0.96 (0.95)
    ("q4_0", 17, 28672, 6912, False),  # 1.11 (1.10)
    ("q4_0", 24, 28672, 6912, True),  # 1.00 (1.02)
    ("iq4_nl", 4, 4096, 2560, False),  # 1.10 (1.00)
    ("iq4_nl", 4, 4096, 14336, True),  # 1.02 (0.96)
    ("iq4_nl", 17, 28672, 4096, False),  # 1.16 (1.18)
    ("iq4_nl", 24, 24576, 4096, True),  # 1.00 (1.00)
    ("q8_0", 4, 4096, 1280, True),  # 1.05 (1.00)
    ("q8_0", 16, 5120, 4096, True),  # 0.68 (0.56)
    ("tq2_0", 4, 2560, 6912, False),  # 1.09 (1.05)
    ("tq2_0", 8, 2560, 6912, True),  # 1.02 (0.96)
    ("tq2_0", 9, 4096, 2560, False),  # 1.03 (1.03)
    ("tq2_0", 4, 2560, 8192, True),  # 0.97 (0.91)
    ("tq2_0", 4, 6912, 2560, True),  # 0.90 (0.86)
    ("q4_k", 16, 2048, 6912, False),  # 1.08 (1.03)
    ("q4_k", 16, 2048, 4096, True),  # 0.97 (0.97)
    ("q4_k", 17, 2560, 6912, False),  # 1.25 (1.20)
    ("q4_k", 33, 4096, 6912, False),  # 1.20 (1.17)
    ("q4_k", 48, 4096, 6912, True),  # 1.03 (1.03)
    ("q4_k", 32, 4096, 4096, True),  # 0.94 (0.92)
    ("q4_k", 8, 6912, 4096, False),  # 1.09 (1.07)
    ("q4_k", 16, 6912, 4096, True),  # 0.90 (0.87)
    ("q4_k", 8, 14336, 4096, False),  # 1.05 (1.01)
    ("q4_k", 12, 14336, 4096, True),  # 0.94 (0.92)
    ("q4_k", 8, 18432, 4096, True),  # 0.82 (0.83)
    ("q4_k", 8, 32768, 4096, False),  # 1.04 (1.05)
    ("q4_k", 12, 32768, 4096, True),  # 0.95 (0.95)
]
# fmt: on


@pytest.mark.parametrize("fmt,m,n,k,tiled", MEASURED)
def test_the_dispatch_keeps_to_the_measured_lines(fmt, m, n, k, tiled):
    assert launch(fmt, m, n, k)[0] == tiled


CSRC = os.path.join(os.path.dirname(_abi.__file__), "csrc")


def built(fmt):
    """(row groups, row tiles, column tiles, K groups) of the tiled plans that the source builds for a format."""
    flags = dict(q4=fmt in ("q4_0", "iq4_nl"), tq2=fmt == "tq2_0", q8=fmt == "q8_0", qk=fmt == "q4_k", true=True)
    with open(os.path.join(CSRC, "gemm_tile.h")) as f:
        lines = re.findall(r"^  KOMP_TILE_PLAN\(([^()]*)\)", f.read(), re.M)
    plans = [line.split(",") for line in lines]
    return {tuple(map(int, p[1:])) for p in plans if eval(p[0].replace("||", " or ").replace("!", " not "), {}, flags)}


def reached(fmt):
    """(tiled, K groups, row groups, row tiles, column tiles) of launches over a grid of shapes, on 256 CUs."""
    blk = host.FORMATS[fmt]["block"]
    cols = (1, 4, 8, 12, 14, 16, 17, 20, 24, 32, 33, 40, 48, 49, 64, 65, 96, 128, 130, 200, 333, 515, 1024, 1100, 2048)
    rows = (64, 300, 700, 1500, 2560, 3584, 4096, 5200, 6912, 8400, 9216, 11000, 12330, 14336, 16500, 20000, 24576, 28700, 40000)
    values = (672, 736, 1280, 1536, 2048, 2560, 4096, 6912, 8192, 14336)
    return {launch(fmt, m, n, k)[:5] for m in cols for n in rows for k in values if k % blk == 0}


@pytest.mark.parametrize("fmt", FMTS)
def test_every_tiled_plan_is_built_reached_and_tested(fmt):
    want = {(wk, rw, wn, cn) for rw, wn, cn, wk in built(fmt)}
    assert {p[1:] for p in reached(fmt) if p[0]} == want
    long = host.FORMATS[fmt]["block"] == 256
    shapes = [(n, k256 if long else k32, m) for n, k32, k256, m in tile_tests.RAGGED]
    shapes += [(n, 1536 if long else 736, m) for n, m in tile_tests.PLANS]
    shapes += [(n, k, m) for f, n, k, m, *_ in (*tile_tests.MORE, *tile_tests.REST) if f == fmt]
    assert {p[1:] for p in (launch(fmt, m, n, k)[:5] for n, k, m in shapes) if p[0]} == want


@pytest.mark.parametrize("fmt", [f for f in FMTS if f != "q4_k"])
def test_batched_plans_that_are_not_built_are_not_asked_for(fmt):
    """Eight or four K groups by four column tiles: only rows that the tiled kernel runs would take them (Q4_K aside; the
    first is built for Q4_0 alone, for the instruction-mix report)."""
    blk = host.FORMATS[fmt]["block"]
    got = {launch(fmt, m, n, nb * blk) for m in (1, 9, 17, 20, 24, 40, 49, 64, 100, 128, 256) for n in range(1, 40000, 499)
           for nb in (1, 2, 3, 4, 6, 8, 12, 16, 17, 100, 700, 2000)}  # fmt: skip
    assert not {p[1:5] for p in got if p and not p[0]} & {(8, 1, 1, 4), (4, 2, 1, 4)}
