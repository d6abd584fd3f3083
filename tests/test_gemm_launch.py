"""Which matrix-core GEMM launch a call makes (the library's plan query; no GPU needed)."""

import pytest

from comp_amd import _abi, host

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
