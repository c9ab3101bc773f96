"""The library's default SpMM tile (host only): the rule restated, at widths
around the edges of its tiles and on both sides of its wave counts."""
import math

import pytest

PAIRS = [(8, 8), (16, 8), (8, 4), (4, 4), (12, 8), (16, 16), (12, 4), (16, 4)]


def mfma_rows(lhs, signed, V):
    planes = 1 if lhs == 4 else (1 if signed else 2) if lhs == 8 else lhs // 4 - (1 if signed else 0)
    return planes * V


def least_slots(rhs, n, k, waves, tiles, rows):
    """Slots per row from which the wide tile is the default."""
    wide_part, narrow_part = math.gcd(-(-tiles // 2), 8), math.gcd(tiles, 8)     # of B, that an XCD reads
    lines, b_bytes, l2 = n * rhs // 8 % 64 == 0, k * n * rhs // 8, 4 * 2 ** 20
    more = wide_part < narrow_part and b_bytes // wide_part > l2
    if more and lines:
        return 420
    if rhs == 16:
        return 0
    if more:
        return 150
    if rows <= 6 and waves >= (8192 if b_bytes > l2 else 4096):
        return 0
    least = 300 if lines else 150
    if b_bytes > l2 and wide_part >= narrow_part:
        least = least // 2 if wide_part == narrow_part else 50
    if waves >= 16384:
        return min(least, 50)
    if waves >= 8192:
        return min(least, 160 if lines and b_bytes > l2 else 100)
    return least


def restated(lhs, rhs, signed, m_vec, V, n, k, slots):
    wide = 256 if rhs == 8 else 128
    tiles = -(-n // wide)
    rows = mfma_rows(lhs, signed, V)
    # the rows' waves in workgroups of two; three tiles leave one of four without columns
    waves = m_vec * (tiles + tiles % 2)
    if rhs != 4 and n % 4 == 0 and rows <= 16 and waves >= 2048 and tiles not in (1, 3):
        if slots == 0 or slots >= least_slots(rhs, n, k, waves, tiles, rows):
            return 24
    cols = 16 * (32 // rhs)
    narrow = -(-n // cols)
    if narrow >= 8 and 4096 <= m_vec * 8 * -(-narrow // 8) < 8192:
        return 13
    per_wg = 4 if narrow >= 4 else 2 if narrow >= 2 else 1
    if m_vec * per_wg * -(-narrow // per_wg) < 2048:
        return 20 if per_wg == 4 else 22
    return {4: 17, 2: 16, 1: 15}[per_wg]


@pytest.mark.parametrize("pair", PAIRS, ids=lambda p: f"L{p[0]}R{p[1]}")
def test_default_tile(mclib, pair):
    lhs, rhs = pair
    cpd = 32 // rhs
    seen = set()
    for n in (8, 64, 72, 128, 136, 248, 256, 260, 264, 320, 384, 388, 392, 508, 512, 516, 520, 580, 640, 768, 772, 776,
              1024, 1028, 1280, 1288, 1408, 1536, 1792, 2048, 2560, 3072, 3468, 3584, 4096):
        if n % cpd:
            continue
        for m_vec in (1, 63, 255, 256, 342, 511, 512, 513, 1023, 1024, 2048, 4096):
            for V in (2, 4, 8):
                for signed in (True, False):
                    for k in (256, 1024, 2049, 8192):
                        for slots in (0, 1, 49, 50, 74, 75, 99, 100, 149, 150, 159, 160, 299, 300, 419, 420):
                            got = mclib.mc_spmm_default_config(lhs, rhs, 0 if signed else 1, m_vec, V, n, k, slots)
                            exp = restated(lhs, rhs, signed, m_vec, V, n, k, slots)
                            assert got == exp, (pair, n, m_vec, V, signed, k, slots)
                            seen.add(got)
    assert seen == ({13, 15, 16, 17, 20, 22} | ({24} if rhs != 4 else set()))


def test_three_wide_tiles_are_not_four(mclib):
    """516 to 768 columns are three tiles of 256: a quarter of the waves would have no columns."""
    for n in (516, 580, 640, 768):
        assert mclib.mc_spmm_default_config(8, 8, 0, 512, 8, n, 4096, 0) == 17
        assert mclib.mc_spmm_default_config(8, 8, 0, 1024, 8, n, 4096, 0) == 17
    for n in (512, 772, 1028):
        assert mclib.mc_spmm_default_config(8, 8, 0, 1024, 8, n, 4096, 0) == 24


def test_short_rows_and_odd_groups(mclib):
    """Rows of 82 slots; seven workgroups per row beside fourteen, with B in and beyond the L2."""
    default = mclib.mc_spmm_default_config
    assert default(8, 8, 0, 1024, 8, 1024, 4096, 82) == 17
    assert default(8, 8, 0, 1024, 2, 3584, 256, 34) == 24
    for slots, tile in ((400, 17), (800, 24), (0, 24)):
        assert default(8, 8, 0, 1024, 8, 3584, 4096, slots) == tile
    assert default(8, 8, 0, 1024, 8, 4096, 4096, 400) == 24
    assert default(16, 16, 0, 1024, 4, 1792, 4096, 400) == 17


def test_rows_length_that_the_products_pass_on(mclib):
    """The slots of the index array per vector row, and nothing where the tile
    does not depend on them."""
    import torch
    from magicube_amd import _lib, spmm
    cols = torch.zeros(1024 * 82, dtype=torch.int32)
    assert spmm._row_slots(8, 1024, 1024, cols) == spmm._row_slots(16, 1024, 1024, cols) == 82
    assert spmm._row_slots(8, 1024, 1024, cols[:16]) == 1
    for args in ((4, 1024, 1024, cols), (8, 1024, 256, cols), (8, 1024, 1024, 1 << 20), (8, 0, 1024, cols)):
        assert spmm._row_slots(*args) == 0
    p = 64
    assert mclib.mc_spmm_run_rows(8, 8, 0, -1, 4, 8, 64, 64, None, p, p, p, p, p, None) == _lib.MC_EINVAL_ARG
    assert mclib.mc_spmm_run_rows(8, 8, 0, 82, 0, 8, 64, 64, None, p, p, p, p, p, None) == _lib.MC_OK


def test_refused_arguments_have_no_tile(mclib):
    for args in ((12, 16, 0, 4, 8, 64, 64, 0), (8, 8, 0, 4, 3, 64, 64, 0), (8, 8, 0, -1, 8, 64, 64, 0),
                 (8, 8, 0, 4, 8, 0, 64, 0), (8, 8, 0, 4, 8, 6, 64, 0), (8, 8, 0, 4, 8, 64, -1, 0),
                 (8, 8, 0, 4, 8, 64, 64, -1)):
        assert mclib.mc_spmm_default_config(*args) == -1
