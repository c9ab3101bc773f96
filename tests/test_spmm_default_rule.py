"""The library's default SpMM tile (host only): the rule restated, at widths
around the edges of its tiles and on both sides of its wave counts."""
import pytest

PAIRS = [(8, 8), (16, 8), (8, 4), (4, 4), (12, 8), (16, 16), (12, 4), (16, 4)]


def mfma_rows(lhs, signed, V):
    planes = 1 if lhs == 4 else (1 if signed else 2) if lhs == 8 else lhs // 4 - (1 if signed else 0)
    return planes * V


def restated(lhs, rhs, signed, m_vec, V, n, slots):
    wide = 256 if rhs == 8 else 128
    tiles = -(-n // wide)
    if rhs != 4 and n % 4 == 0 and mfma_rows(lhs, signed, V) <= 16:
        # the rows' waves in workgroups of two; three tiles leave one of four without columns
        waves = m_vec * (tiles + tiles % 2)
        short = rhs == 8 and 0 < slots < 320 and waves < 16384 and not (waves >= 8192 and slots >= 192)
        if tiles in (2,) + tuple(range(4, 100)) and waves >= 2048 and not short:
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
              1024, 1028, 1280, 1288, 2048, 4096):
        if n % cpd:
            continue
        for m_vec in (1, 63, 255, 256, 257, 341, 342, 511, 512, 513, 1023, 1024, 2048, 4096):
            for V in (2, 4, 8):
                for signed in (True, False):
                    for slots in (0, 1, 191, 192, 319, 320):
                        got = mclib.mc_spmm_default_config(lhs, rhs, 0 if signed else 1, m_vec, V, n, slots)
                        assert got == restated(lhs, rhs, signed, m_vec, V, n, slots), (pair, n, m_vec, V, signed, slots)
                        seen.add(got)
    assert seen == ({13, 15, 16, 17, 20, 22} | ({24} if rhs != 4 else set()))


def test_three_wide_tiles_are_not_four(mclib):
    """516 to 768 columns are three tiles of 256: a quarter of the waves would have no columns."""
    for n in (516, 580, 640, 768):
        assert mclib.mc_spmm_default_config(8, 8, 0, 512, 8, n, 0) == 17
        assert mclib.mc_spmm_default_config(8, 8, 0, 1024, 8, n, 0) == 17
    for n in (512, 772, 1028):
        assert mclib.mc_spmm_default_config(8, 8, 0, 1024, 8, n, 0) == 24


def test_short_rows_of_a_resident_operand(mclib):
    """What the Python products pass on: the slots of the index array, and
    nothing where the tile does not depend on them."""
    import torch
    from magicube_amd import _lib, spmm
    cols = torch.zeros(1024 * 82, dtype=torch.int32)
    assert spmm._row_slots(8, 1024, 1024, cols) == 82
    assert mclib.mc_spmm_default_config(8, 8, 0, 1024, 8, 1024, 82) == 17
    assert spmm._row_slots(8, 1024, 1024, cols[:16]) == 1
    for args in ((16, 1024, 1024, cols), (4, 1024, 1024, cols), (8, 1024, 256, cols), (8, 256, 1024, cols),
                 (8, 1024, 1024, 1 << 20), (8, 0, 1024, cols)):
        assert spmm._row_slots(*args) == 0
    p = 64
    assert mclib.mc_spmm_run_rows(8, 8, 0, -1, 4, 8, 64, 64, None, p, p, p, p, p, None) == _lib.MC_EINVAL_ARG
    assert mclib.mc_spmm_run_rows(8, 8, 0, 82, 0, 8, 64, 64, None, p, p, p, p, p, None) == _lib.MC_OK


def test_refused_arguments_have_no_tile(mclib):
    for args in ((12, 16, 0, 4, 8, 64, 0), (8, 8, 0, 4, 3, 64, 0), (8, 8, 0, -1, 8, 64, 0), (8, 8, 0, 4, 8, 0, 0),
                 (8, 8, 0, 4, 8, 6, 0), (8, 8, 0, 4, 8, 64, -1)):
        assert mclib.mc_spmm_default_config(*args) == -1
