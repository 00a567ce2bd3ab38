"""CPU checks of the rules that choose a kernel and tile for a size, through
the host queries of the C ABI.  No kernel is launched here."""
import ctypes

import pytest

from localmoe35ba3b_amd import _lib

GEMV, KSPLIT, STREAMED, LDS = range(4)
KSPLIT_TILES = [(16, 16), (16, 32), (16, 64), (32, 32), (48, 32), (64, 32), (64, 64), (96, 32)]
STREAMED_TILES = [(96, 128), (128, 128), (128, 256)]
W8A8_TILES = [(32, 64), (64, 64), (64, 128), (128, 128)]
# Sizes [m, n] that take every tile in both ways to deal them to the XCDs, ragged
# in rows and columns; what the GPU tests run.
DENSE = {
    512: [(60, 17), (3, 17), (2100, 17), (3, 4104), (350, 600), (3, 8200), (3000, 34), (17, 4104),
          (2100, 100), (33, 6000), (4000, 70), (60, 4104), (1200, 600), (60, 8200), (1700, 300),
          (385, 1030), (1000, 1030), (97, 8200), (1300, 1030), (1030, 2050), (4000, 2040),
          (1300, 6000)],
    2048: [(60, 17), (3, 17), (2100, 17), (3, 4104), (350, 600), (3, 8200), (3000, 34), (17, 4104),
           (1030, 200), (33, 6000), (4000, 70), (60, 4104), (1030, 600), (33, 8200), (2500, 200),
           (65, 6000), (800, 3500), (200, 8200), (1700, 1030), (1030, 2050), (4000, 2040),
           (1300, 6000)],
    4096: [(60, 17), (3, 17), (2100, 17), (3, 4104), (350, 600), (3, 8200), (3000, 34), (17, 4104),
           (1030, 200), (33, 6000), (4000, 70), (60, 4104), (800, 600), (33, 8200), (530, 900),
           (65, 6000), (800, 3500), (200, 8200), (1700, 1030), (1030, 2050), (4000, 2040),
           (1300, 6000)],
}
W8A8 = [(60, 34), (3, 34), (5000, 70), (33, 8200), (5000, 600), (260, 10000), (3000, 2050),
        (600, 10000)]
SIZES = [(m, n) for n in (16, 64, 128, 256, 512, 1000, 2048, 4096, 8192)
         for m in (9, 45, 130, 333, 700, 1023, 1024, 1100, 1900, 2048, 3000, 4096, 10000, 20000)]


def linear_form(m, n, k):
    form = (ctypes.c_int64 * 4)()
    assert _lib.lib().lm_w8a16_linear_form(m, n, k, form) == _lib.LM_OK
    return tuple(form)


def w8a8_form(m, n, k, swiglu=False):
    form = (ctypes.c_int64 * 4)()
    assert _lib.lib().lm_w8a8_gemm_form(m, n, k, int(swiglu), form) == _lib.LM_OK
    return tuple(form)


@pytest.mark.parametrize('k', DENSE)
def test_sizes_take_every_dense_tile(k):
    forms = [linear_form(m, n, k) for m, n in DENSE[k]]
    assert sorted(forms) == sorted(
        (kernel, *tile, deal) for kernel, tiles in ((KSPLIT, KSPLIT_TILES),
                                                    (STREAMED, STREAMED_TILES))
        for tile in tiles for deal in (0, 1))


@pytest.mark.parametrize('swiglu', [False, True])
def test_sizes_take_every_w8a8_tile(swiglu):
    forms = [w8a8_form(m, n, 128, swiglu) for m, n in W8A8]
    assert sorted(forms) == sorted((LDS, *tile, deal) for tile in W8A8_TILES for deal in (0, 1))


def _rounds(m, n, rows, cols):
    """Rounds of the busiest of 8 XCDs of 32 CUs, one tile a CU: with a row
    tile's columns on one XCD, and with a column tile's rows."""
    rt, ct = -(-m // rows), -(-n // cols)
    return [-(-tiles // 32) for tiles in (ct * -(-rt // 8), rt * -(-ct // 8))]


@pytest.mark.parametrize('kind', ['w8a16 512', 'w8a16 2048', 'w8a16 4096', 'w8a8 2048'])
def test_tiles_are_dealt_to_all_xcds(kind):
    """No XCD works through rounds of tiles that the other way to deal them
    would have spread: the chosen way takes at most one round more (a short
    last row tile, or less to read for each XCD), and no more than the other
    where the matrix has few columns."""
    name, k = kind.split()
    for m, n in SIZES:
        kernel, rows, cols, by_columns = (linear_form if name == 'w8a16' else w8a8_form)(
            m, n, int(k))
        if kernel == GEMV:
            continue
        taken, other = _rounds(m, n, rows, cols)[::-1 if by_columns else 1]
        assert taken <= other + (1 if n > 2 * m or (m % rows and not by_columns) else 0), (m, n)
        assert n > 1000 or taken <= max(other, 1), (m, n)


def test_short_last_row_tile_stays_with_its_columns():
    """[1060, 2048] by [4096, 2048] ends in a row tile of 36 rows: with whole
    row tiles on an XCD the nine take little longer than eight (29 us), dealt
    by columns two rounds (36)."""
    assert linear_form(1060, 4096, 2048) == (STREAMED, 128, 128, 0)
    assert linear_form(1280, 4096, 2048) == (STREAMED, 128, 128, 1)


def test_router_workspace_is_bounded():
    """Calls of many tokens pass over one workspace in slices."""
    need = _lib.lib().lm_router_workspace_bytes
    assert 0 < need(2048, 256, 2048) < need(32768, 256, 2048) == need(65536, 256, 2048)
    assert need(16384, 256, 4096) == need(65536, 256, 4096) == need(1 << 20, 256, 4096) < 336 << 20


def test_router_digits_only_where_they_pay():
    """Few experts, a short row or few tokens keep the fp64 tiles, which take
    half the time there."""
    pays = _lib.lib().lm_router_workspace_pays
    for t, e, h in ((513, 256, 2048), (2048, 256, 2048), (65536, 256, 2048), (2048, 256, 4096),
                    (4096, 256, 1024), (16384, 128, 2048)):
        assert pays(t, e, h), (t, e, h)
    for t, e, h in ((512, 256, 2048), (1024, 128, 2048), (16384, 17, 2048), (65536, 16, 4096),
                    (16384, 256, 256), (600, 256, 512), (2048, 256, 2016), (2048, 256, 8192)):
        assert not pays(t, e, h), (t, e, h)


def test_descriptor_table_of_no_experts():
    """An empty selection is a table without rows, also of an empty bank."""
    lib = _lib.lib()
    none = [None] * 4 + [0] * 4
    assert lib.lm_expert_table(None, 8, 0, 0, *none, None, None) == _lib.LM_OK
    assert lib.lm_expert_table(None, 8, 3, 0, *none, None, None) == _lib.LM_EINVAL
