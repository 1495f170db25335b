"""Dispatch rules of the launchers, evaluated on the CPU (torq-tile_amd/csrc/route.hpp)."""

import ctypes

import pytest


@pytest.fixture()
def rules(route):
    route.tqtr_scale_block_of.restype = ctypes.c_uint32
    route.tqtr_first_wrong_scale_block.restype = ctypes.c_longlong
    route.tqtr_first_wrong_scale_block.argtypes = [ctypes.c_longlong, ctypes.c_longlong]
    route.tqtr_w4a16_skinny_scales_exact.argtypes = [ctypes.c_longlong, ctypes.c_longlong]
    return route


@pytest.mark.parametrize("bl", [32, 64, 96, 128, 1056, 32 * 4097, 32 * 46341, 32 * 65535, 32 * 65536,
                                32 * 65537, 32 * 65538, 1213664, 32 * 131071])
def test_scale_block_exact_where_taken(rules, bl):
    """Every k of whole blocks below 2^22 that the few-row W4A16 kernel takes has exact scale
    indexes; the narrow blocks are all taken."""
    kmax = ((1 << 22) - 1) // bl * bl
    ks = [bl * i for i in (1, 2, 3, kmax // bl) if 0 < bl * i <= kmax]
    for k in ks:
        taken = rules.tqtr_w4a16_skinny_scales_exact(k, bl)
        wrong = rules.tqtr_first_wrong_scale_block(k, bl)
        assert not taken or wrong == -1, (k, bl, wrong)
        if bl <= 32 * 32768:
            assert taken, (k, bl)


@pytest.mark.parametrize("k,bl", [(2097184, 2097184), (3 * 1213664, 1213664)])
def test_wide_scale_blocks_refused(rules, k, bl):
    """The first widths whose last 32-k blocks would read past their scale are left to the other
    kernels."""
    assert rules.tqtr_first_wrong_scale_block(k, bl) >= 0
    assert not rules.tqtr_w4a16_skinny_scales_exact(k, bl)


def test_grid_fits(rules):
    """A grid dimension holds fewer than 2^32 work-items."""
    rules.tqtr_grid_fits.argtypes = [ctypes.c_longlong, ctypes.c_int]
    assert rules.tqtr_grid_fits((1 << 23) - 1, 512) and not rules.tqtr_grid_fits(1 << 23, 512)
    assert rules.tqtr_grid_fits((1 << 24) - 1, 256) and not rules.tqtr_grid_fits(1 << 24, 256)
