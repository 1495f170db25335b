"""Dispatch rules of the launchers, evaluated on the CPU (torq-tile_amd/csrc/route.hpp)."""

import random
import time

import pytest

import tqt_testlib as T


@pytest.fixture()
def rules(route):
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
    assert rules.tqtr_grid_fits((1 << 23) - 1, 512) and not rules.tqtr_grid_fits(1 << 23, 512)
    assert rules.tqtr_grid_fits((1 << 24) - 1, 256) and not rules.tqtr_grid_fits(1 << 24, 256)


# (m, n, k, whether the k-split kernel was the faster one): each from a side-by-side measurement with
# the weights from HBM, where the two differ by 5% and more
@pytest.mark.parametrize("m,n,k,ksplit", [
    (1, 8192, 8192, True), (2, 8192, 8192, True), (8, 8192, 8192, True), (1, 5120, 13824, True),
    (2, 11008, 4096, True), (2, 6272, 2816, True), (8, 4096, 4096, True), (1, 25216, 8448, True),
    (1, 26176, 5888, True), (9, 8192, 8192, True), (17, 1280, 3840, True), (24, 2048, 2048, True),
    (17, 512, 2048, True), (2, 2048, 2048, True), (1, 272, 4608, True),
    (2, 16384, 512, False), (4, 1024, 1024, False), (1, 896, 13824, False), (8, 896, 13824, False),
    (8, 4096, 11008, False), (8, 5120, 13824, False), (8, 17648, 9472, False),
    (4, 9008, 11264, False), (8, 12080, 4608, False), (2, 18720, 1792, False),
    (8, 15712, 3072, False), (12, 6352, 4608, False),
    (16, 4096, 4096, False), (32, 4096, 4096, False), (32, 7616, 1280, False),
])
def test_w4a8_few_rows(rules, m, n, k, ksplit):
    want = T.W4A8_OTHER if ksplit else T.W4A8_FEW_ROW
    assert rules.tqtr_w4a8_route(m, n, k, 1) == want
    # off the 256 grid of k the few-row kernel has only the tiles beside it
    assert rules.tqtr_w4a8_route(m, n, k + 32, 0) != T.W4A8_OTHER


def test_w4a8_one_group(rules):
    """A few outputs of one 32-k group stay with one thread each."""
    for m, n in ((33, 100), (33, 700), (100, 100)):
        assert rules.tqtr_w4a8_route(m, n, 32, 0) == T.W4A8_OTHER
        assert rules.tqtr_w4a8_route(m, n, 64, 0) != T.W4A8_OTHER


# (m, n, k, dynamic, packed, whether the few-row kernel was the faster one), measured side by side with
# the weights from HBM, where the two differ by 8% and more
@pytest.mark.parametrize("m,n,k,dyn,packed,few", [
    (1, 4096, 4096, 0, 0, True), (32, 4096, 4096, 0, 0, True), (8, 4096, 4096, 1, 0, True),
    (1, 28672, 8192, 0, 0, True), (8, 28672, 8192, 1, 0, True), (16, 4096, 11008, 0, 1, True),
    (32, 11008, 4096, 0, 0, True), (17, 16384, 4096, 1, 0, True), (33, 4096, 4096, 0, 0, True),
    (64, 512, 2048, 1, 0, True), (16, 1024, 4112, 0, 0, True),
    (1, 16384, 512, 0, 0, False), (16, 16384, 512, 0, 0, False), (9, 16384, 512, 1, 0, False),
    (17, 16384, 4096, 0, 0, False), (24, 28672, 8192, 0, 0, False), (32, 28672, 8192, 0, 1, False),
    (1, 23232, 128, 0, 0, False), (16, 23232, 128, 1, 0, False), (32, 26768, 384, 0, 1, False),
    (65, 23232, 128, 0, 0, False), (65, 23232, 128, 1, 0, False), (64, 11008, 4096, 0, 0, False),
])
def test_w8a8_few_rows(rules, m, n, k, dyn, packed, few):
    assert rules.tqtr_w8a8_few_row(m, n, k, dyn, packed) == few


# (m, n, k, dynamic, whether large tiles were the faster ones), measured side by side
@pytest.mark.parametrize("m,n,k,dyn,tiles", [
    (4000, 11008, 4096, 0, True), (2048, 4096, 11008, 0, True), (2000, 4096, 4096, 1, True),
    (1000, 4096, 4112, 0, True), (313, 13616, 1280, 0, True), (2048, 4096, 512, 1, True),
    (998, 6880, 192, 0, True), (2572, 1968, 352, 0, True),
    (2048, 4096, 1024, 0, False), (2048, 4096, 512, 0, False), (551, 30304, 128, 0, False),
    (133, 22176, 256, 0, False), (1000, 4096, 4096, 0, False), (512, 4096, 4112, 0, False),
    (64, 32544, 3104, 0, False),
])
def test_w8a8_large_tiles(rules, m, n, k, dyn, tiles):
    assert (rules.tqtr_w8a8_tile(m, n, k, dyn) != T.W8A8_NO_TILE) == tiles


# (form, m, n, k, taps, whether the 64 x 64 tiles were the faster ones), measured side by side, 15% apart
# and more
@pytest.mark.parametrize("form,m,n,k,taps,tiles", [
    (T.EDGE_NK, 64, 64, 44, 0, False), (T.EDGE_NK, 17, 33, 40, 0, False),
    (T.EDGE_NK, 200, 255, 41, 0, False), (T.EDGE_NK, 32, 256, 40, 0, False),
    (T.EDGE_NK, 1, 16, 36, 0, False), (T.EDGE_NK, 1, 255, 100, 0, True),
    (T.EDGE_NK, 200, 4097, 33, 0, True), (T.EDGE_NK, 64, 255, 130, 0, True),
    (T.EDGE_KN_CLAMP, 200, 255, 33, 0, False), (T.EDGE_KN_CLAMP, 17, 33, 40, 0, False),
    (T.EDGE_KN_CLAMP, 1, 255, 65, 0, True), (T.EDGE_KN_CLAMP, 64, 1023, 100, 0, True),
    (T.EDGE_KN_CLAMP, 512, 4097, 33, 0, True),
    (T.EDGE_KN_REQUANT, 64, 255, 81, 0, False), (T.EDGE_KN_REQUANT, 16, 1023, 100, 0, True),
    (T.EDGE_CONV, 784, 32, 27, 9, False), (T.EDGE_CONV, 12544, 8, 27, 9, False),
    (T.EDGE_CONV, 12544, 32, 24, 1, False), (T.EDGE_CONV, 12544, 96, 27, 9, True),
    (T.EDGE_CONV, 784, 32, 147, 49, True), (T.EDGE_CONV, 49, 32, 49, 49, True),
])
def test_int8_edge(rules, form, m, n, k, taps, tiles):
    assert rules.tqtr_int8_edge_faster(form, m, n, k, taps) == tiles


@pytest.mark.parametrize("f32", [0, 1])
@pytest.mark.parametrize("k", [640, 1024, 2048, 4096, 11264])
def test_w4a16_sums(rules, f32, k):
    """32-wide blocks that another kernel sums in f64 or short chains are never left to plain f32
    accumulators; blocks that only one thread per output takes otherwise may be."""
    other = T.W4A16_CHUNK if k % 512 == 0 else T.W4A16_REGISTER
    for m in (33, 64, 100, 256, 1024, 4000):
        for n in (512, 4096, 14336):
            r = rules.tqtr_w4a16_route(m, n, k, 32, f32, other)
            assert r % 100 < T.W4A16_TILE_128X256 or r // 100 > 0
    assert rules.tqtr_w4a16_route(1024, 4096, 11008, 128, f32, T.W4A16_GENERIC) == \
        T.W4A16_TILE_128X128


# (m, n, k, whether the few-row kernel was faster than the 32-row kernels): 32-wide blocks, measured side
# by side with the weights from HBM
@pytest.mark.parametrize("m,n,k,few", [
    (1, 4096, 4096, True), (16, 4096, 4096, True), (1, 14336, 4096, True), (8, 11008, 4096, True),
    (16, 8192, 8192, True), (8, 28672, 8192, True), (1, 1280, 3840, True), (16, 19472, 896, True),
    (12, 11008, 4096, False), (4, 14336, 4096, False), (12, 23200, 512, False),
    (12, 8800, 7168, False),
])
def test_w4a16_few_rows(rules, m, n, k, few):
    other = T.W4A16_CHUNK if k % 512 == 0 else T.W4A16_REGISTER
    assert (rules.tqtr_w4a16_route(m, n, k, 32, 0, other) == T.W4A16_FEW_ROW) == few


def test_cf_halo_rows(rules):
    """The channel-first convolution's halo bound without the walk over the output rows: the same value
    for any geometry, and no work that grows with the output rows."""
    rng = random.Random(7)
    for _ in range(20000):
        OH, OW, IH = rng.randint(1, 90), rng.randint(1, 90), rng.randint(1, 200)
        if rng.random() < 0.3:
            OW = rng.randint(1, 4)
        SH, PH = rng.choice([0, 1, 1, 2, 3, 7]), rng.choice([0, 1, 2, 3, 9, 60])
        ext = rng.choice([1, 3, 5, 9, 17, 40])
        a = (OH, OW, IH, SH, PH, ext, 64)
        assert rules.tqtr_cf_halo_rows(*a) == rules.tqtr_cf_halo_rows_walk(*a), a
    wide = (4096, 4096, 4096, 1, 1, 3, 64)

    def best(f):
        t = []
        for _ in range(50):
            t0 = time.perf_counter()
            f(*wide)
            t.append(time.perf_counter() - t0)
        return min(t)

    assert rules.tqtr_cf_halo_rows(*wide) == rules.tqtr_cf_halo_rows_walk(*wide)
    assert best(rules.tqtr_cf_halo_rows) < 0.5 * best(rules.tqtr_cf_halo_rows_walk)
