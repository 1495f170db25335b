"""W4A8 large-tile kernel (many rows): bit-exact against the CPU oracle at the edges of its tiles
(256 x 256, 128 x 128, 64 x 128 and 32 x 128: one row or channel over, ragged channels, rows that end
inside a 32-row fragment), at stage remainders (k of one 32-k group, and one group past whole stages),
each tile over more stages than its ring holds, with C, clamps, zero points at the int32 limits, row
strides larger than the rows, and 16-bit outputs. Each test asserts the tile that its call takes."""

import ctypes

import numpy as np
import pytest

import tqt_testlib as T
from test_gpu_w4a8_h16 import bounds, run_h16, to16

pytestmark = pytest.mark.gpu


def _gr():
    import gpu_run

    return gpu_run


def _check(got, exp, msg):
    np.testing.assert_array_equal(got.view(np.uint32), exp.view(np.uint32), err_msg=msg)


# (m, n, k, tile)
SHAPES = [
    (33, 2100, 32, T.W4A8_TILE_32X128),    # one 32-k group, one row over
    (63, 129, 2880, T.W4A8_TILE_32X128),   # k % 128 == 64, more stages than the ring's six
    (33, 130, 96, T.W4A8_TILE_32X128),     # ragged rows and channels
    (65, 1001, 160, T.W4A8_TILE_32X128),   # odd channel count: scalar stores
    (300, 1000, 864, T.W4A8_TILE_32X128),
    (3100, 257, 672, T.W4A8_TILE_64X128),  # one channel over, six stages in a ring of four
    (193, 5121, 288, T.W4A8_TILE_64X128),  # one row and one channel over
    (513, 4097, 288, T.W4A8_TILE_128X128),  # one row and one channel over
    (1000, 2052, 2048, T.W4A8_TILE_128X128),
    (1025, 4100, 1056, T.W4A8_TILE_128X128),
    (3970, 3970, 256, T.W4A8_TILE_256X256),
    (3100, 3970, 672, T.W4A8_TILE_256X256),  # six stages in a ring of three
    (256, 256, 16352, T.W4A8_TILE_32X128),  # 128 stages, the last one short
]


@pytest.mark.parametrize("m,n,k,tile", SHAPES)
def test_w4a8_tile(gpu, m, n, k, tile):
    assert T.w4a8_route(m, n, k) == tile
    d = T.gen_w4a8(m, n, k, seed=m + n + k, with_c=bool(m & 1), with_bias=bool(n & 1) or m > 500)
    lo, hi = (-np.inf, np.inf) if m % 2 else (-0.75, 1.25)
    got = _gr().run_w4a8(d, lo, hi)
    exp = T.oracle_w4a8(d["A"], d["Bp"], d["C"], d["bias"], lo, hi, d["scale_a"], d["zp_a"],
                        d["scale_b"])
    _check(got, exp, "m=%d n=%d k=%d" % (m, n, k))


def test_w4a8_tile_zero_points_wrap(gpu):
    """Zero points at the int32 limits: the correction wraps, as in the reference."""
    m, n, k = 70, 200, 416
    assert T.w4a8_route(m, n, k) == T.W4A8_TILE_32X128
    d = T.gen_w4a8(m, n, k, seed=5)
    d["zp_a"] = np.where(np.arange(m) % 2, np.int32(2 ** 31 - 1), np.int32(-2 ** 31)).astype(np.int32)
    got = _gr().run_w4a8(d)
    exp = T.oracle_w4a8(d["A"], d["Bp"], d["C"], d["bias"], -np.inf, np.inf, d["scale_a"],
                        d["zp_a"], d["scale_b"])
    _check(got, exp, "zero points")


@pytest.mark.parametrize("pad_d", [3, 4])
def test_w4a8_tile_strides(gpu, pad_d):
    """Row strides larger than the rows (A, B, C and D), D rows that end off a vector, and nothing
    written outside the m x n results."""
    import torch

    g = _gr()
    m, n, k = 150, 262, 352
    assert T.w4a8_route(m, n, k) == T.W4A8_TILE_32X128
    lda, ldb, ldc, ldd = k + 48, k + 96, n + 5, n + pad_d
    d = T.gen_w4a8(m, n, k, seed=11, with_c=True)
    A = np.full((m, lda), 77, np.int8)
    A[:, :k] = d["A"]
    B = np.full((n, ldb // 2), 0xA5, np.uint8)
    B[:, :k // 2] = d["Bp"]
    C = np.full((m, ldc), np.nan, np.float32)
    C[:, :n] = d["C"]
    dA, dB, dC, dbias = g.dev(A), g.dev(B), g.dev(C), g.dev(d["bias"])
    dsa, dza, dsb = g.dev(d["scale_a"]), g.dev(d["zp_a"]), g.dev(d["scale_b"])
    dD = torch.full((m + 2, ldd), 12345.0, dtype=torch.float32, device="cuda:0")
    p = g._mod.QAI8DXQSI4CXParams(dsa.data_ptr(), dza.data_ptr(), dsb.data_ptr())
    g.lib().fn("w4a8", "run")(m, n, k, g.dp(dA), lda, 0, g.dp(dB), ldb, 0, g.dp(dC), ldc,
                              g.dp(dD), ldd, g.dp(dbias), -np.inf, np.inf, ctypes.byref(p))
    got = dD.cpu().numpy()
    exp = T.oracle_w4a8(d["A"], d["Bp"], d["C"], d["bias"], -np.inf, np.inf, d["scale_a"],
                        d["zp_a"], d["scale_b"])
    _check(np.ascontiguousarray(got[:m, :n]), exp, "strides")
    assert (got[m:] == 12345.0).all() and (got[:m, n:] == 12345.0).all()


@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("m,n,k", [(40, 131, 96), (600, 1030, 544)])
def test_w4a8_tile_16bit(gpu, shim, bf16, m, n, k):
    assert T.w4a8_route(m, n, k) >= T.W4A8_TILE_256X256
    d = T.gen_w4a8(m, n, k, seed=m + k, with_c=True)
    C16, bias16 = to16(d["C"], bf16), to16(d["bias"], bf16)
    lo, hi = bounds(bf16)
    got = run_h16(shim, d, C16, bias16, lo, hi, bf16, False)
    exp = T.oracle_w4a8_h16(d["A"], d["Bp"], C16, bias16, lo, hi, d["scale_a"], d["zp_a"],
                            d["scale_b"], bf16)
    np.testing.assert_array_equal(np.asarray(got).view(np.uint16), np.asarray(exp).view(np.uint16))
