"""W4A16 few-row kernel (groups of up to 16 rows): against exact f64 math and the CPU oracle at its row classes
(2, 8, 16), a ragged last strip of channels, k that leaves waves without a block or with part of one,
both workgroup sizes, every block width class, odd scale strides, C, clamps and infinities."""

import numpy as np
import pytest

import tqt_testlib as T
from test_gpu_parity import check_w4a16
from test_gpu_w4a16_tile import _check_f32, _gr, _run_f32

pytestmark = pytest.mark.gpu

# (m, n, k, bl)
SHAPES = [
    (1, 1, 128, 64),
    (2, 17, 160, 32),        # part of one block: one wave works
    (3, 100, 2048 + 32, 32),
    (8, 31, 2880, 96),       # blocks that straddle the 256-k loads
    (9, 33, 4224, 1056),
    (16, 1000, 1152, 128),   # odd scale stride (9)
    (1, 4096, 4096, 32),
    (7, 515, 11008, 128),
    (1, 8200, 544, 32),      # four waves a workgroup
    (5, 8197, 2304, 64),
    (16, 8193, 1088, 64),
    (17, 100, 2880, 96),     # two row groups, the second of one row
    (33, 515, 4224, 64),
    (64, 300, 11008, 128),
]


@pytest.mark.parametrize("m,n,k,bl", SHAPES)
def test_w4a16_skinny_f32(gpu, m, n, k, bl):
    assert T.w4a16_route(m, n, k, bl, 1, k // bl + m % 2)[0] == T.W4A16_FEW_ROW
    d = T.gen_w4a16(m, n, k, bl=bl, seed=m + n + k, with_c=bool(m & 1), with_bias=bool(n & 1))
    lo, hi = (-np.inf, np.inf) if m % 2 else (-3.0, 4.0)
    _check_f32(_run_f32(d, lo, hi, pad_d=n % 3, pad_s=(m % 2)), d, lo, hi)


@pytest.mark.parametrize("m,n,k,bl", SHAPES)
def test_w4a16_skinny_f16(gpu, shim, m, n, k, bl):
    assert T.w4a16_route(m, n, k, bl, 0)[0] == T.W4A16_FEW_ROW
    d = T.gen_w4a16(m, n, k, bl=bl, seed=m * 3 + n + k, with_c=bool(m & 1), with_bias=bool(n & 1))
    lo, hi = (-65504.0, 65504.0) if m % 2 else (-2.0, 2.5)
    cmin, cmax = int(T.f16_bits(lo)), int(T.f16_bits(hi))
    got = _gr().run_w4a16(shim, d, cmin, cmax)
    exp = T.oracle_w4a16(d["A16"], d["Bp"], d["S16"], bl, d["C16"], d["bias16"], cmin, cmax)
    check_w4a16(got, exp, d, (lo, hi))


@pytest.mark.parametrize("n", [196, 8200])
def test_w4a16_skinny_infinity(gpu, n):
    """An infinite activation gives infinite results of its sign, NaN where its weight is 0, and
    leaves the other rows alone."""
    m, k = 6, 1024 + 64
    assert T.w4a16_route(m, n, k, 64, 1)[0] == T.W4A16_FEW_ROW
    d = T.gen_w4a16(m, n, k, bl=64, seed=9)
    d["A16"][2, 100] = 0x7C00
    d["A16"][5, 1000] = 0xFC00
    got = _run_f32(d)
    for row, byte, sign in ((2, 50, 1), (5, 500, -1)):
        q = (d["Bp"][:, byte] & 15).astype(np.int32) - 8
        assert np.isnan(got[row, q == 0]).all()
        assert (got[row, q > 0] == sign * np.inf).all() and (got[row, q < 0] == -sign * np.inf).all()
    assert np.isfinite(got[[0, 1, 3, 4]]).all()


@pytest.mark.parametrize("k,bl", [(2097184, 2097184), (3 * 1213664, 1213664)])
def test_w4a16_very_wide_blocks(gpu, k, bl):
    """Scale blocks past the few-row kernel's exact indexes (bl / 32 * k / 32 > 2^32): the last 32 k
    count. Only they are not zero, so that the sums are short ones."""
    m, n = 2, 18
    rng = np.random.default_rng(3)
    A = np.zeros((m, k), np.float16)
    A[:, -32:] = rng.standard_normal((m, 32))
    Bp = np.full((n, k // 2), 0x88, np.uint8)
    Bp[:, -16:] = rng.integers(0, 256, (n, 16))
    S = rng.uniform(0.005, 0.02, (n, k // bl)).astype(np.float16)
    d = dict(A16=A.view(np.uint16), Bp=Bp, S16=S.view(np.uint16), bl=bl, C16=None, bias16=None)
    got = _run_f32(d)
    q = np.empty((n, 32))
    q[:, 0::2] = (Bp[:, -16:] & 15).astype(np.float64) - 8
    q[:, 1::2] = (Bp[:, -16:] >> 4).astype(np.float64) - 8
    w = q * S[:, -1:].astype(np.float64)
    a = A[:, -32:].astype(np.float64)
    # 32 products and their sum, the scale, and three additions of zero: 64 roundings at most
    assert (np.abs(got - a @ w.T) <= 64 * 2.0 ** -24 * (np.abs(a) @ np.abs(w).T)).all()
