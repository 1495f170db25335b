"""W4A8 few-row kernel (up to 32 rows, k any multiple of 32): bit for bit against the CPU oracle at
its row classes (4, 8, 16, 32), a ragged last strip of channels, k that leaves waves without a block
or with part of one, both workgroup sizes, zero points at the int32 limits, strides and 16-bit
outputs."""

import ctypes

import numpy as np
import pytest

import tqt_testlib as T
from test_gpu_w4a8_h16 import bounds, run_h16, to16
from test_gpu_w4a8_tile import _check, _gr

pytestmark = pytest.mark.gpu

SHAPES = [
    (1, 1, 32),          # one 32-k group
    (4, 17, 288),        # one block and part of another
    (5, 100, 2048),      # four waves, two blocks each
    (2, 31, 2080),       # eight waves, the first with part of a second block
    (8, 515, 4128),
    (9, 33, 13792),
    (16, 1000, 4096),
    (17, 40, 96),
    (32, 515, 2880),
    (31, 4096, 4096),
    (3, 8200, 2112),     # more than two strips a CU
    (8, 8193, 544),
    (16, 8208, 2304),
]


@pytest.mark.parametrize("m,n,k", SHAPES)
def test_w4a8_skinny(gpu, m, n, k):
    assert T.w4a8_route(m, n, k) == T.W4A8_FEW_ROW
    d = T.gen_w4a8(m, n, k, seed=m + n + k, with_c=bool(m & 1), with_bias=bool(n & 1))
    lo, hi = (-np.inf, np.inf) if m % 2 else (-0.75, 1.25)
    got = _gr().run_w4a8(d, lo, hi)
    exp = T.oracle_w4a8(d["A"], d["Bp"], d["C"], d["bias"], lo, hi, d["scale_a"], d["zp_a"],
                        d["scale_b"])
    _check(got, exp, "m=%d n=%d k=%d" % (m, n, k))


@pytest.mark.parametrize("m", [7, 20])
def test_w4a8_skinny_extremes(gpu, m):
    """Every product at its largest magnitude over the longest k, and zero points at the int32 limits:
    the sums fit, the correction wraps as in the reference."""
    n, k = 40, 65536
    assert T.w4a8_route(m, n, k) == T.W4A8_FEW_ROW
    d = T.gen_w4a8(m, n, k, seed=5)
    d["A"][:] = -128
    d["A"][1] = 127
    d["Bp"][0::2] = 0x00
    d["Bp"][1::2] = 0xFF
    d["zp_a"] = np.where(np.arange(m) % 2, np.int32(2 ** 31 - 1), np.int32(-2 ** 31)).astype(np.int32)
    got = _gr().run_w4a8(d)
    exp = T.oracle_w4a8(d["A"], d["Bp"], d["C"], d["bias"], -np.inf, np.inf, d["scale_a"],
                        d["zp_a"], d["scale_b"])
    _check(got, exp, "extremes")


@pytest.mark.parametrize("m", [6, 19])
def test_w4a8_skinny_strides(gpu, m):
    """Row strides larger than the rows, and nothing written outside the m x n results."""
    import torch

    g = _gr()
    n, k = 262, 352
    assert T.w4a8_route(m, n, k) == T.W4A8_FEW_ROW
    lda, ldb, ldc, ldd = k + 48, k + 96, n + 5, n + 3
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
@pytest.mark.parametrize("m,n,k", [(10, 131, 2144), (25, 1030, 544)])
def test_w4a8_skinny_16bit(gpu, shim, bf16, m, n, k):
    assert T.w4a8_route(m, n, k) == T.W4A8_FEW_ROW
    d = T.gen_w4a8(m, n, k, seed=m + k, with_c=True)
    C16, bias16 = to16(d["C"], bf16), to16(d["bias"], bf16)
    lo, hi = bounds(bf16)
    got = run_h16(shim, d, C16, bias16, lo, hi, bf16, False)
    exp = T.oracle_w4a8_h16(d["A"], d["Bp"], C16, bias16, lo, hi, d["scale_a"], d["zp_a"],
                            d["scale_b"], bf16)
    np.testing.assert_array_equal(np.asarray(got).view(np.uint16), np.asarray(exp).view(np.uint16))
