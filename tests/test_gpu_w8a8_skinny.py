"""W8A8 few-row kernel (up to 32 rows per workgroup, k split over the waves): bit-exact against the
CPU oracle at its row blocks' edges (1, 7, 8, 9, 16, 17, 31, 32, 33, 64 rows), ragged channels, k of
one 16-byte chunk, under, at and one chunk past a round of the waves' blocks (1024), static and
dynamic, plain and packed operands, C, clamps and strides."""

import ctypes

import numpy as np
import pytest

import tqt_testlib as T

pytestmark = pytest.mark.gpu


def _gr():
    import gpu_run

    return gpu_run


ROWS_K = [(1, 16), (7, 144), (8, 1024), (9, 1040), (16, 2000), (17, 128), (31, 1008), (32, 4096),
          (33, 2064), (64, 512)]


@pytest.mark.parametrize("m,k", ROWS_K)
@pytest.mark.parametrize("n", [16, 37, 300])
def test_w8a8_skinny(gpu, m, k, n):
    assert T.routes().tqtr_w8a8_few_row(m, n, k, 0, 0)
    d = T.gen_w8a8(m, n, k, seed=m + n + k, with_c=bool(m & 1))
    cmin, cmax = (-128, 127) if m % 2 else (-50, 70)
    got = _gr().run_w8a8(d, cmin, cmax)
    exp = T.oracle_w8a8(d["A"], d["B"], d["C"], d["bias"], cmin, cmax, d["scale_a"], d["scale_b"],
                        n, d["scale_d"], d["zp_d"])
    np.testing.assert_array_equal(got, exp)


@pytest.mark.parametrize("m,k", ROWS_K)
@pytest.mark.parametrize("packed", ["", "p"])
def test_w8a8_skinny_dynamic(gpu, m, k, packed):
    """f32 results, plain or packed A and B, with zero points beyond 16 bits in some rows."""
    import torch

    g = _gr()
    n = 139
    assert T.routes().tqtr_w8a8_few_row(m, n, k, 1, bool(packed))
    rng = np.random.default_rng(m * k)
    A = rng.integers(-128, 128, size=(m, k), dtype=np.int64).astype(np.int8)
    B = rng.integers(-127, 128, size=(n, k), dtype=np.int64).astype(np.int8)
    sa = rng.uniform(0.01, 0.1, m).astype(np.float32)
    za = rng.integers(-128, 128, m).astype(np.int32)
    za[::5] = 40000 - 70000 * (np.arange(len(za[::5])) % 2)
    sb = rng.uniform(0.001, 0.01, n).astype(np.float32)
    bias = rng.standard_normal(n).astype(np.float32)
    dA, dB = g.dev(A), g.dev(B)
    if packed:
        pA = torch.empty(m * k, dtype=torch.uint8, device="cuda:0")
        pB = torch.empty(n * k, dtype=torch.uint8, device="cuda:0")
        g.lib().fn("w8dynp", "run_a_pack")(m, k, k, k, 0, g.dp(dA), pA.data_ptr())
        g.lib().fn("w8dynp", "run_bt_pack")(n, k, k, k, 0, g.dp(dB), pB.data_ptr())
        dA, dB = pA, pB
    dsa, dza, dsb, dbias = g.dev(sa), g.dev(za), g.dev(sb), g.dev(bias)
    dD = torch.zeros((m, n), dtype=torch.float32, device="cuda:0")
    p = g._mod.QAI8DXPQSI8CXPParams(dsa.data_ptr(), dza.data_ptr(), dsb.data_ptr())
    g.lib().fn("w8dyn" + packed, "run")(m, n, k, g.dp(dA), k, 0, g.dp(dB), k, 0, None, n, g.dp(dD),
                                        n, g.dp(dbias), -np.inf, np.inf, ctypes.byref(p))
    got = dD.cpu().numpy()
    exp = T.oracle_w8a8dyn(A, B, bias, -np.inf, np.inf, sa, za, sb)
    np.testing.assert_array_equal(got.view(np.uint32), exp.view(np.uint32))


@pytest.mark.parametrize("m", [5, 20])
def test_w8a8_skinny_strides(gpu, m):
    """Row strides larger than the rows; nothing written outside the results."""
    import torch

    g = _gr()
    n, k = 70, 1200
    assert T.routes().tqtr_w8a8_few_row(m, n, k, 0, 0)
    lda, ldb, ldc, ldd = k + 16, k + 48, n + 3, n + 5
    d = T.gen_w8a8(m, n, k, seed=m, with_c=True)
    A = np.full((m, lda), 99, np.int8)
    A[:, :k] = d["A"]
    B = np.full((n, ldb), 55, np.int8)
    B[:, :k] = d["B"]
    C = np.full((m, ldc), 1 << 20, np.int32)
    C[:, :n] = d["C"]
    dA, dB, dC, dbias, dsb = g.dev(A), g.dev(B), g.dev(C), g.dev(d["bias"]), g.dev(d["scale_b"])
    dD = torch.full((m + 1, ldd), 77, dtype=torch.int8, device="cuda:0")
    p = g.w8a8_params(d, dsb)
    g.lib().fn("w8a8", "run")(m, n, k, g.dp(dA), lda, 0, g.dp(dB), ldb, 0, g.dp(dC), ldc, g.dp(dD),
                              ldd, g.dp(dbias), -128, 127, ctypes.byref(p))
    got = dD.cpu().numpy()
    exp = T.oracle_w8a8(d["A"], d["B"], d["C"], d["bias"], -128, 127, d["scale_a"], d["scale_b"],
                        n, d["scale_d"], d["zp_d"])
    np.testing.assert_array_equal(got[:m, :n], exp)
    assert (got[m:] == 77).all() and (got[:m, n:] == 77).all()
