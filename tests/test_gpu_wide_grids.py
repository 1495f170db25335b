"""Calls of so many channels that a workgroup per 16 of them (or per 64 x 64 outputs) would pass the
2^32 work-items of a grid dimension: they run, on the kernels with larger tiles or one thread per
output. Every channel shares one row of weights (row stride 0) and one scale, so that the operands are
small and every result is the same."""

import ctypes

import numpy as np
import pytest

import tqt_testlib as T

pytestmark = pytest.mark.gpu


def _gr():
    import gpu_run

    return gpu_run


def _all_equal(dD, want):
    assert dD.min().item() == dD.max().item() == want


@pytest.mark.parametrize("m,n,k", [(1, (1 << 27) + 20, 16), (1, (1 << 30) + 20, 33)],
                         ids=["few-row", "edge"])
def test_w8a8_wide(gpu, m, n, k):
    import torch

    g = _gr()
    d = T.gen_w8a8(m, 1, k, seed=k)
    d["scale_d"] = np.float32(0.5)
    exp = T.oracle_w8a8(d["A"], d["B"], None, None, -128, 127, d["scale_a"], d["scale_b"], 1,
                        d["scale_d"], d["zp_d"])
    dA, dB, dsb = g.dev(d["A"]), g.dev(d["B"]), g.dev(d["scale_b"])
    dD = torch.full((n,), 99, dtype=torch.int8, device="cuda:0")
    p = g.w8a8_params(dict(d, qcb=1), dsb)
    g.lib().fn("w8a8", "run")(m, n, k, g.dp(dA), k, 0, g.dp(dB), 0, 0, None, n, g.dp(dD), n, None,
                              -128, 127, ctypes.byref(p))
    _all_equal(dD, int(exp[0, 0]))


def test_w4a8_wide(gpu):
    import torch

    g = _gr()
    m, n, k = 1, (1 << 28) + 20, 32
    d = T.gen_w4a8(m, 1, k, seed=1, with_bias=False)
    exp = T.oracle_w4a8(d["A"], d["Bp"], None, None, -np.inf, np.inf, d["scale_a"], d["zp_a"],
                        d["scale_b"])
    dA, dB, dsa, dza = g.dev(d["A"]), g.dev(d["Bp"]), g.dev(d["scale_a"]), g.dev(d["zp_a"])
    dsb = torch.full((n,), float(d["scale_b"][0]), dtype=torch.float32, device="cuda:0")
    dD = torch.full((n,), 9e9, dtype=torch.float32, device="cuda:0")
    p = g._mod.QAI8DXQSI4CXParams(dsa.data_ptr(), dza.data_ptr(), dsb.data_ptr())
    g.lib().fn("w4a8", "run")(m, n, k, g.dp(dA), k, 0, g.dp(dB), 0, 0, None, n, g.dp(dD), n, None,
                              -np.inf, np.inf, ctypes.byref(p))
    _all_equal(dD, float(exp[0, 0]))


def test_w4a16_wide(gpu):
    import torch

    g = _gr()
    m, n, k, bl = 1, (1 << 28) + 20, 128, 64
    d = T.gen_w4a16(m, 1, k, bl=bl, seed=2, with_bias=False)
    d["A16"][:] = T.f16_bits(np.round(T.bits_f16(d["A16"]).astype(np.float32)))  # exact sums
    d["S16"][:] = T.f16_bits(np.float32(0.125))
    q = np.empty(k)
    q[0::2] = (d["Bp"][0] & 15).astype(np.float64) - 8
    q[1::2] = (d["Bp"][0] >> 4).astype(np.float64) - 8
    want = float(T.bits_f16(d["A16"])[0].astype(np.float64) @ q) * 0.125
    dA, dB, dS = g.dev(d["A16"].view(np.int16)), g.dev(d["Bp"]), g.dev(d["S16"].view(np.int16))
    dD = torch.full((n,), 9e9, dtype=torch.float32, device="cuda:0")
    g.lib().fn("w4a16f", "run")(m, n, k, bl, g.dp(dA), k, 0, g.dp(dB), 0, 0, g.dp(dS), 0, None, n,
                                g.dp(dD), n, None, -np.inf, np.inf)
    _all_equal(dD, want)
