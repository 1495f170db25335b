"""The int8 tile kernel for operands off the 16-byte grid: bit for bit against the CPU oracle at the edges
of its 64 x 64 tiles and 128-byte stages, for every operand form that reaches it ([k, n] and [n, k] B,
implicit convolutions), misaligned base pointers and strides, C, clamps and partial pixel ranges."""

import numpy as np
import pytest

import tqt_testlib as T
from test_gpu_conv_cf import oracle as mx1_oracle
from test_gpu_conv_cf import run_mx1

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1, 201), (65, 63, 127), (64, 66, 129), (3, 4097, 257), (200, 131, 1000), (129, 65, 145)]


def _tiles(form, m, n, k, taps=0):
    return T.routes().tqtr_int8_edge_faster(form, m, n, k, taps)


def _gr():
    import gpu_run

    return gpu_run


def _shifted(g, x, by):
    """x on the device at `by` bytes past an aligned address, followed by nothing."""
    import torch

    t = torch.empty(x.size + by, dtype=torch.int8, device="cuda:0")
    t[by:] = torch.from_numpy(np.ascontiguousarray(x).reshape(-1)).to("cuda:0")
    return t


@pytest.mark.parametrize("m,n,k", SHAPES)
def test_edge_clamp(gpu, m, n, k):
    assert _tiles(T.EDGE_KN_CLAMP, m, n, k)
    A, B, C = T.gen_clamp(m, n, k, seed=m + n + k, with_c=bool(m & 1))
    lo, hi = (-2 ** 31, 2 ** 31 - 1) if n % 2 else (-20000, 30000)
    np.testing.assert_array_equal(_gr().run_clamp(A, B, C, lo, hi), T.oracle_clamp(A, B, C, lo, hi))


@pytest.mark.parametrize("m,n,k", SHAPES)
def test_edge_w8a8(gpu, m, n, k):
    assert _tiles(T.EDGE_NK, m, n, k)
    d = T.gen_w8a8(m, n, k, seed=m + n + k, with_c=bool(m & 1))
    exp = T.oracle_w8a8(d["A"], d["B"], d["C"], d["bias"], -128, 127, d["scale_a"], d["scale_b"], n,
                        d["scale_d"], d["zp_d"])
    np.testing.assert_array_equal(_gr().run_w8a8(d), exp)


# (a multiplier per row: the tiles pay from a longer k)
@pytest.mark.parametrize("m,n,k", [(65, 63, 255) if x == (65, 63, 127) else x for x in SHAPES])
def test_edge_mx1bias(gpu, m, n, k):
    assert _tiles(T.EDGE_KN_REQUANT, m, n, k)
    d = T.gen_mx1bias(m, n, k, seed=m + n + k, with_c=bool(m & 1))
    np.testing.assert_array_equal(run_mx1(d, False), mx1_oracle(d))


@pytest.mark.parametrize("by", [1, 2, 8])
def test_edge_misaligned(gpu, by):
    """Aligned sizes at misaligned bases, C and D with longer rows: nothing is written outside."""
    import torch

    g = _gr()
    m, n, k, ldd = 70, 96, 160, 101
    assert _tiles(T.EDGE_KN_CLAMP, m, n, k)
    A, B, C = T.gen_clamp(m, n, k, seed=by, with_c=True)
    dA, dB, dC = _shifted(g, A, by), _shifted(g, B, by), g.dev(C)
    dD = torch.full((m + 1, ldd), 7, dtype=torch.int32, device="cuda:0")
    g.lib().fn("clamp", "run")(m, n, k, dA.data_ptr() + by, k, 0, dB.data_ptr() + by, n, 0, g.dp(dC),
                               n, g.dp(dD), ldd, -9000, 9000)
    got = dD.cpu().numpy()
    np.testing.assert_array_equal(got[:m, :n], T.oracle_clamp(A, B, C, -9000, 9000))
    assert (got[m:] == 7).all() and (got[:, n:] == 7).all()


@pytest.mark.parametrize("ID,IH,IW,IC,OC,KH,KW,stride,pad,dil,KD", [
    (2, 40, 41, 3, 70, 7, 7, (2, 2), (3, 3), (1, 1), 1),
    (1, 30, 33, 5, 33, 3, 5, (1, 2), (1, 0), (2, 1), 1),
    (4, 9, 9, 24, 65, 3, 3, (1, 1), (1, 1), (1, 1), 2),
    (1, 12, 11, 1, 400, 7, 7, (1, 1), (0, 6), (1, 1), 1),
    (3, 64, 60, 4, 40, 3, 3, (1, 1), (1, 1), (1, 1), 1),   # short k, many outputs
])
@pytest.mark.parametrize("m_idx", [0, 17])
def test_edge_conv(gpu, ID, IH, IW, IC, OC, KH, KW, stride, pad, dil, KD, m_idx):
    d = T.gen_igemmcl(ID, IH, IW, IC, OC, KH, KW, stride=stride, pad=pad, dil=dil, KD=KD,
                      seed=IC + OC + IH)
    out = d["conv"].output_shape
    assert _tiles(T.EDGE_CONV, out[0] * out[1] * out[2] - m_idx, OC, KD * KH * KW * IC, KD * KH * KW)
    exp = T.oracle_igemmcl(d["inp"], d["W"], d["bias"], -128, 127, d["conv"], d["scale_a"],
                           d["scale_b"], OC, d["scale_d"], d["zp_d"])
    got = _gr().run_igemmcl(d, m_idx=m_idx)
    np.testing.assert_array_equal(got[m_idx:], exp[m_idx:])
    assert not got[:m_idx].any()
