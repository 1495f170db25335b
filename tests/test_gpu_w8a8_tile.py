"""W8A8 large-tile kernel (outputs of more than one round of 128 x 128 tiles): bit-exact against the
CPU oracle for 256 x 256 and 128 x 128 tiles, one row and one channel past whole tiles, k of one
16-byte chunk, of part of a stage and of more stages than the ring's two, static (C, clamps, shared
scale) and per-row dynamic (f32, f16) with zero points beyond 16 bits, plain and packed operands, row
strides. Each test asserts the tile that its call takes."""

import ctypes

import numpy as np
import pytest

import tqt_testlib as T
from test_gpu_w8a8_dyn import check as check_dyn

pytestmark = pytest.mark.gpu


def _gr():
    import gpu_run

    return gpu_run


def _gen(m, n, k, seed, with_c=False):
    d = T.gen_w8a8(m, n, k, seed=seed, with_c=with_c)
    # an output scale that spreads the results over most of int8
    d["scale_d"] = np.float32(0.02 * 0.0055 * 50 * 73 * np.sqrt(k) / 40)
    return d


def _run(d, kind="w8a8", lda=None, ldd=None, cmin=-128, cmax=127):
    import torch

    g = _gr()
    (m, k), n = d["A"].shape, d["B"].shape[0]
    lda, ldd = lda or k, ldd or n
    A = np.full((m, lda), 3, np.int8)
    A[:, :k] = d["A"]
    dA, dB, dC, dbias = g.dev(A), g.dev(d["B"]), g.dev(d["C"]), g.dev(d["bias"])
    dsb = g.dev(d["scale_b"])
    if kind != "w8a8":
        pB = torch.empty(n * k, dtype=torch.uint8, device="cuda:0")
        g.lib().fn(kind, "run_bt_pack")(n, k, k, k, 0, g.dp(dB), pB.data_ptr())
        dB = pB
    if kind == "w8a8p":
        pA = torch.empty(m * k, dtype=torch.uint8, device="cuda:0")
        g.lib().fn(kind, "run_a_pack")(m, k, k, k, 0, g.dp(dA), pA.data_ptr())
        dA = pA
    dD = torch.full((m + 1, ldd), 77, dtype=torch.int8, device="cuda:0")
    p = g.w8a8_params(d, dsb)
    g.lib().fn(kind, "run")(m, n, k, g.dp(dA), lda, 0, g.dp(dB), k, 0, g.dp(dC), n, g.dp(dD), ldd,
                            g.dp(dbias), cmin, cmax, ctypes.byref(p))
    got = dD.cpu().numpy()
    assert (got[m:] == 77).all() and (got[:m, n:] == 77).all()
    return np.ascontiguousarray(got[:m, :n])


def _oracle(d, cmin=-128, cmax=127):
    return T.oracle_w8a8(d["A"], d["B"], d["C"], d["bias"], cmin, cmax, d["scale_a"], d["scale_b"],
                         int(d.get("qcb", d["B"].shape[0])), d["scale_d"], d["zp_d"])


S, B = T.W8A8_TILE_128X128, T.W8A8_TILE_256X256

# (m, n, k, tile)
SHAPES = [(2049, 2049, 16, S), (2100, 2051, 144, S), (1153, 4208, 656, S), (3841, 4097, 272, S),
          (3841, 1030, 1280, S), (1540, 8000, 656, B), (3900, 8000, 1040, B)]


def _tile(m, n, k, dyn=False):
    assert not T.routes().tqtr_w8a8_few_row(m, n, k, dyn, 0)
    return T.routes().tqtr_w8a8_tile(m, n, k, dyn)


@pytest.mark.parametrize("m,n,k,tile", SHAPES)
def test_w8a8_tile(gpu, m, n, k, tile):
    assert _tile(m, n, k) == tile
    d = _gen(m, n, k, seed=m + k, with_c=k < 700)
    cmin, cmax = (-128, 127) if m % 2 else (-90, 100)
    np.testing.assert_array_equal(_run(d, cmin=cmin, cmax=cmax), _oracle(d, cmin, cmax))


@pytest.mark.parametrize("kind", ["w8a8pb", "w8a8p"])
@pytest.mark.parametrize("m,n,k,tile", [(2100, 2051, 144, S), (3841, 4097, 272, S),
                                        (1153, 4208, 656, S), (1540, 8000, 656, B)])
def test_w8a8_tile_packed(gpu, kind, m, n, k, tile):
    assert _tile(m, n, k) == tile
    d = _gen(m, n, k, seed=m + n)
    np.testing.assert_array_equal(_run(d, kind), _oracle(d))


def test_w8a8_tile_strides_and_shared_scale(gpu):
    assert _tile(2177, 2200, 400) == S
    d = _gen(2177, 2200, 400, seed=3)
    d["qcb"] = 1
    np.testing.assert_array_equal(_run(d, lda=432, ldd=2211), _oracle(d))


@pytest.mark.parametrize("packed", [False, True], ids=["plain", "packed"])
@pytest.mark.parametrize("f16", [False, True], ids=["f32", "f16"])
@pytest.mark.parametrize("m,n,k,tile", [(2050, 2052, 208, S), (3970, 4100, 144, S),
                                        (3600, 1030, 656, S), (1540, 8000, 1040, B)])
def test_w8a8_tile_dynamic(gpu, shim, f16, packed, m, n, k, tile):
    assert _tile(m, n, k, True) == tile
    rng = np.random.default_rng(m + k)
    zp = rng.integers(-128, 128, m).astype(np.int32)
    zp[[5, m - 1]] = [40000, -2 ** 31]
    d = dict(A=rng.integers(-128, 128, (m, k)).astype(np.int8),
             B=rng.integers(-127, 128, (n, k)).astype(np.int8),
             scale_a=rng.uniform(0.01, 0.05, m).astype(np.float32), zp_a=zp,
             scale_b=rng.uniform(0.001, 0.01, n).astype(np.float32),
             bias=rng.uniform(-1, 1, n).astype(np.float16).astype(np.float32))
    check_dyn(shim, d, f16, packed)
