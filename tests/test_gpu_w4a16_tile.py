"""W4A16 large-tile kernel (many rows, scale blocks that are any multiple of 32, k beyond the
register kernel): against the CPU oracle and exact f64 math at the edges of its tiles, at stage
remainders, with every block width class (32, 64, 96, 128, one block over the whole of k), odd scale
strides (a scale is then the upper half of its dword in every other row), C, clamps, strides,
infinities, and f16 and f32 results; and every instance (tile, block class, compensation) over more
stages than its ring holds. Each test asserts that its call takes the tiles it names."""

import numpy as np
import pytest

import tqt_testlib as T
from test_gpu_parity import check_w4a16

pytestmark = pytest.mark.gpu


def _gr():
    import gpu_run

    return gpu_run


def _run_f32(d, lo=-np.inf, hi=np.inf, pad_d=0, pad_s=0):
    import torch

    g = _gr()
    A16, Bp, S16, bl = d["A16"], d["Bp"], d["S16"], d["bl"]
    (m, k), n, nb = A16.shape, Bp.shape[0], S16.shape[1]
    S = np.full((n, nb + pad_s), 0x7E00, np.uint16)  # NaN beyond the blocks
    S[:, :nb] = S16
    dA, dB, dS = g.dev(A16.view(np.int16)), g.dev(Bp), g.dev(S.view(np.int16))
    C = None if d["C16"] is None else T.bits_f16(d["C16"]).astype(np.float32)
    bias = None if d["bias16"] is None else T.bits_f16(d["bias16"]).astype(np.float32)
    dC, dbias = g.dev(C), g.dev(bias)
    dD = torch.full((m + 1, n + pad_d), 12345.0, dtype=torch.float32, device="cuda:0")
    g.lib().fn("w4a16f", "run")(m, n, k, bl, g.dp(dA), k, 0, g.dp(dB), k, 0, g.dp(dS), nb + pad_s,
                                g.dp(dC), n, g.dp(dD), n + pad_d, g.dp(dbias), lo, hi)
    got = dD.cpu().numpy()
    assert (got[m:] == 12345.0).all() and (got[:m, n:] == 12345.0).all()
    return np.ascontiguousarray(got[:m, :n])


def _exact(d):
    """f64 sums and the sum of the terms' magnitudes, C and bias included."""
    a = T.bits_f16(d["A16"]).astype(np.float64)
    bl = d["bl"]
    q = np.empty((d["Bp"].shape[0], a.shape[1]), np.float64)
    q[:, 0::2] = (d["Bp"] & 15).astype(np.float64) - 8
    q[:, 1::2] = (d["Bp"] >> 4).astype(np.float64) - 8
    w = q * np.repeat(T.bits_f16(d["S16"]).astype(np.float64), bl, axis=1)
    v, mag = a @ w.T, np.abs(a) @ np.abs(w).T
    for x in (d["C16"], d["bias16"]):
        if x is not None:
            f = T.bits_f16(x).astype(np.float64)
            v, mag = v + f, mag + np.abs(f)
    return v, mag


def _check_f32(got, d, lo=-np.inf, hi=np.inf):
    """Each block's products and sum round at most bl times (exact products), its scaled value and
    the accumulation once each, and C, bias and the k groups a few times more: (bl + k / bl + 16)
    roundings of 2^-24 of the terms' magnitude."""
    v, mag = _exact(d)
    k = d["A16"].shape[1]
    bound = (d["bl"] + k / d["bl"] + 16) * 2.0 ** -24 * mag
    v = np.clip(v, lo, hi)
    bad = np.abs(got.astype(np.float64) - v) > bound
    assert not bad.any(), "%d of %d outputs out of bounds" % (bad.sum(), bad.size)


# (m, n, k, bl)
SHAPES = [
    (65, 65, 160, 32),       # one row and channel past whole tiles
    (300, 400, 32, 32),      # one block of k
    (520, 130, 96, 96),
    (97, 130, 864, 32),      # k % 128 == 96
    (129, 65, 160, 32),
    (65, 129, 2880, 96),     # blocks that straddle stages
    (129, 257, 1152, 128),   # odd scale stride (9)
    (100, 1000, 4416, 64),   # k beyond the register kernel, odd scale stride (69)
    (300, 1001, 1056, 1056),  # one block over all of k, odd channels
    (700, 2100, 544, 32),
    (1030, 4100, 320, 64),
    (2100, 2100, 256, 128),
    (100, 2050, 8192, 32),   # compensated, another kernel's shape otherwise
]

# (m, n, k, bl, f32 results, kernel, blocks per compensation): every instance of the kernel, more stages
# of 128 k than its ring holds, and a part of one where another kernel does not ask for whole ones
INSTANCES = [
    (2050, 3000, 1056, 32, 0, T.W4A16_TILE_128X256, 0),
    (2050, 1001, 1056, 32, 0, T.W4A16_TILE_128X128, 0),
    (200, 5000, 1056, 32, 0, T.W4A16_TILE_64X128, 0),
    (65, 67, 1056, 32, 0, T.W4A16_TILE_32X64, 0),
    (2050, 2052, 1088, 64, 0, T.W4A16_TILE_128X256, 0),
    (1000, 4000, 2752, 64, 0, T.W4A16_TILE_128X128, 0),
    (200, 5000, 1088, 64, 0, T.W4A16_TILE_64X128, 0),
    (65, 67, 1088, 64, 0, T.W4A16_TILE_32X64, 0),
    (2050, 2052, 1152, 128, 1, T.W4A16_TILE_128X256, 0),
    (1000, 4000, 2944, 128, 1, T.W4A16_TILE_128X128, 0),
    (200, 5000, 1152, 128, 1, T.W4A16_TILE_64X128, 0),
    (65, 67, 1152, 128, 1, T.W4A16_TILE_32X64, 0),
    (200, 5000, 1056, 32, 1, T.W4A16_TILE_64X128, 1),
    (65, 67, 1056, 32, 1, T.W4A16_TILE_32X64, 1),
    (200, 5000, 2080, 32, 1, T.W4A16_TILE_64X128, 2),
    (65, 67, 2080, 32, 1, T.W4A16_TILE_32X64, 2),
    (200, 5000, 1024, 32, 0, T.W4A16_TILE_64X128, 1),
    (65, 1500, 1024, 32, 0, T.W4A16_TILE_32X64, 1),
    (200, 5000, 2048, 32, 0, T.W4A16_TILE_64X128, 2),
    (65, 1500, 2048, 32, 0, T.W4A16_TILE_32X64, 2),
    (200, 5000, 3584, 32, 0, T.W4A16_TILE_64X128, 4),
    (65, 1500, 3584, 32, 0, T.W4A16_TILE_32X64, 4),
    (200, 5000, 1152, 32, 0, T.W4A16_TILE_64X128, 8),
    (65, 1500, 6656, 32, 0, T.W4A16_TILE_32X64, 8),
]


def test_w4a16_instances_covered():
    """The list above holds every instance that the rules can pick."""
    tiles = (T.W4A16_TILE_128X256, T.W4A16_TILE_128X128, T.W4A16_TILE_64X128, T.W4A16_TILE_32X64)
    want = {(32, 0, t, 0) for t in tiles}
    want |= {(64, f32, t, 0) for t in tiles for f32 in (0, 1)}
    want |= {(32, 0, t, c) for t in tiles[2:] for c in (1, 2, 4, 8)}
    want |= {(32, 1, t, c) for t in tiles[2:] for c in (1, 2)}
    assert {(32 if bl % 64 else 64, f32, t, c) for _, _, _, bl, f32, t, c in INSTANCES} == want


@pytest.mark.parametrize("m,n,k,bl,f32,kernel,comp", INSTANCES)
def test_w4a16_tile_instance(gpu, shim, m, n, k, bl, f32, kernel, comp):
    """Against f64 math: _check_f32's bound, and for f16 results half a unit in the last place more."""
    assert T.w4a16_route(m, n, k, bl, f32) == (kernel, comp)
    d = T.gen_w4a16(m, n, k, bl=bl, seed=m + n + k, with_c=bool(m & 1), with_bias=bool(n & 1))
    if f32:
        _check_f32(_run_f32(d), d)
        return
    got = T.bits_f16(_gr().run_w4a16(shim, d, 0xFBFF, 0x7BFF)).astype(np.float64)
    v, mag = _exact(d)
    v = np.clip(v, -65504.0, 65504.0)
    bound = (bl + k / bl + 16) * 2.0 ** -24 * mag + 2.0 ** -11 * np.abs(v) + 2.0 ** -25
    bad = np.abs(got - v) > bound
    assert not bad.any(), "%d of %d outputs out of bounds" % (bad.sum(), bad.size)


@pytest.mark.parametrize("m,n,k,bl", SHAPES)
def test_w4a16_tile_f32(gpu, m, n, k, bl):
    assert T.w4a16_route(m, n, k, bl, 1, k // bl + m % 2)[0] >= T.W4A16_TILE_128X256
    d = T.gen_w4a16(m, n, k, bl=bl, seed=m + n + k, with_c=bool(m & 1), with_bias=bool(n & 1))
    lo, hi = (-np.inf, np.inf) if m % 2 else (-3.0, 4.0)
    _check_f32(_run_f32(d, lo, hi, pad_d=n % 3, pad_s=(m % 2)), d, lo, hi)


@pytest.mark.parametrize("m,n,k,bl", SHAPES)
def test_w4a16_tile_f16(gpu, shim, m, n, k, bl):
    assert T.w4a16_route(m, n, k, bl, 0)[0] >= T.W4A16_TILE_128X256
    d = T.gen_w4a16(m, n, k, bl=bl, seed=m * 3 + n + k, with_c=bool(m & 1), with_bias=bool(n & 1))
    lo, hi = (-65504.0, 65504.0) if m % 2 else (-2.0, 2.5)
    cmin, cmax = int(T.f16_bits(lo)), int(T.f16_bits(hi))
    got = _gr().run_w4a16(shim, d, cmin, cmax)
    exp = T.oracle_w4a16(d["A16"], d["Bp"], d["S16"], bl, d["C16"], d["bias16"], cmin, cmax)
    check_w4a16(got, exp, d, (lo, hi))


@pytest.mark.parametrize("bl,k,comp", [(32, 1056, 1), (32, 2080, 2), (64, 1088, 0)])
@pytest.mark.parametrize("m,n", [(100, 196), (200, 5000)], ids=["32x64", "64x128"])
def test_w4a16_tile_infinity(gpu, m, n, bl, k, comp):
    """An infinite activation gives infinite results of its sign, NaN where its weight is 0 (as the
    oracle's order of operations does), also through the compensated accumulators, and leaves the
    other rows alone."""
    tile = T.W4A16_TILE_32X64 if m == 100 else T.W4A16_TILE_64X128
    assert T.w4a16_route(m, n, k, bl, 1) == (tile, comp)
    d = T.gen_w4a16(m, n, k, bl=bl, seed=9)
    d["A16"][7, 100] = 0x7C00
    d["A16"][9, 1000] = 0xFC00
    got = _run_f32(d)
    for row, byte, sign in ((7, 50, 1), (9, 500, -1)):
        q = (d["Bp"][:, byte] & 15).astype(np.int32) - 8
        assert np.isnan(got[row, q == 0]).all()
        assert (got[row, q > 0] == sign * np.inf).all() and (got[row, q < 0] == -sign * np.inf).all()
    rest = np.ones(m, bool)
    rest[[7, 9]] = False
    assert np.isfinite(got[rest]).all()


@pytest.mark.parametrize("m,n,k,comp,bound", [(256, 4096, 1024, 1, 6.8e-8),
                                              (256, 4096, 2048, 2, 7.2e-8),
                                              (256, 4096, 4096, 4, 8.0e-8),
                                              (300, 2050, 8192, 8, 9.5e-8),
                                              (1000, 1040, 640, 8, 8.3e-8)])
def test_w4a16_tile_f16_sums(gpu, shim, m, n, k, comp, bound):
    """f16 results keep the sums of 32-wide blocks as exact as the chunk-stream and register kernels do.
    C cancels all but the last bits of each sum, so that its error shows beside the 11 bits of the
    result (whose own rounding, at most 2^-12 of a difference of at most 2^-11 of the sum, is part of
    it): of the sums' rms, the chunk-stream kernel is off by 6.0e-8 at k 1024, 6.5e-8 at 2048, 7.4e-8 at
    4096 and 9.0e-8 at 8192, plain f32 accumulators by 8.8e-8, 1.1e-7, 1.5e-7 and 2.1e-7. The bounds lie
    a tenth above the former."""
    kernel, got = T.w4a16_route(m, n, k, 32, 0)
    assert kernel >= T.W4A16_TILE_128X256 and got == comp
    d = T.gen_w4a16(m, n, k, bl=32, seed=k, with_bias=False)
    v, _ = _exact(d)
    d["C16"] = T.f16_bits(-v)
    out = T.bits_f16(_gr().run_w4a16(shim, d, 0xFBFF, 0x7BFF)).astype(np.float64)
    left = v + T.bits_f16(d["C16"]).astype(np.float64)
    err = np.sqrt(np.mean((out - left) ** 2) / np.mean(v ** 2))
    assert err <= bound, err
