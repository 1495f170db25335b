"""Channel-first implicit convolution kernel (igemmcf, plain weights, 1 / 9 / 25 taps, channels a
multiple of 16): bit-exact against the oracle where it can go wrong - planes whose size is no
multiple of 4 (every channel's rows then start at another byte of a dword), tiles that cross images,
tiles past the last pixel, the input's last bytes, strides, dilation, padding wider than the window,
output rows wholly in the padding, channel blocks of 1 to 9 chunks of 16, ragged output channels,
groups and pixel windows."""

import numpy as np
import pytest

from test_gpu_conv_cf import cf_problem, oracle_cf, run_cf

pytestmark = pytest.mark.gpu

# (IC, OC, ID, IH, IW, groups, kernel, stride, pad, dilation)
CASES = [
    (16, 8, 1, 3, 3, 1, (1, 3, 3), (1, 1, 1), (0, 1, 1), (1, 1, 1)),
    (32, 70, 3, 7, 7, 1, (1, 3, 3), (1, 1, 1), (0, 1, 1), (1, 1, 1)),
    (144, 40, 2, 15, 15, 1, (1, 3, 3), (1, 1, 1), (0, 1, 1), (1, 1, 1)),
    (48, 64, 2, 13, 17, 1, (1, 3, 3), (1, 2, 2), (0, 1, 1), (1, 1, 1)),
    (64, 65, 1, 28, 28, 1, (1, 3, 3), (1, 1, 1), (0, 2, 2), (1, 2, 2)),
    (16, 33, 2, 5, 6, 1, (1, 3, 3), (1, 1, 1), (0, 4, 4), (1, 1, 1)),
    (16, 16, 2, 9, 130, 1, (1, 3, 3), (1, 1, 2), (0, 0, 1), (1, 1, 1)),
    (32, 32, 1, 10, 150, 1, (1, 3, 3), (1, 2, 1), (0, 1, 1), (1, 1, 1)),  # wide halo
    (96, 130, 2, 11, 9, 1, (1, 1, 1), (1, 1, 1), (0, 0, 0), (1, 1, 1)),
    (32, 24, 4, 14, 14, 2, (1, 1, 1), (1, 2, 2), (0, 0, 0), (1, 1, 1)),
    (32, 48, 2, 12, 11, 1, (1, 5, 5), (1, 1, 1), (0, 2, 2), (1, 1, 1)),
    (16, 20, 1, 20, 21, 1, (1, 5, 5), (1, 2, 2), (0, 2, 2), (1, 1, 1)),
    (48, 96, 6, 4, 3, 3, (1, 3, 3), (1, 1, 1), (0, 1, 1), (1, 1, 1)),
]


@pytest.mark.parametrize("IC,OC,ID,IH,IW,groups,kern,stride,pad,dil", CASES)
def test_igemmcf_tile(gpu, shim, IC, OC, ID, IH, IW, groups, kern, stride, pad, dil):
    d = cf_problem(IC, OC, ID, IH, IW, groups, kern, stride, pad, dil, seed=IC + OC + IH)
    for grp in range(groups):
        np.testing.assert_array_equal(run_cf(shim, d, grp, "igemmcf", False), oracle_cf(d, grp))


def test_igemmcf_tile_windows(gpu, shim):
    """A window of pixels that starts inside an image and crosses into the next."""
    d = cf_problem(32, 48, 3, 9, 11, 1, (1, 3, 3), (1, 1, 1), (0, 1, 1), (1, 1, 1), seed=7)
    for n_idx, n in ((0, 65), (61, 130), (d["N"] - 5, 5)):
        got = run_cf(shim, d, 0, "igemmcf", False, n_idx, n)
        np.testing.assert_array_equal(got, oracle_cf(d, 0, n_idx, n))
