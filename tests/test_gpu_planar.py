"""Planar tensors: the one-pass transposition with channel padding, and kernels that write planar outputs themselves, at the
edges of their tiles, against the CPU oracle."""
import numpy as np
import pytest

import oracle_lib as O
from harness import diff_report, eden, gpu_conv, gpu_deconv, synth, to_eh_requant

pytestmark = pytest.mark.gpu
SEED = 0xEDE2 + 16 * 31

CASES = [
    # n, c, h, w, cout, k, stride, groups
    (2, 13, 9, 7, 19, 3, 1, 1),         # channels padded 13 -> 16, odd plane
    (3, 33, 11, 13, 17, 1, 1, 1),       # padded 33 -> 48
    (1, 70, 5, 3, 40, 3, 2, 1),         # more than 32 padded channels, fifteen pixels
    (2, 32, 31, 33, 40, 1, 1, 1),       # one tap
    (5, 64, 30, 30, 24, 3, 1, 1),       # patch kernel
    (2, 3, 33, 31, 37, 3, 2, 1),        # three channels
    (2, 3, 40, 36, 20, 3, 2, 1),        # ... below 32 output channels
    (2, 4, 30, 31, 33, 7, 2, 1),        # kernel rows
    (4, 64, 40, 40, 100, 5, 2, 1),      # tiled kernels
    (2, 64, 13, 13, 48, 3, 1, 4),       # groups: planes behind one another
    (2, 6, 9, 9, 6, 3, 1, 2),           # grouped and padded
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(str(v) for v in c))
def test_planar_conv(case):
    n, c, h, w, cout, k, stride, groups = case
    s = O.conv_shape(n, c, h, w, cout, k, k, stride=(stride, stride), pad=(k // 2,) * 4, groups=groups)
    red = c // groups * k * k
    x, wt = synth.fill_u8((n, c, h, w), SEED + c), synth.fill_u8((cout, c // groups, k, k), SEED + cout)
    b = synth.fill_i32((cout,), SEED + 2, -1000, 1000)
    q = O.make_quant(0.02, 131, 0.005, 126, 0.02 * 0.005 * 74 * 74 * red ** 0.5 / 40, 120)
    want = O.conv2d(x, wt, b, s, q)
    got = gpu_conv(x, wt, b, s, to_eh_requant(q), layout=eden.NCHW)
    assert np.array_equal(got, want), diff_report(got, want)
    assert want.std() > 4


@pytest.mark.parametrize("case", [(2, 64, 7, 9, 21, 4, 2), (1, 48, 9, 8, 33, 3, 2), (3, 20, 6, 5, 7, 2, 2)], ids=lambda c: "x".join(str(v) for v in c))
def test_planar_deconv(case):
    n, c, h, w, cout, k, stride = case
    s = O.conv_shape(n, c, h, w, cout, k, k, stride=(stride, stride), pad=((k - stride) // 2,) * 4)
    x, wt = synth.fill_u8((n, c, h, w), SEED + 11), synth.fill_u8((c, cout, k, k), SEED + 12)
    b = synth.fill_i32((cout,), SEED + 13, -1000, 1000)
    q = O.make_quant(0.02, 121, 0.005, 133, 0.02 * 0.005 * 74 * 74 * (c * 4) ** 0.5 / 40, 128)
    want, got = O.deconv2d(x, wt, b, s, q), gpu_deconv(x, wt, b, s, to_eh_requant(q), layout=eden.NCHW)
    assert np.array_equal(got, want), diff_report(got, want)
    assert want.std() > 4
