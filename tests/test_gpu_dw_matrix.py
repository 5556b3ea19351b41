"""The matrix form of 5x5 and 7x7 depthwise windows at the edges of its tiles, its channel pieces and its launch rule,
against the CPU oracle."""
import numpy as np
import pytest

import oracle_lib as O
from harness import diff_report, eden, gpu_dwconv, synth, to_eh_requant

pytestmark = pytest.mark.gpu
SEED = 0xEDE2 + 16 * 29

CASES = [
    # n, c, h, w, k, stride, (top, bottom, left, right)
    (1, 4, 5, 5, 5, 1, (0, 0, 0, 0)),          # one output, a quarter of a piece
    (2, 20, 9, 9, 7, 1, (3, 3, 3, 3)),         # a tile and one row more, tensor ends inside a piece
    (1, 48, 8, 16, 5, 2, (1, 2, 2, 1)),        # whole tiles at stride 2, unequal padding
    (1, 36, 7, 3, 7, 2, (6, 6, 6, 6)),         # windows wholly in the padding
    (16, 64, 15, 17, 5, 1, (2, 2, 2, 2)),      # the two-strip tiles of 7 rows, three column groups
    (24, 16, 40, 61, 5, 1, (2, 2, 2, 2)),      # one piece per workgroup, seven column groups and one more
    (40, 112, 29, 18, 7, 1, (3, 3, 3, 3)),     # seven pieces: blocks of four and three
    (12, 100, 57, 30, 7, 2, (3, 3, 3, 3)),
]


@pytest.mark.parametrize("zp_w,spread", [(128, 30), (131, 60), (0, 60), (255, 60)])   # differences within int8, slightly beyond, up to 255 of either sign
@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(str(v) for v in c[:6]))
def test_matrix_depthwise(case, zp_w, spread):
    n, c, h, w, k, stride, pad = case
    s = O.conv_shape(n, c, h, w, c, k, k, stride=(stride, stride), pad=pad)
    x = synth.fill_u8((n, c, h, w), SEED + c)
    wt = synth.fill_u8_normal((c, 1, k, k), SEED + k, 128, spread)
    b = synth.fill_i32((c,), SEED + 1, -1000, 1000)
    zp_in = 128 if zp_w in (0, 255) else 93
    q = O.make_quant(0.02, zp_in, 0.005, zp_w, 0.02 * 0.005 * 74 * (160 if zp_w in (0, 255) else spread) * k / 40, 120)
    want = O.dwconv2d(x, wt, b, s, q)
    got = gpu_dwconv(x, wt, b, s, to_eh_requant(q), layout=eden.NHWC)
    assert np.array_equal(got, want), diff_report(got, want)
    assert want.std() > 4


@pytest.mark.parametrize("k", [5, 7])
@pytest.mark.parametrize("scale", [3.0, 1e-7], ids=["left_shift", "long_shift"])   # multipliers outside the single-shift form
def test_matrix_depthwise_two_step_requantization(k, scale):
    n, c, hw = 4, 40, 20
    s = O.conv_shape(n, c, hw, hw, c, k, k, pad=(k // 2,) * 4)
    x, wt = synth.fill_u8((n, c, hw, hw), SEED + 7), synth.fill_u8((c, 1, k, k), SEED + 8)
    b = synth.fill_i32((c,), SEED + 9, -2 ** 30, 2 ** 30) if scale < 1 else synth.fill_i32((c,), SEED + 9, -1000, 1000)
    q = O.make_quant(1.0, 128, 1.0, 128, 1.0 / scale, 128)
    want = O.dwconv2d(x, wt, b, s, q)
    got = gpu_dwconv(x, wt, b, s, to_eh_requant(q), layout=eden.NHWC)
    assert np.array_equal(got, want), diff_report(got, want)
    assert want.std() > 4
