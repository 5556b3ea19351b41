"""The fused expansion + depthwise launch on tiles whose depthwise stage walks down 16 columns, 8 in two strips of rows or 4 in four:
bit for bit the oracle's chain, at tiles that end past the image on either side, column groups that are partly or wholly past the
tile, ranges of channels that end inside a block, weights whose differences from their zero point fit int8 or leave it on either
side, and depthwise scales in the single-shift forms and beyond them."""
import numpy as np
import pytest

import oracle_lib as O
from harness import diff_report, eden, synth, to_eh_requant
from test_gpu_block import oracle_block

pytestmark = pytest.mark.gpu
SEED = 0x3A1C

CASES = [
    # n, h, w, cin, c, stride, rows, cols, depthwise zp_w, depthwise output scale
    (24, 28, 28, 24, 144, 1, 0, 0, 128, 0.4),    # the tile chosen here; differences fit int8
    (1, 230, 205, 8, 64, 1, 0, 0, 100, 0.4),     # ... of an image of many tiles either way
    (1, 300, 290, 8, 128, 2, 0, 0, 100, 0.4),
    (2, 23, 37, 24, 144, 1, 8, 16, 0, 0.4),      # whole column groups; differences up to 255
    (1, 23, 37, 40, 240, 2, 5, 13, 255, 0.4),    # an odd number of rows: 16 columns only; differences down to -255
    (2, 17, 19, 16, 96, 1, 6, 9, 100, 0.4),      # nine columns
    (1, 17, 19, 16, 96, 2, 8, 4, 128, 0.4),      # four columns, a tile as tall as the image
    (1, 9, 40, 8, 112, 1, 9, 20, 90, 0.4),       # the whole height; a last block of sixteen channels
    (3, 14, 14, 96, 576, 1, 7, 14, 120, 0.4),    # three reduction steps
    (2, 15, 15, 160, 192, 1, 8, 15, 0, 0.4),     # five
    (1, 31, 33, 24, 80, 1, 16, 33, 60, 0.0003),  # 0.6, above one half: the two-step form
    (1, 31, 33, 24, 80, 2, 16, 17, 200, 0.00025),
]


@pytest.mark.parametrize("act_min_at_zero_point", [True, False], ids=["relu", "linear"])
@pytest.mark.parametrize("per_channel", [False, True], ids=["tensor", "channel"])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(str(v) for v in c))
def test_walking_depthwise_stage_matches_oracle(case, per_channel, act_min_at_zero_point):
    n, h, w, cin, c, stride, rows, cols, zp_w, scale = case
    print("block", case, per_channel, act_min_at_zero_point, flush=True)
    x, w1 = synth.fill_u8((n, h, w, cin), SEED + h), synth.fill_u8((c, cin, 1, 1), SEED + 1)
    b1, b2 = synth.fill_i32((c,), SEED + 2, -1000, 1000), synth.fill_i32((c,), SEED + 4, -1000, 1000)
    w2 = synth.fill_u8((c, 1, 3, 3), SEED + 3)
    q1 = O.make_quant(0.02, 117, 0.004, 121, 0.03, 5, O.ACT_RELU6, True)
    two_step = scale < 0.001
    if two_step:   # small operands, so that results at such a scale are bytes of their own and not the clamp's
        w2, b2 = (zp_w + w2.astype(np.int16) % 3 - 1).astype(np.uint8), b2 // 20
        q1 = O.make_quant(0.02, 117, 0.004, 121, 0.5, 5, O.ACT_RELU6, True)
    q2 = O.make_quant(0.03, 5, 0.006, zp_w, scale, 128, O.ACT_RELU, act_min_at_zero_point)
    ho, wo = (h + 2 - 3) // stride + 1, (w + 2 - 3) // stride + 1
    d1 = eden.conv_desc(n, cin, h, w, c, 1, 1, layout=eden.NHWC)
    d2 = eden.conv_desc(n, c, h, w, c, 3, 3, stride=(stride, stride), pad=(1, 1, 1, 1), dm=1, layout=eden.NHWC)
    keep = [eden.DeviceBuffer(host=a) for a in (w1, b1, w2, b2)]
    e1, e2 = to_eh_requant(q1), to_eh_requant(q2)
    pw, dw = eden.ConvPlan(d1, keep[0], keep[1], e1), eden.DwConvPlan(d2, keep[2], keep[3], e2)
    want, _ = oracle_block(x, w1, b1, q1, w2, b2, q2, stride, (1, 1, 1, 1))
    if per_channel:   # the tensors' own pair for every channel: the same results through the per-channel code
        for plan, e in ((pw, e1), (dw, e2)):
            plan.set_perchannel(np.full(c, e.multiplier), np.full(c, e.shift))
    assert eden.conv_dw_block_applies(pw, dw) and not eden.conv_dw_block_tile(pw, dw, rows, cols)[3]
    d_x, d_o = eden.DeviceBuffer(host=x), eden.DeviceBuffer(nbytes=n * ho * wo * c)
    eden.conv_dw_block_run(pw, dw, d_x, d_o, e1, e2, rows, cols)
    got = d_o.download((n, ho, wo, c))
    assert np.array_equal(got, want), diff_report(got, want)
    assert not two_step or ((want > 0) & (want < 255)).mean() > 0.9
    assert act_min_at_zero_point or want.std() > 1   # (differences down to -255 leave nothing above the zero point)
