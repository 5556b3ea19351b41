"""The fused expansion + depthwise launch with its depthwise stage on the matrix cores, which small tiles take (up to four
units of sixteen outputs x sixteen channels per workgroup, up to eight that are more than half full; fewer with one pair per channel), and tiles just
beyond that: bit for bit the oracle's chain, at groups of sixteen output pixels that end early, several chunks and
groups per wave, waves without work, and weights whose differences from their zero point leave int8 on either side."""
import numpy as np
import pytest

import oracle_lib as O
from harness import diff_report, eden, synth, to_eh_requant
from test_gpu_block import oracle_block

pytestmark = pytest.mark.gpu
SEED = 0xB10D

CASES = [
    # n, h, w, cin, c, stride, rows, cols (0: the library's), depthwise zp_w, on the matrix cores with one pair per tensor / per channel
    (1, 3, 3, 8, 16, 1, 1, 1, 128, True, True),       # one output per workgroup, one chunk: three waves without work
    (2, 9, 7, 16, 48, 1, 3, 5, 0, True, True),        # fifteen pixels; differences up to 255
    (1, 9, 7, 24, 48, 2, 4, 4, 255, True, True),      # sixteen pixels; differences down to -255
    (1, 11, 13, 32, 80, 1, 3, 7, 100, False, False),  # ten units, two groups of five chunks
    (1, 11, 13, 32, 48, 1, 3, 7, 100, True, False),   # six units: two groups, the second of five pixels
    (1, 11, 13, 32, 48, 2, 3, 7, 100, True, True),    # ... at stride 2
    (2, 9, 9, 32, 80, 2, 3, 3, 100, True, True),      # five units of nine pixels; a range that ends inside a block
    (1, 16, 16, 40, 32, 1, 8, 8, 150, True, False),   # eight units: four groups
    (1, 16, 17, 40, 32, 1, 8, 9, 150, False, False),  # ten
    (3, 8, 8, 160, 96, 2, 2, 3, 127, False, False),   # six units of six pixels
    (3, 8, 8, 160, 64, 2, 2, 3, 127, True, True),     # four of them, behind five reduction steps
    (2, 8, 8, 24, 64, 1, 2, 4, 127, True, False),     # four units of eight pixels, half a group
    (2, 8, 8, 24, 64, 2, 2, 4, 127, True, True),      # ... at stride 2
    (2, 8, 8, 24, 64, 1, 3, 3, 127, True, False),     # of nine
    (1, 5, 6, 16, 16, 1, 5, 6, 90, True, True),       # the whole image in one workgroup
    (4, 28, 28, 32, 128, 2, 0, 0, 100, True, True),   # the library's own tile at stride 2: fifteen pixels, one channel block
    (6, 31, 29, 24, 144, 2, 0, 0, 0, True, True),     # ... ten, ranges of four chunks and one of one
    (3, 39, 41, 40, 240, 2, 0, 0, 255, True, True),   # ... twelve, two reduction steps, ranges of four chunks and one of three
    (2, 21, 23, 160, 960, 2, 0, 0, 127, True, True),  # ... nine, five steps
]


@pytest.mark.parametrize("per_channel", [False, True], ids=["tensor", "channel"])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(str(v) for v in c))
def test_matrix_form_matches_oracle(case, per_channel):
    n, h, w, cin, c, stride, rows, cols, zp_w = case[:9]
    print("block", case, per_channel, flush=True)
    x, w1 = synth.fill_u8((n, h, w, cin), SEED + h), synth.fill_u8((c, cin, 1, 1), SEED + 1)
    b1, b2 = synth.fill_i32((c,), SEED + 2, -1000, 1000), synth.fill_i32((c,), SEED + 4, -1000, 1000)
    w2 = synth.fill_u8((c, 1, 3, 3), SEED + 3)
    q1 = O.make_quant(0.02, 117, 0.004, 121, 0.03, 5, O.ACT_RELU6, True)
    q2 = O.make_quant(0.03, 5, 0.006, zp_w, 0.4, 128)
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
    assert eden.conv_dw_block_applies(pw, dw) and eden.conv_dw_block_tile(pw, dw, rows, cols)[3] == case[10 if per_channel else 9]
    d_x, d_o = eden.DeviceBuffer(host=x), eden.DeviceBuffer(nbytes=n * ho * wo * c)
    eden.conv_dw_block_run(pw, dw, d_x, d_o, e1, e2, rows, cols)
    got = d_o.download((n, ho, wo, c))
    assert np.array_equal(got, want), diff_report(got, want)
    assert want.std() > 1
