"""The fused expansion + depthwise launch with its depthwise stage on the matrix cores, which small tiles take (up to 128 units of
four output pixels x four channels per workgroup, in groups of sixteen outputs x sixteen channels, one a wave or more than half full),
and tiles just beyond that: bit for bit the oracle's chain, at groups of sixteen output pixels that end early, several chunks and
groups per wave, waves without work, and weights whose differences from their zero point leave int8 on either side."""
import numpy as np
import pytest

import oracle_lib as O
from harness import diff_report, eden, synth, to_eh_requant
from test_gpu_block import oracle_block

pytestmark = pytest.mark.gpu
SEED = 0xB10D

CASES = [
    # n, h, w, cin, c, stride, rows, cols, depthwise zp_w, on the matrix cores
    (1, 3, 3, 8, 16, 1, 1, 1, 128, True),      # one output per workgroup, one chunk: three waves without work
    (2, 9, 7, 16, 48, 1, 3, 5, 0, True),       # fifteen pixels; differences up to 255
    (1, 9, 7, 24, 48, 2, 4, 4, 255, True),     # sixteen pixels; differences down to -255
    (1, 11, 13, 32, 80, 1, 3, 7, 100, True),   # two groups, the second of five; a range that ends inside a block
    (1, 16, 16, 40, 32, 1, 8, 8, 150, True),   # 128 units: four groups
    (1, 16, 17, 40, 32, 1, 8, 9, 150, False),   # 192 units: the vector form
    (3, 8, 8, 160, 96, 2, 2, 3, 127, False),    # five reduction steps; six groups of six outputs: the vector form
    (2, 8, 8, 24, 64, 1, 2, 4, 127, True),     # eight outputs, half a group: the matrix form with up to four chunks to a workgroup
    (2, 8, 8, 24, 64, 1, 3, 3, 127, True),     # nine
    (1, 5, 6, 16, 16, 1, 5, 6, 90, True),      # the whole image in one workgroup
]


@pytest.mark.parametrize("per_channel", [False, True], ids=["tensor", "channel"])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(str(v) for v in c))
def test_matrix_form_matches_oracle(case, per_channel):
    n, h, w, cin, c, stride, rows, cols, zp_w, matrix = case
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
    assert eden.conv_dw_block_applies(pw, dw) and eden.conv_dw_block_tile(pw, dw, rows, cols)[3] == matrix
    d_x, d_o = eden.DeviceBuffer(host=x), eden.DeviceBuffer(nbytes=n * ho * wo * c)
    eden.conv_dw_block_run(pw, dw, d_x, d_o, e1, e2, rows, cols)
    got = d_o.download((n, ho, wo, c))
    assert np.array_equal(got, want), diff_report(got, want)
    assert want.std() > 1
