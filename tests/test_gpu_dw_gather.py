"""Channels-last 3x3 depthwise layers whose channels are no multiple of four or have a multiplier, straight from the caller's
tensors: bit for bit the oracle, at a last quad of one, two and three channels, pixels of four channels and just beyond, quads whose
input channels are one, two or four, multipliers that leave a quad's edges inside a channel's repeats, tensors at any byte; pairs that differ
from channel to channel; and not a byte beside the result.  (test_launch_grid.py holds that these cases take the gathering kernel.)"""
import numpy as np
import pytest

import oracle_lib as O
from harness import diff_report, eden, synth
from test_gpu_dw_planar import problem

pytestmark = pytest.mark.gpu
SEED = 0xD6A7

CASES = [
    # n, c, dm, h, w, stride, bytes that the tensors start past a word
    (1, 4, 2, 1, 1, 1, 0),
    (1, 5, 1, 3, 2, 1, 1),
    (2, 6, 1, 7, 5, 2, 2),
    (1, 7, 1, 9, 6, 1, 3),
    (1, 7, 3, 9, 6, 1, 1),
    (2, 4, 4, 8, 9, 2, 0),
    (1, 5, 5, 11, 13, 1, 2),
    (3, 33, 1, 22, 23, 1, 0),
    (2, 50, 2, 15, 14, 2, 3),
    (4, 101, 1, 30, 31, 2, 1),
]


@pytest.mark.parametrize("form", ["u8", "u8pc", "s8", "s8pc"])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(str(v) for v in c))
def test_unpadded_depthwise_matches_oracle(case, form):
    n, c, dm, h, w, stride, lead = case
    print("dw gather", case, form, flush=True)
    cout, pad = c * dm, (1, 1, 1, 1)
    s = O.conv_shape(n, c, h, w, cout, 3, 3, stride=(stride, stride), pad=pad, groups=c, dm=dm)
    ho, wo = O.conv_out_hw(s)
    x, wt, e, pairs, want = problem(s, form, SEED + h, SEED + c, 0.15)
    desc = eden.conv_desc(n, c, h, w, cout, 3, 3, stride=(stride, stride), pad=pad, dm=dm, layout=eden.NHWC | (eden.IO_SIGNED if x.dtype == np.int8 else 0),
                          weight_layout=eden.W_OIHW | (eden.W_SIGNED if wt.dtype == np.int8 else 0))
    d_w, d_b = eden.DeviceBuffer(host=wt), eden.DeviceBuffer(host=synth.fill_i32((cout,), 0xD3A1 + 1, -2000, 2000))
    plan = eden.DwConvPlan(desc, d_w, d_b, e)
    if pairs:
        plan.set_perchannel(*pairs)
    count = n * cout * ho * wo
    padded = np.concatenate([np.full(lead, 7, np.uint8), np.ascontiguousarray(x.transpose(0, 2, 3, 1)).view(np.uint8).ravel()])
    d_x, d_o = eden.DeviceBuffer(host=padded), eden.DeviceBuffer(host=np.full(count + 8, 0xA5, np.uint8))
    plan.run(eden.BufferView(d_x, lead), eden.BufferView(d_o, lead), e)
    whole = d_o.download((count + 8,))
    got = whole[lead:lead + count].reshape(n, ho, wo, cout).transpose(0, 3, 1, 2).view(want.dtype)
    assert np.array_equal(got, want), diff_report(got, want)
    assert (whole[:lead] == 0xA5).all() and (whole[lead + count:] == 0xA5).all()
    assert count < 64 or want.std() > 1
