"""Channels-last 3x3 depthwise layers whose channels are no multiple of four or have a multiplier, straight from the caller's
tensors: bit for bit the oracle, at a last quad of one, two and three channels, pixels of four channels and just beyond, quads whose
input channels are one, two or four, multipliers that leave a quad's edges inside a channel's repeats, tensors at any byte."""
import numpy as np
import pytest

import oracle_lib as O
from harness import diff_report, eden, synth, to_eh_requant

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


@pytest.mark.parametrize("form", ["u8", "u8pc", "s8"])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(str(v) for v in c))
def test_unpadded_depthwise_matches_oracle(case, form):
    n, c, dm, h, w, stride, lead = case
    k = 3
    print("dw gather", case, form, flush=True)
    cout, pad = c * dm, (k // 2,) * 4
    s = O.conv_shape(n, c, h, w, cout, k, k, stride=(stride, stride), pad=pad, groups=c, dm=dm)
    x, wt = synth.fill_u8((n, c, h, w), SEED + h), synth.fill_u8((cout, 1, k, k), SEED + c)
    bias = synth.fill_i32((cout,), SEED + 1, -2000, 2000)
    ho, wo = (h + 2 * pad[0] - k) // stride + 1, (w + 2 * pad[0] - k) // stride + 1
    signed, layout = form == "s8", eden.NHWC
    if signed:
        q = O.make_quant_s8(0.02, 9, 0.004, 0, 0.05 * k, -4)
        x, wt = x.view(np.int8), wt.view(np.int8)
        want = O.dwconv2d_s8(x, wt, bias, s, q)
        layout |= eden.IO_SIGNED
    else:
        q = O.make_quant(0.02, 117, 0.004, 121, 0.05 * k, 128)
        want = O.dwconv2d(x, wt, bias, s, q)
    e = to_eh_requant(q)
    weight_layout = eden.W_OIHW | (eden.W_SIGNED if signed else 0)
    desc = eden.conv_desc(n, c, h, w, cout, k, k, stride=(stride, stride), pad=pad, dm=dm, layout=layout, weight_layout=weight_layout)
    d_w, d_b = eden.DeviceBuffer(host=wt), eden.DeviceBuffer(host=bias)
    plan = eden.DwConvPlan(desc, d_w, d_b, e)
    if form == "u8pc":   # the tensors' own pair for every channel: the same results through the per-channel code
        plan.set_perchannel(np.full(cout, e.multiplier), np.full(cout, e.shift))
    padded = np.concatenate([np.full(lead, 7, np.uint8), x.view(np.uint8).transpose(0, 2, 3, 1).ravel()])
    d_x, d_o = eden.DeviceBuffer(host=padded), eden.DeviceBuffer(nbytes=n * cout * ho * wo + 8)
    plan.run(eden.BufferView(d_x, lead), eden.BufferView(d_o, lead), e)
    got = d_o.download((n * cout * ho * wo + 8,))[lead:lead + n * cout * ho * wo].reshape(n, ho, wo, cout).transpose(0, 3, 1, 2).view(want.dtype)
    assert np.array_equal(got, want), diff_report(got, want)
    assert n * cout * ho * wo < 64 or want.std() > 1
