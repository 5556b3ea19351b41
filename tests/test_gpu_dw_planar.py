"""Planar depthwise layers straight from the caller's tensors: bit for bit the oracle, at widths that leave a thread's four
outputs, and its loads at the tensor's first and last bytes, in every position against the words of memory; windows wider than
the image; one row and four rows to a thread; depth multipliers, channel counts of any kind, int8 tensors, pairs per channel."""
import numpy as np
import pytest

import oracle_lib as O
from harness import diff_report, eden, synth, to_eh_requant

pytestmark = pytest.mark.gpu
SEED = 0xD3A1

CASES = [
    # n, c, dm, h, w, k, stride, bytes that the input starts past a word
    (1, 1, 1, 1, 1, 3, 1, 0),
    (1, 1, 1, 1, 2, 7, 1, 1),
    (1, 3, 1, 2, 3, 5, 2, 3),
    (2, 5, 1, 7, 5, 3, 1, 2),
    (1, 4, 2, 9, 6, 5, 1, 1),
    (3, 7, 3, 8, 7, 7, 2, 0),
    (2, 16, 1, 13, 13, 3, 2, 3),
    (2, 40, 1, 13, 7, 7, 1, 2),
    (1, 6, 1, 30, 29, 5, 1, 0),
    (3, 64, 1, 56, 57, 3, 1, 1),      # four rows to a thread
    (3, 64, 1, 57, 58, 5, 1, 3),
    (1, 256, 1, 47, 51, 7, 1, 2),
    (6, 96, 1, 61, 60, 3, 2, 0),
    (2, 144, 2, 62, 59, 5, 2, 1),
]


@pytest.mark.parametrize("form", ["u8", "u8pc", "s8"])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(str(v) for v in c))
def test_planar_depthwise_matches_oracle(case, form):
    n, c, dm, h, w, k, stride, lead = case
    print("dw planar", case, form, flush=True)
    cout, pad = c * dm, (k // 2,) * 4
    s = O.conv_shape(n, c, h, w, cout, k, k, stride=(stride, stride), pad=pad, groups=c, dm=dm)
    x, wt = synth.fill_u8((n, c, h, w), SEED + h), synth.fill_u8((cout, 1, k, k), SEED + c)
    bias = synth.fill_i32((cout,), SEED + 1, -2000, 2000)
    ho, wo = (h + 2 * pad[0] - k) // stride + 1, (w + 2 * pad[0] - k) // stride + 1
    signed, layout = form == "s8", eden.NCHW
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
    padded = np.concatenate([np.full(lead, 7, np.uint8), x.view(np.uint8).ravel()])
    d_x, d_o = eden.DeviceBuffer(host=padded), eden.DeviceBuffer(nbytes=n * cout * ho * wo + 8)
    plan.run(eden.BufferView(d_x, lead), eden.BufferView(d_o, lead), e)
    got = d_o.download((n * cout * ho * wo + 8,))[lead:lead + n * cout * ho * wo].reshape(n, cout, ho, wo).view(want.dtype)
    assert np.array_equal(got, want), diff_report(got, want)
    assert n * cout * ho * wo < 64 or want.std() > 1
