"""Planar depthwise layers straight from the caller's tensors: bit for bit the oracle, at widths that leave a thread's four
outputs, and its loads at the tensor's first and last bytes, in every position against the words of memory; windows wider than
the image; one row and four rows to a thread; depth multipliers, channel counts of any kind, uneven paddings and none; int8 tensors, pairs
that differ from channel to channel; and not a byte beside the result.  (test_launch_grid.py holds that these cases take the planar kernels.)"""
import numpy as np
import pytest

import oracle_lib as O
from harness import diff_report, eden, synth, to_eh_requant

pytestmark = pytest.mark.gpu
SEED = 0xD3A1

CASES = [
    # n, c, dm, h, w, k, stride, bytes that the input starts past a word, padding (top, bottom, left, right) if not half the window
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
    (2, 6, 1, 11, 13, 3, 1, 1, (0, 0, 0, 0)),
    (1, 5, 2, 12, 9, 5, 2, 2, (0, 2, 0, 1)),
    (2, 9, 1, 10, 10, 7, 1, 3, (5, 1, 3, 0)),      # more rows above than the window has over its centre
    (1, 8, 1, 9, 14, 3, 2, 0, (2, 0, 3, 2)),       # windows wholly in the padding
    (4, 64, 1, 50, 47, 5, 1, 2, (0, 4, 1, 3)),
    (1, 7, 1, 8, 21, 7, 2, 1, (1, 0, 2, 5)),
]


def problem(s, form, x_seed, w_seed, out_scale):
    """(input, weights, requantization, pairs of the channels or None, the oracle's result) of a depthwise layer"""
    x, wt = synth.fill_u8((s.n, s.c, s.h, s.w), x_seed), synth.fill_u8((s.cout, 1, s.kh, s.kw), w_seed)
    bias, pairs = synth.fill_i32((s.cout,), SEED + 1, -2000, 2000), None
    if form == "s8":
        q = O.make_quant_s8(0.02, 9, 0.004, 0, out_scale, -4)
        x, wt = x.view(np.int8), wt.view(np.int8)
        return x, wt, to_eh_requant(q), None, O.dwconv2d_s8(x, wt, bias, s, q)
    if form == "u8":
        q = O.make_quant(0.02, 117, 0.004, 121, out_scale, 128)
        return x, wt, to_eh_requant(q), None, O.dwconv2d(x, wt, bias, s, q)
    wt = wt.view(np.int8)
    scales = (0.001 * (1.0 + 15.0 * synth.fill_u8((s.cout,), SEED + 2) / 255.0)).astype(np.float32)   # shifts that differ as well
    if form == "u8pc":
        e, *pairs = eden.make_requant_perchannel(0.02, 117, scales, out_scale, 128)
        return x, wt, e, pairs, O.dwconv2d_perchannel(x, wt, bias, s, O.raw_quant(zp_in=117, zp_w=0, zp_out=128), *pairs)
    e, *pairs = eden.make_requant_perchannel(0.02, 9, scales, out_scale, -4)
    e.act_min, e.act_max = -128, 127
    x = x.view(np.int8)
    return x, wt, e, pairs, O.dwconv2d_s8(x, wt, bias, s, O.raw_quant(zp_in=9, zp_w=0, zp_out=-4, act_min=-128, act_max=127), *pairs)


@pytest.mark.parametrize("form", ["u8", "u8pc", "s8", "s8pc"])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(str(v) for v in c))
def test_planar_depthwise_matches_oracle(case, form):
    n, c, dm, h, w, k, stride, lead = case[:8]
    print("dw planar", case, form, flush=True)
    cout, pad = c * dm, case[8] if len(case) > 8 else (k // 2,) * 4
    s = O.conv_shape(n, c, h, w, cout, k, k, stride=(stride, stride), pad=pad, groups=c, dm=dm)
    ho, wo = O.conv_out_hw(s)
    x, wt, e, pairs, want = problem(s, form, SEED + h, SEED + c, 0.05 * k)
    desc = eden.conv_desc(n, c, h, w, cout, k, k, stride=(stride, stride), pad=pad, dm=dm, layout=eden.NCHW | (eden.IO_SIGNED if x.dtype == np.int8 else 0),
                          weight_layout=eden.W_OIHW | (eden.W_SIGNED if wt.dtype == np.int8 else 0))
    bias = synth.fill_i32((cout,), SEED + 1, -2000, 2000)
    d_w, d_b = eden.DeviceBuffer(host=wt), eden.DeviceBuffer(host=bias)
    plan = eden.DwConvPlan(desc, d_w, d_b, e)
    if pairs:
        plan.set_perchannel(*pairs)
    count = n * cout * ho * wo
    d_x, d_o = eden.DeviceBuffer(host=np.concatenate([np.full(lead, 7, np.uint8), x.view(np.uint8).ravel()])), eden.DeviceBuffer(host=np.full(count + 8, 0xA5, np.uint8))
    plan.run(eden.BufferView(d_x, lead), eden.BufferView(d_o, lead), e)
    whole = d_o.download((count + 8,))
    got = whole[lead:lead + count].reshape(n, cout, ho, wo).view(want.dtype)
    assert np.array_equal(got, want), diff_report(got, want)
    assert (whole[:lead] == 0xA5).all() and (whole[lead + count:] == 0xA5).all()
    assert count < 64 or want.std() > 1
