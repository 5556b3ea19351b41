"""Runs whose output lies on their input, wholly or in part, of layers that otherwise read the caller's tensor while they store
(channels off 16 and planar tensors): the same bytes as the oracle's.  Enough tiles that several workgroups are at it."""
import numpy as np
import pytest

import oracle_lib as O
from harness import diff_report, eden, synth, to_eh_requant

pytestmark = pytest.mark.gpu
SEED = 0x1A9C


def in_place(plan, x, out_bytes, q, shift):
    """the plan's result with its output `shift` bytes behind its input in the same memory"""
    x = np.ascontiguousarray(x).view(np.uint8).ravel()
    d = eden.DeviceBuffer(host=np.concatenate([x, np.zeros(max(0, shift + out_bytes - x.size), np.uint8)]))
    plan.run(d, eden.BufferView(d, shift), q)
    return d.download((d.nbytes,))[shift:shift + out_bytes]


@pytest.mark.parametrize("kind,n,c,h,cout,k,layout,shift", [
    ("conv", 2, 21, 33, 21, 3, eden.NHWC, 0),
    ("conv", 2, 21, 33, 21, 3, eden.NHWC, 160),
    ("conv", 1, 40, 31, 24, 1, eden.NHWC, 0),
    ("conv", 3, 21, 47, 21, 3, eden.NCHW, 0),
    ("conv", 2, 64, 20, 30, 3, eden.NCHW, 0),
    ("deconv", 2, 23, 15, 17, 3, eden.NHWC, 0),
    ("deconv", 2, 23, 15, 17, 3, eden.NCHW, 0),
    ("fc", 1, 113, 97, 113, 1, eden.NHWC, 0),      # 97 rows
    ("dw", 2, 33, 41, 33, 3, eden.NHWC, 0),
    ("dw", 2, 33, 41, 33, 3, eden.NHWC, 33 * 41),
    ("dw", 2, 22, 41, 44, 3, eden.NHWC, 0),        # a multiplier
    ("dw", 2, 24, 41, 24, 3, eden.NCHW, 0),
    ("dw", 2, 24, 41, 24, 5, eden.NCHW, 41 * 41),
    ("dw", 1, 64, 56, 64, 7, eden.NCHW, 0),        # four rows to a thread
])
def test_in_place(kind, n, c, h, cout, k, layout, shift):
    print("in place", kind, n, c, h, cout, k, layout, shift, flush=True)
    q = O.make_quant(0.02, 131, 0.005, 117, float(0.02 * 0.005 * 74 * 74 * np.sqrt((1 if kind == "dw" else c) * k * k) / 40), 120)
    b, pad = synth.fill_i32((cout,), SEED + 1, -1000, 1000), (k // 2,) * 4
    d_b = eden.DeviceBuffer(host=b)
    if kind == "fc":
        x, w = synth.fill_u8((h, c), SEED), synth.fill_u8((cout, c), SEED + 2)
        want, d_w = O.fc(x, w, b, q), eden.DeviceBuffer(host=w)
        plan = eden.FcPlan(h, c, cout, d_w, d_b, to_eh_requant(q))
    elif kind == "dw":
        x, w = synth.fill_u8((n, c, h, h), SEED), synth.fill_u8((cout, 1, k, k), SEED + 2)
        want = O.dwconv2d(x, w, b, O.conv_shape(n, c, h, h, cout, k, k, pad=pad, groups=c, dm=cout // c), q)
        d_w = eden.DeviceBuffer(host=w)
        plan = eden.DwConvPlan(eden.conv_desc(n, c, h, h, cout, k, k, (1, 1), pad, dm=cout // c, layout=layout), d_w, d_b, to_eh_requant(q))
    else:
        deconv = kind == "deconv"
        x, w = synth.fill_u8((n, c, h, h), SEED), synth.fill_u8((c, cout, k, k) if deconv else (cout, c, k, k), SEED + 2)
        want = (O.deconv2d if deconv else O.conv2d)(x, w, b, O.conv_shape(n, c, h, h, cout, k, k, pad=pad), q)
        desc = eden.conv_desc(n, c, h, h, cout, k, k, (1, 1), pad, layout=layout, weight_layout=eden.W_IOHW if deconv else eden.W_OIHW)
        d_w = eden.DeviceBuffer(host=w)
        plan = (eden.DeconvPlan if deconv else eden.ConvPlan)(desc, d_w, d_b, to_eh_requant(q))
    if kind != "fc" and layout == eden.NHWC:
        x, want = x.transpose(0, 2, 3, 1), want.transpose(0, 2, 3, 1)
    got = in_place(plan, x, want.size, to_eh_requant(q), shift).reshape(want.shape)
    assert np.array_equal(got, want), diff_report(got, want)
