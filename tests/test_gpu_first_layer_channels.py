"""First layers of one to four channels (a kernel row per reduction step) with a pair per channel, on launches that fill the GPU: bit for
bit the oracle in each of several runs, for every number of rows, clamps at the zero point and away from it, channels-last and planar
tensors.  A wave's last channels had gone wrong in some runs (see test_wide_shifts.py)."""
import numpy as np
import pytest

import oracle_lib as O
from harness import diff_report, eden, synth

pytestmark = pytest.mark.gpu
SEED = 0xF1C7


@pytest.mark.parametrize("linear", [True, False], ids=["linear", "relu6"])
@pytest.mark.parametrize("layout", [eden.NHWC, eden.NCHW], ids=["nhwc", "nchw"])
@pytest.mark.parametrize("form", ["u8", "s8"])
@pytest.mark.parametrize("n,c,h,cout,k", [(12, 3, 144, 56, 7), (6, 3, 120, 90, 7), (10, 3, 100, 40, 5), (10, 4, 90, 72, 3), (4, 3, 96, 33, 9), (4, 2, 96, 48, 11)])
def test_first_layer_with_pairs_matches_oracle(n, c, h, cout, k, form, layout, linear):
    print("first layer, pairs", n, c, h, cout, k, form, layout, linear, flush=True)
    pad, signed = (k // 2,) * 4, form == "s8"
    s = O.conv_shape(n, c, h, h, cout, k, k, stride=(2, 2), pad=pad)
    x, b = synth.fill_u8((n, c, h, h), SEED + h), synth.fill_i32((cout,), SEED + 1, -1000, 1000)
    w = (synth.fill_u8((cout, c, k, k), SEED + k).astype(np.int16) - 128).astype(np.int8)
    w_scales = (0.002 * (1.0 + 3.0 * synth.fill_u8((cout,), SEED + 2) / 255.0)).astype(np.float32)
    s_out, zp_out = float(0.02 * w_scales.max() * 74.0 * 74.0 * np.sqrt(c * k * k) / 50.0), 128 if linear else 0
    off = 128 if signed else 0
    q, *pairs = eden.make_requant_perchannel(0.02, 117 - off, w_scales, s_out, zp_out - off, eden.ACT_NONE if linear else eden.ACT_RELU, not linear)
    if signed:
        q.act_min, q.act_max = -128, 127
        x = (x.astype(np.int16) - 128).astype(np.int8)
        want = O.conv2d_s8(x, w, b, s, O.raw_quant(zp_in=117 - off, zp_w=0, zp_out=zp_out - off, act_min=-128, act_max=127), *pairs)
    else:
        want = O.conv2d_perchannel(x, w, b, s, O.raw_quant(zp_in=117, zp_w=0, zp_out=zp_out, act_min=q.act_min, act_max=q.act_max), *pairs)
    desc = eden.conv_desc(n, c, h, h, cout, k, k, (2, 2), pad, layout=layout | (eden.IO_SIGNED if signed else 0), weight_layout=eden.W_OIHW | eden.W_SIGNED)
    assert k == 3 or eden.conv_kernels(desc) == ["few_channel_rows"]
    nhwc = layout == eden.NHWC
    d_x = eden.DeviceBuffer(host=np.ascontiguousarray(x.transpose(0, 2, 3, 1) if nhwc else x).view(np.uint8))
    d_w, d_b, d_o = eden.DeviceBuffer(host=w), eden.DeviceBuffer(host=b), eden.DeviceBuffer(nbytes=want.size)
    plan = eden.ConvPlan(desc, d_w, d_b, q)
    plan.set_perchannel(*pairs)
    ho, wo = want.shape[2:]
    for _ in range(4):
        plan.run(d_x, d_o, q)
        got = d_o.download((n, ho, wo, cout)).transpose(0, 3, 1, 2) if nhwc else d_o.download((n, cout, ho, wo))
        same = np.array_equal(got.view(want.dtype), want)
        assert same, diff_report(got.view(want.dtype), want)
    assert want.std() > 10
