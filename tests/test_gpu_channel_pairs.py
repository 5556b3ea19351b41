"""One multiplier and shift per channel at the edges of the four-channel requantization: every shift from -2 to -20 among the channels
of one layer and multipliers at both ends of their range, in the kernels that use it (one tap, 3x3 patch, first layer); and the fused
expansion + depthwise launch with a depthwise shift of -1, which takes the two-step order there.  Bit for bit the oracle."""
import numpy as np
import pytest

import oracle_lib as O
from harness import diff_report, eden, synth
from test_gpu_perchannel import gpu_conv_perchannel

pytestmark = pytest.mark.gpu
SEED = 0xC4A1


def edge_pairs(count, first_shift):
    shifts = np.array([first_shift - i % (21 + first_shift) for i in range(count)], np.int32)
    ends = [1 << 30, (1 << 31) - 1, 1518500250, (1 << 30) + 1]
    return np.array([ends[(i // 3) % 4] for i in range(count)], np.int32), shifts


def int8(shape, seed):
    return (synth.fill_u8(shape, seed).astype(np.int16) - 128).astype(np.int8)


@pytest.mark.parametrize("act_min", [0, 90], ids=["signed", "rectified"])
@pytest.mark.parametrize("case", [(3, 32, 63, 61, 72, 1, 1), (1, 144, 40, 30, 40, 1, 1), (9, 64, 31, 30, 48, 3, 1), (2, 3, 33, 31, 40, 3, 2)],
                         ids=lambda c: "x".join(str(v) for v in c))
def test_shift_range_matches_oracle(case, act_min):
    n, c, h, w, cout, k, stride = case
    print("pairs", case, act_min, flush=True)
    x, wt = synth.fill_u8((n, c, h, w), SEED + c), int8((cout, c, k, k), SEED + cout)
    bias = synth.fill_i32((cout,), SEED + 1, -500, 500)
    s = O.conv_shape(n, c, h, w, cout, k, k, stride=(stride, stride), pad=(k // 2,) * 4)
    mults, shifts = edge_pairs(cout, -2)
    zp_out = 90
    q = eden.Requant(117, 0, zp_out, int(mults[0]), int(shifts[0]), act_min, 231)
    oq = O.raw_quant(zp_in=117, zp_w=0, zp_out=zp_out, act_min=act_min, act_max=231)
    want = O.conv2d_perchannel(x, wt, bias, s, oq, mults, shifts)
    got, _ = gpu_conv_perchannel(x, wt, bias, s, q, mults, shifts, eden.NHWC)
    assert np.array_equal(got, want), diff_report(got, want)
    assert want.std() > 4


@pytest.mark.parametrize("rows, cols, c, matrix", [(3, 4, 48, True), (8, 9, 64, False)], ids=["matrix", "vector"])
@pytest.mark.parametrize("depthwise_shift", [-1, -2])
def test_fused_launch_at_the_largest_depthwise_scales(depthwise_shift, rows, cols, c, matrix):
    n, h, w, cin = 2, 9, 11, 24
    x, w1, w2 = synth.fill_u8((n, h, w, cin), SEED + 7), int8((c, cin, 1, 1), SEED + 8), int8((c, 1, 3, 3), SEED + 9)
    b1, b2 = synth.fill_i32((c,), SEED + 10, -500, 500), synth.fill_i32((c,), SEED + 11, -500, 500)
    m1, sh1 = edge_pairs(c, -8)
    m2, sh2 = edge_pairs(c, depthwise_shift)
    q1, q2 = eden.Requant(117, 0, 128, int(m1[0]), int(sh1[0]), 0, 255), eden.Requant(128, 0, 128, int(m2[0]), int(sh2[0]), 0, 255)
    o1, o2 = O.raw_quant(zp_in=117, zp_w=0, zp_out=128), O.raw_quant(zp_in=128, zp_w=0, zp_out=128)
    mid = O.conv2d_perchannel(np.ascontiguousarray(x.transpose(0, 3, 1, 2)), w1, b1, O.conv_shape(n, cin, h, w, c, 1, 1), o1, m1, sh1)
    s2 = O.conv_shape(n, c, h, w, c, 3, 3, pad=(1, 1, 1, 1), groups=c)
    want = np.ascontiguousarray(O.dwconv2d_perchannel(mid, w2, b2, s2, o2, m2, sh2).transpose(0, 2, 3, 1))
    keep = [eden.DeviceBuffer(host=a) for a in (w1, b1, w2, b2)]
    pw = eden.ConvPlan(eden.conv_desc(n, cin, h, w, c, 1, 1, layout=eden.NHWC, weight_layout=eden.W_OIHW | eden.W_SIGNED), keep[0], keep[1], q1)
    dw = eden.DwConvPlan(eden.conv_desc(n, c, h, w, c, 3, 3, pad=(1, 1, 1, 1), dm=1, layout=eden.NHWC, weight_layout=eden.W_OIHW | eden.W_SIGNED), keep[2],
                         keep[3], q2)
    pw.set_perchannel(m1, sh1)
    dw.set_perchannel(m2, sh2)
    assert eden.conv_dw_block_applies(pw, dw) and eden.conv_dw_block_tile(pw, dw, rows, cols)[3] == matrix
    d_x, d_o = eden.DeviceBuffer(host=x), eden.DeviceBuffer(nbytes=n * h * w * c)
    eden.conv_dw_block_run(pw, dw, d_x, d_o, q1, q2, rows, cols)
    got = d_o.download((n, h, w, c))
    assert np.array_equal(got, want), diff_report(got, want)
    assert want.std() > 4
