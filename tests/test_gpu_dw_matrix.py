"""The matrix form of 5x5 and 7x7 depthwise windows at the edges of its tiles, its channel pieces and its launch rule,
against the CPU oracle."""
import numpy as np
import pytest

import oracle_lib as O
from harness import diff_report, eden, gpu_dwconv, synth, to_eh_requant

pytestmark = pytest.mark.gpu
SEED = 0xEDE2 + 16 * 29

CASES = [
    # n, c, h, w, k, stride, (top, bottom, left, right)
    (1, 4, 5, 5, 5, 1, (0, 0, 0, 0)),          # one output, a quarter of a piece
    (2, 20, 9, 9, 7, 1, (3, 3, 3, 3)),         # a tile and one row more, tensor ends inside a piece
    (1, 48, 8, 16, 5, 2, (1, 2, 2, 1)),        # whole tiles at stride 2, unequal padding
    (1, 36, 7, 3, 7, 2, (6, 6, 6, 6)),         # windows wholly in the padding
    (16, 64, 15, 17, 5, 1, (2, 2, 2, 2)),      # the two-strip tiles of 7 rows, three column groups
    (24, 16, 40, 61, 5, 1, (2, 2, 2, 2)),      # one piece per workgroup, seven column groups and one more
    (40, 112, 29, 18, 7, 1, (3, 3, 3, 3)),     # seven pieces: blocks of four and three
    (12, 100, 57, 30, 7, 2, (3, 3, 3, 3)),
]


@pytest.mark.parametrize("zp_w,spread", [(128, 30), (131, 60), (0, 60), (255, 60)])   # differences within int8, slightly beyond, up to 255 of either sign
@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(str(v) for v in c[:6]))
def test_matrix_depthwise(case, zp_w, spread):
    n, c, h, w, k, stride, pad = case
    s = O.conv_shape(n, c, h, w, c, k, k, stride=(stride, stride), pad=pad)
    x = synth.fill_u8((n, c, h, w), SEED + c)
    wt = synth.fill_u8_normal((c, 1, k, k), SEED + k, 128, spread)
    b = synth.fill_i32((c,), SEED + 1, -1000, 1000)
    zp_in = 128 if zp_w in (0, 255) else 93
    q = O.make_quant(0.02, zp_in, 0.005, zp_w, 0.02 * 0.005 * 74 * (160 if zp_w in (0, 255) else spread) * k / 40, 120)
    want = O.dwconv2d(x, wt, b, s, q)
    got = gpu_dwconv(x, wt, b, s, to_eh_requant(q), layout=eden.NHWC)
    assert np.array_equal(got, want), diff_report(got, want)
    assert want.std() > 4


@pytest.mark.parametrize("k", [5, 7])
@pytest.mark.parametrize("scale", [3.0, 1e-7], ids=["left_shift", "long_shift"])   # multipliers outside the single-shift form
def test_matrix_depthwise_two_step_requantization(k, scale):
    n, c, hw = 4, 40, 20
    s = O.conv_shape(n, c, hw, hw, c, k, k, pad=(k // 2,) * 4)
    x, wt = synth.fill_u8((n, c, hw, hw), SEED + 7), synth.fill_u8((c, 1, k, k), SEED + 8)
    b = synth.fill_i32((c,), SEED + 9, -2 ** 30, 2 ** 30) if scale < 1 else synth.fill_i32((c,), SEED + 9, -1000, 1000)
    q = O.make_quant(1.0, 128, 1.0, 128, 1.0 / scale, 128)
    want = O.dwconv2d(x, wt, b, s, q)
    got = gpu_dwconv(x, wt, b, s, to_eh_requant(q), layout=eden.NHWC)
    assert np.array_equal(got, want), diff_report(got, want)
    assert want.std() > 4


@pytest.mark.parametrize("quant", ["u8pc", "s8", "s8pc"])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(str(v) for v in c[:6]))
def test_matrix_depthwise_per_channel_and_int8(case, quant):
    n, c, h, w, k, stride, pad = case
    s = O.conv_shape(n, c, h, w, c, k, k, stride=(stride, stride), pad=pad)
    signed, pc = quant.startswith("s8"), quant.endswith("pc")
    x = synth.fill_u8((n, c, h, w), SEED + 41)
    if signed:
        x = (x.astype(np.int16) - 128).astype(np.int8)
    wt = (synth.fill_u8((c, 1, k, k), SEED + 42).astype(np.int16) - 128).astype(np.int8)   # the whole range, -128 among it
    b = synth.fill_i32((c,), SEED + 43, -1000, 1000)
    desc = eden.conv_desc(n, c, h, w, c, k, k, (stride,) * 2, pad, (1, 1), 1, 1, eden.NHWC | (eden.IO_SIGNED if signed else 0), eden.W_OIHW | eden.W_SIGNED)
    d_x, d_w, d_b = eden.DeviceBuffer(host=np.ascontiguousarray(x.transpose(0, 2, 3, 1))), eden.DeviceBuffer(host=wt), eden.DeviceBuffer(host=b)
    d_o = eden.DeviceBuffer(nbytes=int(np.prod(O.conv_out_hw(s))) * n * c)

    def compare(plan, q, want):
        plan.run(d_x, d_o, q)
        got = d_o.download((n, want.shape[2], want.shape[3], c)).transpose(0, 3, 1, 2).view(want.dtype)
        assert np.array_equal(got, want), diff_report(got, want)
        assert want.std() > 4

    if not pc:
        # weights about zero points at the ends of int8 too: differences of up to 255
        for zp_w, spread in ((3, 74), (-128, 147), (127, 147)):
            oq = O.make_quant_s8(0.02, -14, 0.005, zp_w, 0.02 * 0.005 * 74 * spread * k / 40, -3)
            q = to_eh_requant(oq)
            compare(eden.DwConvPlan(desc, d_w, d_b, q), q, O.dwconv2d_s8(x, wt, b, s, oq))
        return
    zp_in, zp_out = (-14, 5) if signed else (93, 131)
    scales = (0.002 * (1.0 + 9.0 * synth.fill_u8((c,), SEED + 44) / 255.0)).astype(np.float32)
    q, mults, shifts = eden.make_requant_perchannel(0.02, zp_in, scales, float(0.02 * 0.02 * 74 * 74 * k / 60), zp_out)
    oq = O.raw_quant(zp_in=zp_in, zp_w=0, zp_out=zp_out)
    if signed:
        q.act_min, q.act_max = oq.act_min, oq.act_max = -128, 127
    oracle = lambda sh: O.dwconv2d_s8(x, wt, b, s, oq, mults, sh) if signed else O.dwconv2d_perchannel(x, wt, b, s, oq, mults, sh)
    plan = eden.DwConvPlan(desc, d_w, d_b, q)
    plan.set_perchannel(mults, shifts)
    compare(plan, q, oracle(shifts))
    # one channel's shift outside the single-shift form's range: the whole launch takes the two-step order
    odd = shifts.copy()
    odd[c // 3] = 0
    plan.set_perchannel(mults, odd)
    compare(plan, q, oracle(odd))
    # the clamp's floor at the output zero point: the single-shift form without its sign test
    q.act_min = oq.act_min = zp_out
    plan.set_perchannel(mults, shifts)
    plan.run(d_x, d_o, q)
    want = oracle(shifts)
    assert np.array_equal(d_o.download((n, want.shape[2], want.shape[3], c)).transpose(0, 3, 1, 2).view(want.dtype), want)
