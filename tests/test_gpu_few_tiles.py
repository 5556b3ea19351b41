"""The kernel for few output tiles (the reduction shared by a workgroup's waves) at the edges of its tiles, of its 128-byte
groups of the reduction and of its launch rule, against the CPU oracle."""
import numpy as np
import pytest

import oracle_lib as O
from harness import diff_report, eden, gpu_conv, gpu_deconv, gpu_fc, synth, to_eh_add, to_eh_requant

pytestmark = pytest.mark.gpu
SEED = 0xEDE2 + 16 * 23

CASES = [
    dict(n=1, c=16, h=5, w=7, cout=3, kh=3, kw=3, pad=(1, 1, 1, 1)),                       # 35 pixels, 3 channels, a group over eight taps
    dict(n=1, c=48, h=8, w=8, cout=33, kh=3, kw=3, stride=(2, 1), pad=(1, 0, 1, 2)),       # groups that cross taps
    dict(n=1, c=256, h=14, w=14, cout=256, kh=3, kw=3, pad=(1, 1, 1, 1)),                  # three groups per wave
    dict(n=2, c=512, h=7, w=7, cout=100, kh=3, kw=3, pad=(1, 1, 1, 1)),                    # more groups than travel together
    dict(n=1, c=144, h=9, w=5, cout=40, kh=5, kw=5, pad=(2, 2, 2, 2), dil=(2, 1)),         # dilation, 13.5 KiB of weights per channel block
    dict(n=3, c=320, h=1, w=11, cout=7, kh=1, kw=1),                                       # 33 pixels, one tap
    dict(n=1, c=272, h=6, w=6, cout=64, kh=1, kw=1, stride=(2, 2), pad=(1, 1, 1, 1)),      # a tap that leaves the image
    dict(n=2, c=64, h=10, w=10, cout=64, kh=3, kw=3, pad=(1, 1, 1, 1), groups=4),          # channel groups
    dict(n=1, c=21, h=9, w=8, cout=21, kh=3, kw=3, pad=(1, 1, 1, 1)),                      # on the channel-padded copy
    dict(n=1, c=64, h=16, w=31, cout=512, kh=1, kw=1),                                     # 256 tiles, the largest launch of a one-tap plan
]


@pytest.mark.parametrize("layout", [eden.NHWC, eden.NCHW], ids=["nhwc", "nchw"])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(str(v) for v in list(c.values())[:7]))
def test_few_tiles_conv(case, layout):
    s = O.conv_shape(**case)
    red = s.c // s.groups * s.kh * s.kw
    x, w = synth.fill_u8((s.n, s.c, s.h, s.w), SEED + s.c), synth.fill_u8((s.cout, s.c // s.groups, s.kh, s.kw), SEED + s.cout)
    b = synth.fill_i32((s.cout,), SEED + 2, -1000, 1000)
    for zp_x, zp_w in ((131, 128), (127, 97)):   # without and with the activation sums
        q = O.make_quant(0.02, zp_x, 0.005, zp_w, 0.02 * 0.005 * 74 * 74 * red ** 0.5 / 40, 120)
        want = O.conv2d(x, w, b, s, q)
        got = gpu_conv(x, w, b, s, to_eh_requant(q), layout=layout)
        assert np.array_equal(got, want), diff_report(got, want)
        assert want.std() > 2


@pytest.mark.parametrize("m,k,n", [(17, 272, 10), (31, 4096, 65), (33, 512, 31), (64, 3456, 184), (257, 640, 30), (100, 8192, 34)])
@pytest.mark.parametrize("flags", [0, eden.W_SIGNED | eden.IO_SIGNED], ids=["u8", "s8"])
def test_few_tiles_fully_connected(m, k, n, flags):
    a, w = synth.fill_u8((m, k), SEED + 5), synth.fill_u8_normal((n, k), SEED + 6, 128, 25)
    b = synth.fill_i32((n,), SEED + 7, -1000, 1000)
    s_out = 0.01 * 0.002 * 74 * 25 * k ** 0.5 / 40
    if flags:
        a, w = (a.astype(np.int16) - 128).astype(np.int8), (w.astype(np.int16) - 128).astype(np.int8)
        q = O.make_quant_s8(0.01, 3, 0.002, -2, s_out, 5, O.ACT_NONE, False)
        want, got = O.fc_s8(a, w, b, q), gpu_fc(a, w, b, to_eh_requant(q), flags=flags).view(np.int8)
    else:
        q = O.make_quant(0.01, 125, 0.002, 120, s_out, 128)
        want, got = O.fc(a, w, b, q), gpu_fc(a, w, b, to_eh_requant(q))
    assert np.array_equal(got, want), diff_report(got, want)
    assert want.std() > 4


@pytest.mark.parametrize("m,k,n", [(1, 1 << 20, 33), (1, (1 << 20) + 16, 33), (11, (1 << 20) + 16, 33), (17, (1 << 20) + 32, 5)])
def test_fully_connected_reductions_beyond_2_to_the_20(m, k, n):
    # (inputs near their zero points: the sums of the oracle and of the kernels stay far inside 32 bits)
    a, w = synth.fill_u8_normal((m, k), SEED + 31, 120, 6), synth.fill_u8_normal((n, k), SEED + 32, 128, 6)
    b = synth.fill_i32((n,), SEED + 33, -1000, 1000)
    q = O.make_quant(0.01, 120, 0.002, 128, 0.01 * 0.002 * 36 * k ** 0.5 / 40, 128)
    want, got = O.fc(a, w, b, q), gpu_fc(a, w, b, to_eh_requant(q))
    assert np.array_equal(got, want), diff_report(got, want)
    assert want.std() > 4


@pytest.mark.parametrize("case", [dict(n=1, c=32, h=5, w=6, cout=8, kh=4, kw=4, stride=(2, 2), pad=(1, 1, 1, 1)),     # phases side by side
                                  dict(n=2, c=48, h=7, w=7, cout=10, kh=3, kw=3, stride=(2, 2), pad=(1, 1, 1, 1)),    # phases of unequal taps and pixel counts
                                  dict(n=1, c=64, h=4, w=5, cout=21, kh=8, kw=8, stride=(4, 4), pad=(2, 2, 2, 2))],
                         ids=["4x4s2", "3x3s2", "8x8s4"])
def test_few_tiles_deconv(case):
    s = O.conv_shape(**case)
    x, w = synth.fill_u8((s.n, s.c, s.h, s.w), SEED + 11), synth.fill_u8((s.c, s.cout, s.kh, s.kw), SEED + 12)
    b = synth.fill_i32((s.cout,), SEED + 13, -1000, 1000)
    q = O.make_quant(0.02, 121, 0.005, 133, 0.02 * 0.005 * 74 * 74 * (s.c * 4) ** 0.5 / 40, 128)
    want, got = O.deconv2d(x, w, b, s, q), gpu_deconv(x, w, b, s, to_eh_requant(q), layout=eden.NHWC)
    assert np.array_equal(got, want), diff_report(got, want)
    assert want.std() > 4


@pytest.mark.parametrize("cout", [160, 34, 5])
def test_few_tiles_residual_add_and_per_channel(cout):
    s = O.conv_shape(2, 320, 7, 7, cout, 1, 1)
    x, res = synth.fill_u8((2, 320, 7, 7), SEED + 21), synth.fill_u8((2, 7, 7, cout), SEED + 22)
    w = (synth.fill_u8((cout, 320, 1, 1), SEED + 23).astype(np.int16) - 128).clip(-127, 127).astype(np.int8)
    b = synth.fill_i32((cout,), SEED + 24, -1000, 1000)
    scales = (0.002 * (1.0 + 9.0 * synth.fill_u8((cout,), SEED + 25) / 255.0)).astype(np.float32)
    q, mults, shifts = eden.make_requant_perchannel(0.02, 120, scales, 2.0, 128)
    oq = O.raw_quant(zp_in=120, zp_w=0, zp_out=128)
    conv = np.ascontiguousarray(O.conv2d_perchannel(x, w, b, s, oq, mults, shifts).transpose(0, 2, 3, 1))
    aq = O.make_add_quant(0.03, 110, 0.05, 128, 0.06, 120)
    desc = eden.conv_desc(2, 320, 7, 7, cout, 1, 1, layout=eden.NHWC, weight_layout=eden.W_OIHW | eden.W_SIGNED)
    d_x, d_w, d_b, d_r = (eden.DeviceBuffer(host=t) for t in (np.ascontiguousarray(x.transpose(0, 2, 3, 1)), w, b, res))
    d_o = eden.DeviceBuffer(nbytes=conv.size)
    plan = eden.ConvPlan(desc, d_w, d_b, q)
    plan.set_perchannel(mults, shifts)
    assert plan.fuses_add()
    plan.run(d_x, d_o, q)
    assert np.array_equal(d_o.download(conv.shape), conv)
    plan.run_add(d_x, d_r, d_o, q, to_eh_add(aq))
    assert np.array_equal(d_o.download(conv.shape), O.add(res, conv, aq))


def test_the_cases_above_run_on_the_kernel_for_few_tiles():
    for case in CASES:
        s = O.conv_shape(**case)
        for layout in (eden.NHWC, eden.NCHW):
            desc = eden.conv_desc(s.n, s.c, s.h, s.w, s.cout, s.kh, s.kw, (s.stride_h, s.stride_w), (s.pad_t, s.pad_b, s.pad_l, s.pad_r), (s.dil_h, s.dil_w), s.groups,
                                  layout=layout)
            assert set(eden.conv_kernels(desc, launched=True)) == {"few_tiles"}, (case, eden.conv_kernels(desc, launched=True))
    rows = [(17, 272, 10), (31, 4096, 65), (33, 512, 31), (64, 3456, 184), (257, 640, 30), (100, 8192, 34), (11, (1 << 20) + 16, 33), (17, (1 << 20) + 32, 5)]
    for m, k, n in rows:
        assert eden.conv_kernels(eden.conv_desc(m, k, 1, 1, n, 1, 1, layout=eden.NHWC), launched=True) == ["few_tiles"], (m, k, n)
    for m, k, n in ((1, 1 << 20, 33), (1, (1 << 20) + 16, 33)):
        assert eden.conv_kernels(eden.conv_desc(m, k, 1, 1, n, 1, 1, layout=eden.NHWC), launched=True) == ["skinny"], (m, k, n)
    for c, h, w, cout, k, st, pad, n in ((32, 5, 6, 8, 4, 2, 1, 1), (48, 7, 7, 10, 3, 2, 1, 2), (64, 4, 5, 21, 8, 4, 2, 1)):
        desc = eden.conv_desc(n, c, h, w, cout, k, k, (st, st), (pad,) * 4, layout=eden.NHWC, weight_layout=eden.W_IOHW)
        assert set(eden.conv_kernels(desc, deconv=True, launched=True)) == {"few_tiles"}, (c, cout, k)
    for cout in (160, 34, 5):
        assert eden.conv_kernels(eden.conv_desc(2, 320, 7, 7, cout, 1, 1, layout=eden.NHWC), launched=True) == ["few_tiles"]
