"""Planar tensors: the one-pass transposition with channel padding, and kernels that write planar outputs themselves, at the
edges of their tiles, against the CPU oracle."""
import numpy as np
import pytest

import oracle_lib as O
from harness import diff_report, eden, gpu_conv, gpu_deconv, synth, to_eh_requant

pytestmark = pytest.mark.gpu
SEED = 0xEDE2 + 16 * 31

CASES = [
    # n, c, h, w, cout, k, stride, groups
    (2, 13, 9, 7, 19, 3, 1, 1),         # channels padded 13 -> 16, odd plane
    (3, 33, 11, 13, 17, 1, 1, 1),       # padded 33 -> 48
    (1, 70, 5, 3, 40, 3, 2, 1),         # more than 32 padded channels, fifteen pixels
    (2, 32, 31, 33, 40, 1, 1, 1),       # one tap
    (5, 64, 30, 30, 24, 3, 1, 1),       # patch kernel
    (2, 3, 33, 31, 37, 3, 2, 1),        # three channels
    (2, 3, 40, 36, 20, 3, 2, 1),        # ... below 32 output channels
    (2, 4, 30, 31, 33, 7, 2, 1),        # kernel rows
    (4, 64, 40, 40, 100, 5, 2, 1),      # tiled kernels
    (2, 64, 13, 13, 48, 3, 1, 4),       # groups: planes behind one another
    (2, 6, 9, 9, 6, 3, 1, 2),           # grouped and padded
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(str(v) for v in c))
def test_planar_conv(case):
    n, c, h, w, cout, k, stride, groups = case
    s = O.conv_shape(n, c, h, w, cout, k, k, stride=(stride, stride), pad=(k // 2,) * 4, groups=groups)
    red = c // groups * k * k
    x, wt = synth.fill_u8((n, c, h, w), SEED + c), synth.fill_u8((cout, c // groups, k, k), SEED + cout)
    b = synth.fill_i32((cout,), SEED + 2, -1000, 1000)
    q = O.make_quant(0.02, 131, 0.005, 126, 0.02 * 0.005 * 74 * 74 * red ** 0.5 / 40, 120)
    want = O.conv2d(x, wt, b, s, q)
    got = gpu_conv(x, wt, b, s, to_eh_requant(q), layout=eden.NCHW)
    assert np.array_equal(got, want), diff_report(got, want)
    assert want.std() > 4


KERNELS = {  # what the cases are for (the others: whatever serves them)
    (2, 13, 9, 7, 19, 3, 1, 1): "few_tiles", (2, 32, 31, 33, 40, 1, 1, 1): "few_tiles", (5, 64, 30, 30, 24, 3, 1, 1): "few_tiles", (2, 3, 33, 31, 37, 3, 2, 1): "c3k3",
    (2, 3, 40, 36, 20, 3, 2, 1): "c3k3", (2, 4, 30, 31, 33, 7, 2, 1): "few_channel_rows", (4, 64, 40, 40, 100, 5, 2, 1): "few_tiles",
    (9, 64, 31, 30, 33, 3, 1, 1): "conv3x3_patch", (9, 32, 31, 33, 40, 1, 1, 1): "one_tap", (24, 48, 31, 33, 70, 3, 2, 1): "dma_64x64_splitk",
    (66, 48, 31, 33, 70, 3, 2, 1): "dma_128x128", (9, 21, 57, 55, 40, 3, 1, 1): "conv3x3_patch",
}
MORE = [(9, 64, 31, 30, 33, 3, 1, 1), (9, 32, 31, 33, 40, 1, 1, 1), (24, 48, 31, 33, 70, 3, 2, 1), (66, 48, 31, 33, 70, 3, 2, 1), (9, 21, 57, 55, 40, 3, 1, 1)]


@pytest.mark.parametrize("quant", ["u8", "u8pc", "s8", "s8pc"])
@pytest.mark.parametrize("case", CASES + MORE, ids=lambda c: "x".join(str(v) for v in c))
def test_planar_conv_per_channel_and_int8(case, quant):
    n, c, h, w, cout, k, stride, groups = case
    s = O.conv_shape(n, c, h, w, cout, k, k, stride=(stride, stride), pad=(k // 2,) * 4, groups=groups)
    red, pc, signed = c // groups * k * k, quant.endswith("pc"), quant.startswith("s8")
    x = synth.fill_u8((n, c, h, w), SEED + 21)
    wt = synth.fill_u8((cout, c // groups, k, k), SEED + 22)
    b = synth.fill_i32((cout,), SEED + 23, -1000, 1000)
    if signed:
        x = (x.astype(np.int16) - 128).astype(np.int8)
    if signed or pc:
        wt = (wt.astype(np.int16) - 128).astype(np.int8)
    pairs = None
    if pc:
        zp_in, zp_out = (-9, 5) if signed else (117, 131)
        scales = (0.002 * (1.0 + 9.0 * synth.fill_u8((cout,), SEED + 24) / 255.0)).astype(np.float32)
        q, *pairs = eden.make_requant_perchannel(0.02, zp_in, scales, float(0.02 * 0.02 * 74 * 74 * red ** 0.5 / 60), zp_out)
        oq = O.raw_quant(zp_in=zp_in, zp_w=0, zp_out=zp_out)
        if signed:
            q.act_min, q.act_max = oq.act_min, oq.act_max = -128, 127
        want = O.conv2d_s8(x, wt, b, s, oq, *pairs) if signed else O.conv2d_perchannel(x, wt, b, s, oq, *pairs)
    elif signed:
        oq = O.make_quant_s8(0.02, -11, 0.005, 3, 0.02 * 0.005 * 74 * 74 * red ** 0.5 / 40, -3)
        q, want = to_eh_requant(oq), O.conv2d_s8(x, wt, b, s, oq)
    else:
        oq = O.make_quant(0.02, 131, 0.005, 126, 0.02 * 0.005 * 74 * 74 * red ** 0.5 / 40, 120)
        q, want = to_eh_requant(oq), O.conv2d(x, wt, b, s, oq)
    desc = eden.conv_desc(n, c, h, w, cout, k, k, (stride,) * 2, (k // 2,) * 4, (1, 1), groups, 1, eden.NCHW | (eden.IO_SIGNED if signed else 0),
                          eden.W_OIHW | (eden.W_SIGNED if signed or pc else 0))
    if case in KERNELS:
        assert eden.conv_kernels(desc, launched=True) == [KERNELS[case]], eden.conv_kernels(desc, launched=True)
    d_x, d_w, d_b, d_o = eden.DeviceBuffer(host=x), eden.DeviceBuffer(host=wt), eden.DeviceBuffer(host=b), eden.DeviceBuffer(nbytes=want.size)
    plan = eden.ConvPlan(desc, d_w, d_b, q)
    if pairs:
        plan.set_perchannel(*pairs)
    plan.run(d_x, d_o, q)
    got = d_o.download(want.shape).view(want.dtype)
    assert np.array_equal(got, want), diff_report(got, want)
    assert want.std() > 4


# the tiled kernels write planar outputs as they compute them, of any size
@pytest.mark.parametrize("images,cout,kernel", [(41, 48, "dma_128x64"), (42, 48, "dma_128x64"), (20, 72, "dma_128x128"), (28, 72, "dma_128x128")])
def test_planar_tiled_kernels_on_both_sides_of_their_rule(images, cout, kernel):
    s = O.conv_shape(images, 16, 57, 57, cout, 2, 2)
    assert (images * 56 * 56 * cout <= 6 << 20) == (images in (41, 20))
    assert eden.conv_kernels(eden.conv_desc(images, 16, 57, 57, cout, 2, 2, layout=eden.NCHW), launched=True) == [kernel]
    x, wt = synth.fill_u8((images, 16, 57, 57), SEED + 31), synth.fill_u8((cout, 16, 2, 2), SEED + 32)
    b = synth.fill_i32((cout,), SEED + 33, -1000, 1000)
    q = O.make_quant(0.02, 131, 0.005, 126, 0.02 * 0.005 * 74 * 74 * 8 / 40, 120)
    want, got = O.conv2d(x, wt, b, s, q), gpu_conv(x, wt, b, s, to_eh_requant(q), layout=eden.NCHW)
    assert np.array_equal(got, want), diff_report(got, want)
    assert want.std() > 4


@pytest.mark.parametrize("case", [(2, 64, 7, 9, 21, 4, 2), (1, 48, 9, 8, 33, 3, 2), (3, 20, 6, 5, 7, 2, 2)], ids=lambda c: "x".join(str(v) for v in c))
def test_planar_deconv(case):
    n, c, h, w, cout, k, stride = case
    s = O.conv_shape(n, c, h, w, cout, k, k, stride=(stride, stride), pad=((k - stride) // 2,) * 4)
    x, wt = synth.fill_u8((n, c, h, w), SEED + 11), synth.fill_u8((c, cout, k, k), SEED + 12)
    b = synth.fill_i32((cout,), SEED + 13, -1000, 1000)
    q = O.make_quant(0.02, 121, 0.005, 133, 0.02 * 0.005 * 74 * 74 * (c * 4) ** 0.5 / 40, 128)
    want, got = O.deconv2d(x, wt, b, s, q), gpu_deconv(x, wt, b, s, to_eh_requant(q), layout=eden.NCHW)
    assert np.array_equal(got, want), diff_report(got, want)
    assert want.std() > 4
