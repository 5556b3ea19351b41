"""The kernel for few tiles on tensors that it reads as they are: channel counts off 16 (chunks at any address, the last ones ending behind
the tensor) and planar tensors, uint8 and int8, of convolutions, transposed ones and with a fused residual add, against the oracle.  The tensors lie at the end of their allocation's own bytes, one byte in, so that
no alignment is there by chance."""
import numpy as np
import pytest

import oracle_lib as O
from harness import diff_report, eden, gpu_fc, synth, to_eh_requant

pytestmark = pytest.mark.gpu
SEED = 0xEDE2 + 16 * 27


@pytest.mark.parametrize("m,k,n", [(1, 17, 3), (1, 16 * 9 + 15, 40), (2, 9, 5), (31, 33, 33), (33, 127, 31), (128, 129, 64), (7, 1025, 12), (3, 3506, 37), (900, 250, 90), (1, 8191, 20)])
@pytest.mark.parametrize("signed", [False, True])
def test_fc(m, k, n, signed):
    print("fc", m, k, n, signed, flush=True)
    a, w, b = synth.fill_u8((m, k), SEED + 1), synth.fill_u8((n, k), SEED + 2), synth.fill_i32((n,), SEED + 3, -1000, 1000)
    s_out = float(0.02 * 0.005 * 74.0 * 74.0 * np.sqrt(k) / 50.0)
    if signed:
        a, w = (a.astype(np.int16) - 128).astype(np.int8), (w.astype(np.int16) - 128).astype(np.int8)
        want = O.fc_s8(a, w, b, O.make_quant_s8(0.02, -11, 0.005, 3, s_out, -3))
        got = gpu_fc(a, w, b, eden.make_requant_s8(0.02, -11, 0.005, 3, s_out, -3), eden.IO_SIGNED | eden.W_SIGNED).view(np.int8)
    else:
        q = O.make_quant(0.02, 117, 0.005, 131, s_out, 120)
        want, got = O.fc(a, w, b, q), gpu_fc(a, w, b, to_eh_requant(q))
    assert np.array_equal(got, want), diff_report(got, want)


@pytest.mark.parametrize("pc", [False, True])
@pytest.mark.parametrize("layout", [eden.NHWC, eden.NCHW])
@pytest.mark.parametrize("n,c,h,w,cout,k,stride,dil,groups", [
    (1, 21, 9, 7, 5, 3, 1, 1, 1), (3, 17, 5, 6, 33, 3, 2, 1, 1), (2, 40, 11, 13, 24, 3, 1, 2, 1), (2, 23, 8, 8, 40, 1, 1, 1, 1), (1, 115, 6, 5, 7, 1, 2, 1, 1),
    (2, 26, 9, 9, 14, 3, 1, 1, 2), (1, 9, 17, 19, 12, 5, 1, 1, 1), (1, 5, 3, 3, 70, 3, 1, 1, 1), (2, 64, 12, 9, 30, 1, 1, 1, 1), (1, 100, 9, 9, 20, 3, 1, 1, 1), (3, 21, 65, 47, 21, 3, 1, 1, 1),
])
def test_conv(n, c, h, w, cout, k, stride, dil, groups, layout, pc):
    print("conv", n, c, h, w, cout, k, stride, dil, groups, layout, pc, flush=True)
    pad = dil * (k - 1) // 2
    s = O.conv_shape(n, c, h, w, cout, k, k, stride=(stride, stride), pad=(pad,) * 4, dil=(dil, dil), groups=groups)
    x, b = synth.fill_u8((n, c, h, w), SEED + 4), synth.fill_i32((cout,), SEED + 6, -1000, 1000)
    wt = synth.fill_u8((cout, c // groups, k, k), SEED + 5)
    scale = 74.0 * 74.0 * np.sqrt(c // groups * k * k)
    pairs = ()
    if pc:
        wt = (wt.astype(np.int16) - 128).astype(np.int8)
        w_scales = (0.002 * (1.0 + 9.0 * synth.fill_u8((cout,), SEED + 7) / 255.0)).astype(np.float32)
        q, *pairs = eden.make_requant_perchannel(0.02, 117, w_scales, float(0.02 * 0.02 * scale / 60.0), 131)
        want = O.conv2d_perchannel(x, wt, b, s, O.raw_quant(zp_in=117, zp_w=0, zp_out=131), *pairs)
    else:
        oq = O.make_quant(0.02, 131, 0.005, 117, float(0.02 * 0.005 * scale / 40.0), 120)
        q, want = to_eh_requant(oq), O.conv2d(x, wt, b, s, oq)
    desc = eden.conv_desc(n, c, h, w, cout, k, k, (stride, stride), (pad,) * 4, (dil, dil), groups, 1, layout, eden.W_OIHW | (eden.W_SIGNED if pc else 0))
    assert set(eden.conv_kernels(desc, launched=True)) == {"few_tiles"}
    flat = np.ascontiguousarray(x if layout == eden.NCHW else x.transpose(0, 2, 3, 1)).reshape(-1)
    d_x = eden.BufferView(eden.DeviceBuffer(host=np.concatenate([[7], flat]).astype(np.uint8)), 1)
    d_w, d_b, d_o = eden.DeviceBuffer(host=wt), eden.DeviceBuffer(host=b), eden.DeviceBuffer(nbytes=want.size)
    plan = eden.ConvPlan(desc, d_w, d_b, q)
    if pc:
        plan.set_perchannel(*pairs)
    if layout == eden.NHWC and c // groups % 16 == 0:   # (whole chunks are read as such, from aligned tensors)
        d_x = eden.DeviceBuffer(host=flat)
    for _ in range(2):
        plan.run(d_x, d_o, q)
    ho, wo = O.conv_out_hw(s)
    got = d_o.download((n, cout, ho, wo)) if layout == eden.NCHW else d_o.download((n, ho, wo, cout)).transpose(0, 3, 1, 2)
    plan.destroy()
    assert np.array_equal(got, want), diff_report(got, want)


@pytest.mark.parametrize("layout", [eden.NHWC, eden.NCHW])
@pytest.mark.parametrize("deconv,n,c,h,w,cout,k,stride", [(False, 2, 21, 9, 7, 13, 3, 1), (False, 1, 37, 12, 11, 40, 1, 1), (False, 3, 10, 8, 13, 9, 5, 2),
                                                        (True, 2, 23, 7, 9, 17, 3, 1), (True, 1, 40, 6, 5, 24, 3, 2), (True, 2, 20, 5, 6, 33, 4, 2)])
def test_int8_and_transposed(deconv, n, c, h, w, cout, k, stride, layout):
    print("int8", deconv, n, c, h, w, cout, k, stride, layout, flush=True)
    pad = ((k - stride) // 2 if deconv else k // 2,) * 4
    s = O.conv_shape(n, c, h, w, cout, k, k, stride=(stride, stride), pad=pad)
    x, b = synth.fill_u8((n, c, h, w), SEED + 8), synth.fill_i32((cout,), SEED + 10, -1000, 1000)
    wt = synth.fill_u8((c, cout, k, k) if deconv else (cout, c, k, k), SEED + 9)
    x, wt = (x.astype(np.int16) - 128).astype(np.int8), (wt.astype(np.int16) - 128).astype(np.int8)
    s_out = float(0.02 * 0.005 * 74.0 * 74.0 * np.sqrt(c * max(1, k // stride if deconv else k) ** 2) / 40.0)
    want = (O.deconv2d_s8 if deconv else O.conv2d_s8)(x, wt, b, s, O.make_quant_s8(0.02, -11, 0.005, 3, s_out, -3))
    q = eden.make_requant_s8(0.02, -11, 0.005, 3, s_out, -3)
    desc = eden.conv_desc(n, c, h, w, cout, k, k, (stride, stride), pad, layout=layout | eden.IO_SIGNED, weight_layout=(eden.W_IOHW if deconv else eden.W_OIHW) | eden.W_SIGNED)
    assert set(eden.conv_kernels(desc, deconv, launched=True)) == {"few_tiles"}
    nhwc = layout == eden.NHWC
    flat = np.ascontiguousarray(x.transpose(0, 2, 3, 1) if nhwc else x).view(np.uint8).reshape(-1)
    d_x = eden.BufferView(eden.DeviceBuffer(host=np.concatenate([[7], flat]).astype(np.uint8)), 1)
    d_w, d_b, d_o = eden.DeviceBuffer(host=wt), eden.DeviceBuffer(host=b), eden.DeviceBuffer(nbytes=want.size)
    (eden.DeconvPlan if deconv else eden.ConvPlan)(desc, d_w, d_b, q).run(d_x, d_o, q)
    ho, wo = want.shape[2:]
    got = (d_o.download((n, ho, wo, cout)).transpose(0, 3, 1, 2) if nhwc else d_o.download((n, cout, ho, wo))).view(np.int8)
    assert np.array_equal(got, want), diff_report(got, want)
    assert want.std() > 4


@pytest.mark.parametrize("n,c,h,w,cout,k", [(2, 21, 9, 7, 13, 1), (1, 37, 12, 11, 48, 1), (2, 26, 9, 9, 32, 3)])
def test_residual_add(n, c, h, w, cout, k):
    print("residual", n, c, h, w, cout, k, flush=True)
    pad = (k // 2,) * 4
    s = O.conv_shape(n, c, h, w, cout, k, k, pad=pad)
    x, b = synth.fill_u8((n, c, h, w), SEED + 11), synth.fill_i32((cout,), SEED + 12, -1000, 1000)
    wt, res = synth.fill_u8((cout, c, k, k), SEED + 13), synth.fill_u8((n, cout, h, w), SEED + 14)
    s_out = float(0.02 * 0.005 * 74.0 * 74.0 * np.sqrt(c * k * k) / 40.0)
    q = O.make_quant(0.02, 131, 0.005, 117, s_out, 120)
    want = O.add(res, O.conv2d(x, wt, b, s, q), O.make_add_quant(0.05, 120, s_out, 120, 0.07, 128))
    aq, e = eden.make_add_requant(0.05, 120, s_out, 120, 0.07, 128), to_eh_requant(q)
    d_x = eden.BufferView(eden.DeviceBuffer(host=np.concatenate([[7], x.transpose(0, 2, 3, 1).ravel()]).astype(np.uint8)), 1)
    d_w, d_b, d_r = eden.DeviceBuffer(host=wt), eden.DeviceBuffer(host=b), eden.DeviceBuffer(host=res.transpose(0, 2, 3, 1))
    d_o = eden.DeviceBuffer(nbytes=want.size)
    plan = eden.ConvPlan(eden.conv_desc(n, c, h, w, cout, k, k, (1, 1), pad, layout=eden.NHWC), d_w, d_b, e)
    plan.run_add(d_x, d_r, d_o, e, aq)
    got = d_o.download((n, h, w, cout)).transpose(0, 3, 1, 2)
    assert np.array_equal(got, want), diff_report(got, want)
    assert want.std() > 4
