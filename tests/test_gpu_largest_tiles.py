"""The 256 x 256 tiles (240 of them or more in a launch) against the oracle, beyond what whole 16-byte stores and row sums cover: weights
whose zero point is their own (no row sums), a pair per channel, output rows on and off 16-byte boundaries, edge tiles."""
import numpy as np
import pytest

import oracle_lib as O
from harness import eden, gpu_conv, gpu_fc, synth, to_eh_requant

pytestmark = pytest.mark.gpu
SEED = 0xEDE2 + 16 * 23


@pytest.mark.parametrize("m,k,n", [(7937, 272, 2034), (7700, 256, 2112), (8000, 129, 1930)])
@pytest.mark.parametrize("zp_w", [0, 9])
def test_fc_s8(m, k, n, zp_w):
    assert (m + 255) // 256 * ((n + 255) // 256) >= 240   # what the largest tile is chosen from
    print("fc", m, k, n, zp_w, flush=True)
    a = (synth.fill_u8((m, k), SEED + 1).astype(np.int16) - 128).astype(np.int8)
    w = (synth.fill_u8((n, k), SEED + 2).astype(np.int16) - 128).astype(np.int8)
    b = synth.fill_i32((n,), SEED + 3, -1000, 1000)
    s_out = float(0.02 * 0.005 * 74.0 * 74.0 * np.sqrt(k) / 50.0)
    want = O.fc_s8(a, w, b, O.make_quant_s8(0.02, -11, 0.005, zp_w, s_out, -3))
    got = gpu_fc(a, w, b, eden.make_requant_s8(0.02, -11, 0.005, zp_w, s_out, -3), eden.IO_SIGNED | eden.W_SIGNED).view(np.int8)
    assert np.array_equal(got, want)
    assert want.std() > 20


@pytest.mark.parametrize("deconv,n,c,h,cout,k,stride", [
    (False, 9, 240, 85, 232, 1, 1),     # (a reduction that ends inside its last slab: table-driven)
    (False, 9, 16, 85, 250, 5, 1),      # rows of 250 bytes
    (True, 4, 48, 45, 40, 16, 8),       # four kernel columns side by side, rows of 160 bytes at distances of 320
    (True, 5, 32, 45, 37, 16, 8),
])
def test_a_pair_per_channel(deconv, n, c, h, cout, k, stride):
    print("per channel", deconv, n, c, h, cout, k, stride, flush=True)
    pad = (k - stride) // 2
    s = O.conv_shape(n, c, h, h, cout, k, k, stride=(stride, stride), pad=(pad,) * 4)
    x = synth.fill_u8((n, c, h, h), SEED + 4)
    w = (synth.fill_u8((c, cout, k, k) if deconv else (cout, c, k, k), SEED + 5).astype(np.int16) - 128).astype(np.int8)
    b = synth.fill_i32((cout,), SEED + 6, -500, 500)
    w_scales = (0.002 * (1.0 + 29.0 * synth.fill_u8((cout,), SEED + 7) / 255.0)).astype(np.float32)
    taps = (k // stride) ** 2 if deconv else k * k
    s_out = float(0.02 * float(w_scales.max()) * 74.0 * 74.0 * np.sqrt(taps * c) / 60.0)
    q, mults, shifts = eden.make_requant_perchannel(0.02, 117, w_scales, s_out, 131)
    oq = O.raw_quant(zp_in=117, zp_w=0, zp_out=131)
    want = (O.deconv2d_perchannel if deconv else O.conv2d_perchannel)(x, w, b, s, oq, mults, shifts)
    ho, wo = (O.deconv_out_hw if deconv else O.conv_out_hw)(s)
    desc = eden.conv_desc(n, c, h, h, cout, k, k, (stride, stride), (pad,) * 4, layout=eden.NHWC, weight_layout=(eden.W_IOHW if deconv else eden.W_OIHW) | eden.W_SIGNED)
    assert "dma_256x256" in eden.conv_kernels(desc, deconv, True)
    d_x, d_w, d_b = eden.DeviceBuffer(host=x.transpose(0, 2, 3, 1)), eden.DeviceBuffer(host=w), eden.DeviceBuffer(host=b)
    d_o = eden.DeviceBuffer(nbytes=n * cout * ho * wo)
    plan = (eden.DeconvPlan if deconv else eden.ConvPlan)(desc, d_w, d_b, q)
    plan.set_perchannel(mults, shifts)
    plan.run(d_x, d_o, q)
    got = d_o.download((n, ho, wo, cout)).transpose(0, 3, 1, 2)
    plan.destroy()
    assert np.array_equal(got, want)
    assert want.std() > 4


# row sums (weights around a zero point of their own), shared by the waves of a row block where a SIMD runs two of them
@pytest.mark.parametrize("n,c,h,cout,k,dil,kernel", [
    (21, 128, 28, 121, 3, 2, "dma_128x128"),   # at most one tile per CU
    (13, 16, 71, 250, 5, 1, "dma_256x256"),
    (20, 16, 57, 72, 2, 1, "dma_128x128"),     # one slab
    (30, 16, 57, 72, 3, 2, "dma_128x128"),     # more tiles than CUs
])
def test_row_sums(n, c, h, cout, k, dil, kernel):
    print("row sums", n, c, h, cout, k, dil, kernel, flush=True)
    pad = dil * (k - 1) // 2
    s = O.conv_shape(n, c, h, h, cout, k, k, pad=(pad,) * 4, dil=(dil, dil))
    desc = eden.conv_desc(n, c, h, h, cout, k, k, (1, 1), (pad,) * 4, (dil, dil), layout=eden.NHWC)
    assert eden.conv_kernels(desc, launched=True) == [kernel]
    x, w = synth.fill_u8((n, c, h, h), SEED + 8), synth.fill_u8((cout, c, k, k), SEED + 9)
    b = synth.fill_i32((cout,), SEED + 10, -1000, 1000)
    q = O.make_quant(0.02, 131, 0.005, 117, 0.02 * 0.005 * 74 * 74 * (c * k * k) ** 0.5 / 40, 120)
    want, got = O.conv2d(x, w, b, s, q), gpu_conv(x, w, b, s, to_eh_requant(q), layout=eden.NHWC)
    assert np.array_equal(got, want)
    assert want.std() > 20
