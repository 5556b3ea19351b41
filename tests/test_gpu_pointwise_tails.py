"""The one-tap kernel over reduction lengths around its step of 32 bytes: last steps of 8, 16, 24 and 32 bytes, which lanes read from
the pixel's first bytes where they lie past the end, every number of steps up to eight, one and several channel blocks, pixel counts
that end inside a block of 32; bit for bit the oracle, with one pair and with one pair per channel."""
import numpy as np
import pytest

import oracle_lib as O
from harness import diff_report, eden, synth, to_eh_requant

pytestmark = pytest.mark.gpu
SEED = 0x7A11
LENGTHS = [8, 16, 24, 32, 40, 48, 56, 64, 72, 96, 104, 128, 136, 144, 160, 184, 192, 200, 216, 224, 240, 256]


@pytest.mark.parametrize("per_channel", [False, True], ids=["tensor", "channel"])
@pytest.mark.parametrize("cout", [20, 72])
@pytest.mark.parametrize("c", LENGTHS)
def test_one_tap_tails_match_oracle(c, cout, per_channel):
    n, h, w = 3, 63, 61   # 11529 pixels: the last block holds nine
    print("one tap", c, cout, per_channel, flush=True)
    x, wt = synth.fill_u8((n, c, h, w), SEED + c), synth.fill_u8((cout, c, 1, 1), SEED + cout)
    bias = synth.fill_i32((cout,), SEED + 1, -1000, 1000)
    s = O.conv_shape(n, c, h, w, cout, 1, 1)
    q = O.make_quant(0.02, 117, 0.004, 121, 0.02 * 0.004 * 74 * 74 * c ** 0.5 / 40, 128)
    e = to_eh_requant(q)
    keep = [eden.DeviceBuffer(host=a) for a in (np.ascontiguousarray(x.transpose(0, 2, 3, 1)), wt, bias)]
    d_o = eden.DeviceBuffer(nbytes=n * cout * h * w)
    plan = eden.ConvPlan(eden.conv_desc(n, c, h, w, cout, 1, 1, layout=eden.NHWC), keep[1], keep[2], e)
    if per_channel:   # the tensor's own pair for every channel: the same results through the per-channel code
        plan.set_perchannel(np.full(cout, e.multiplier), np.full(cout, e.shift))
    plan.run(keep[0], d_o, e)
    got, want = d_o.download((n, h, w, cout)).transpose(0, 3, 1, 2), O.conv2d(x, wt, bias, s, q)
    assert np.array_equal(got, want), diff_report(got, want)
    assert want.std() > 1
