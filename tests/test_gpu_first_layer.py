"""The first-layer convolution (three channels, 3x3) where a row's twelve bytes would leave the tensor: images of one to five pixels,
whose rows are shifted into place or read byte by byte, windows that hang over every edge, and the last pixels of an ordinary image;
bit for bit the oracle, for the matrix cores' kernel (32 channels on) and the vector one."""
import numpy as np
import pytest

import oracle_lib as O
from harness import diff_report, eden, gpu_conv, synth, to_eh_requant

pytestmark = pytest.mark.gpu
SEED = 0xF125

SHAPES = [
    # n, h, w, stride, pad
    (1, 1, 1, 1, 1), (1, 1, 3, 1, 1), (3, 1, 1, 1, 1),   # at most nine bytes
    (1, 1, 4, 1, 1), (4, 1, 1, 1, 1), (1, 4, 1, 2, 1), (2, 1, 2, 1, 1),   # exactly twelve
    (1, 1, 5, 1, 2), (1, 5, 1, 1, 2), (5, 1, 1, 1, 2),   # shifts by one and two pixels at both ends
    (2, 2, 3, 1, 1), (1, 3, 3, 1, 0), (1, 6, 4, 1, 0),   # no padding: the last row ends with the tensor
    (2, 9, 11, 2, 1), (1, 13, 37, 1, 2),
]


@pytest.mark.parametrize("cout", [20, 32, 72])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(str(v) for v in s))
def test_first_layer_matches_oracle(shape, cout):
    n, h, w, stride, pad = shape
    print("first layer", shape, cout, flush=True)
    x, wt = synth.fill_u8((n, 3, h, w), SEED + h * 64 + w), synth.fill_u8((cout, 3, 3, 3), SEED + cout)
    bias = synth.fill_i32((cout,), SEED + 1, -1000, 1000)
    s = O.conv_shape(n, 3, h, w, cout, 3, 3, stride=(stride, stride), pad=(pad,) * 4)
    q = O.make_quant(0.02, 117, 0.004, 121, 0.05, 128)
    want, got = O.conv2d(x, wt, bias, s, q), gpu_conv(x, wt, bias, s, to_eh_requant(q), layout=eden.NHWC)
    assert np.array_equal(got, want), diff_report(got, want)
    assert want.std() > 1
