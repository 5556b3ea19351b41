"""What is launched, without a GPU: the library runs on a stand-in for the HIP runtime (tests/hip_stub.cpp) that notes each
launch's kernel and grid."""
import os
import re
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)

PRELUDE = """
import importlib, sys
import numpy as np
sys.path.insert(0, %r)
eden = importlib.import_module("cl-eden-kernel_amd")
eden.init(0)
q = eden.make_requant(0.02, 117, 0.004, 121, 0.03, 5)
def buf(*shape, dtype=np.uint8):
    return eden.DeviceBuffer(host=np.full(shape, 121, dtype))
def run(plan_type, n, c, h, cout, k, stride):
    out = h * stride if plan_type is eden.DeconvPlan else h
    w = (c, cout, k, k) if plan_type is eden.DeconvPlan else (cout, c, k, k)
    desc = eden.conv_desc(n, c, h, h, cout, k, k, (stride, stride), layout=eden.NHWC,
                          weight_layout=eden.W_IOHW if plan_type is eden.DeconvPlan else eden.W_OIHW)
    plan_type(desc, buf(*w), buf(cout, dtype=np.int32), q).run(buf(n, h, h, c), eden.DeviceBuffer(nbytes=n * out * out * cout), q)
""" % ROOT


@pytest.fixture(scope="module")
def stub(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("stub") / "hip_stub.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-shared", "-fPIC", os.path.join(HERE, "hip_stub.cpp"), "-o", so], check=True)
    return so


def launches(stub, tmp_path, program, full=""):
    """[(kernel, grid x, y, z, LDS bytes)] of a program on the stand-in"""
    log = tmp_path / "launches"
    log.write_text("")
    env = dict(os.environ, LD_PRELOAD=stub, HIP_STUB_LOG=str(log), HIP_STUB_FULL=full)
    subprocess.run([sys.executable, "-c", PRELUDE + program], check=True, env=env, cwd=ROOT)
    return [(a[0],) + tuple(int(v) for v in a[1:]) for a in (line.split() for line in log.read_text().splitlines())]


def test_one_tap_grid_does_not_depend_on_what_ran_before(stub, tmp_path):
    """96 -> 16 channels as the four phases of a transposed convolution (one launch of the batched kernel) and 96 -> 24 as a
    convolution (the plain one), of equal LDS: each grid follows its own kernel's occupancy, in either order."""
    batched, plain = "run(eden.DeconvPlan, 16, 96, 56, 16, 2, 2)\n", "run(eden.ConvPlan, 64, 96, 56, 24, 1, 1)\n"
    grids = []
    for program in (batched + plain, plain + batched):
        own = sorted(l for l in launches(stub, tmp_path, program, full="ELb0ELb1ELb0EEEv") if "direct_gemm_kernel" in l[0])
        assert len(own) == 2 and {l[3] for l in own} == {1, 4} and own[0][4] == own[1][4], own
        grids.append(own)
    assert grids[0] == grids[1]


@pytest.mark.parametrize("desc,packs", [
    ("1, 32, 9, 9, 32, 3, 3, (1, 1), (1, 1, 1, 1)", 1),
    ("1, 32, 9, 9, 32, 3, 3, (2, 2), (0, 1, 0, 1)", 1),
    ("1, 32, 9, 9, 32, 3, 3, (3, 3), (1, 1, 1, 1)", 0),
    ("1, 32, 9, 9, 32, 3, 3, (1, 1), (2, 2, 2, 2), (2, 2)", 0),
    ("1, 24, 9, 9, 24, 3, 3, (1, 1), (1, 1, 1, 1)", 0),
    ("1, 16, 9, 9, 32, 3, 3, (1, 1), (1, 1, 1, 1), (1, 1), 1, 2", 0),
    ("1, 32, 9, 9, 32, 3, 3, (1, 1), (1, 1, 1, 1), layout=eden.NCHW", 0),
    ("1, 32, 9, 9, 32, 3, 3, (1, 1), (1, 1, 1, 1), layout=eden.NHWC | eden.IO_SIGNED", 0),
    ("1, 20, 9, 9, 20, 5, 5, (1, 1), (2, 2, 2, 2)", 1),
])
def test_matrix_form_of_depthwise_weights_is_packed_where_a_kernel_reads_it(stub, tmp_path, desc, packs):
    """5x5 and 7x7 layers, and of the 3x3 ones those that the fused expansion + depthwise launch can end with."""
    if "layout" not in desc:
        desc += ", layout=eden.NHWC"
    if "dm" not in desc and ", 1, 2" not in desc:
        desc += ", dm=1"
    program = """
d = eden.conv_desc(%s)
if d.layout & eden.IO_SIGNED:
    q = eden.make_requant_s8(0.02, 3, 0.004, 121, 0.03, 5)
plan = eden.DwConvPlan(d, buf(d.cout, 1, d.kh, d.kw), buf(d.cout, dtype=np.int32), q)
""" % desc
    assert sum("dw_pack_mfma_kernel" in l[0] for l in launches(stub, tmp_path, program)) == packs


@pytest.mark.parametrize("shape,tile,tensor,channel,own", [
    # n, cin, expanded, extent, stride; rows and columns asked for; whether the library's own tile takes units
    ((1, 32, 64, 28, 2), (2, 4), 1, 1, 0),      # four units of sixteen outputs by sixteen channels, half full
    ((1, 32, 96, 28, 2), (2, 4), 0, 0, 0),      # six, half full
    ((4, 24, 144, 56, 2), (2, 8), 0, 0, 1),     # nine at stride 2
    ((4, 16, 96, 14, 1), (4, 4), 1, 0, 0),      # six, full
    ((4, 32, 128, 28, 2), (4, 4), 1, 0, 1),     # eight, full
    ((4, 16, 64, 28, 1), (3, 5), 1, 0, 0),      # four
    ((4, 16, 48, 28, 1), (3, 5), 1, 1, 0),      # three
    ((4, 96, 576, 14, 1), (7, 14), 0, 0, 0),    # many
])
def test_form_of_the_fused_launchs_depthwise_stage(stub, tmp_path, shape, tile, tensor, channel, own):
    """Units of sixteen outputs for small tiles that are asked for, with one pair per tensor and with one per channel, where they are the faster
    form; tiles of the library's own choice walk, but for some at stride 2; the plan notices that its pairs and the requested tile have changed."""
    program = """
n, cin, c, h, stride = %r
pw = eden.ConvPlan(eden.conv_desc(n, cin, h, h, c, 1, 1, layout=eden.NHWC), buf(c, cin, 1, 1), buf(c, dtype=np.int32), q)
dw = eden.DwConvPlan(eden.conv_desc(n, c, h, h, c, 3, 3, (stride,) * 2, (1,) * 4, dm=1, layout=eden.NHWC), buf(c, 1, 3, 3), buf(c, dtype=np.int32), q)
forms = []
for pairs in (False, True, False):
    for plan in (pw, dw):
        plan.set_perchannel(*((np.full(c, q.multiplier), np.full(c, q.shift)) if pairs else (None, None)))
    forms += [eden.conv_dw_block_tile(pw, dw, *%r)[3], eden.conv_dw_block_tile(pw, dw)[3]]
assert forms == [%d, %d, %d, %d, %d, %d], forms
""" % (shape, tile, tensor, own, channel, own, tensor, own)
    launches(stub, tmp_path, program)


@pytest.mark.parametrize("shape", [
    # n, cin, expanded, height, width, stride, a pair per channel
    (11, 152, 912, 17, 17, 1, True),     # 65 workgroups to an XCD that holds 64
    (7, 96, 576, 37, 37, 1, True),       # 99, 96
    (22, 24, 144, 77, 77, 2, False),     # three workgroups of 54336 bytes fill 160 KB, and two of the 55040 that are given out
    (37, 40, 240, 75, 79, 1, False),     # 54080
    (4, 72, 432, 106, 106, 2, False),    # 54592
])
def test_rounds_of_a_fused_launch_are_counted_as_the_hardware_deals_them_out(stub, tmp_path, shape):
    """The tile of a fused launch is chosen by its rounds of workgroups: those that the launch has on XCDs of 32 CUs with whole tiles and LDS in
    pieces of 1280 bytes are no more than an even split of everything would have."""
    program = """
import os
n, cin, c, h, w, stride, pairs = %r
pw = eden.ConvPlan(eden.conv_desc(n, cin, h, w, c, 1, 1, layout=eden.NHWC), buf(c, cin, 1, 1), buf(c, dtype=np.int32), q)
dw = eden.DwConvPlan(eden.conv_desc(n, c, h, w, c, 3, 3, (stride,) * 2, (1,) * 4, dm=1, layout=eden.NHWC), buf(c, 1, 3, 3), buf(c, dtype=np.int32), q)
for plan in (pw, dw):
    plan.set_perchannel(*((np.full(c, q.multiplier), np.full(c, q.shift)) if pairs else (None, None)))
ho, wo = (h - 1) // stride + 1, (w - 1) // stride + 1
eden.conv_dw_block_run(pw, dw, buf(n, h, w, cin), eden.DeviceBuffer(nbytes=n * ho * wo * c), q, eden.make_requant(0.02, 5, 0.004, 121, 0.03, 5))
rows, cols = eden.conv_dw_block_tile(pw, dw)[:2]
print("tiles", n * -(-ho // rows) * -(-wo // cols), file=open(os.environ["HIP_STUB_LOG"], "a"))
""" % (shape,)
    log = launches(stub, tmp_path, program)
    (_, x, y, _, lds), = [l for l in log if "pwdw_block_kernel" in l[0]]
    tiles, held = log[-1][1], 4 if shape[-1] else 5   # by their registers
    ceil = lambda a, b: -(-a // b)
    even = ceil(tiles * y, 256 * min(held, 163840 // lds))
    dealt = ceil(ceil(tiles, 8) * y, 32 * min(held, 163840 // (ceil(lds, 1280) * 1280)))
    assert x == ceil(tiles, 8) * 8 and dealt <= even, (tiles, y, lds, dealt, even)


@pytest.mark.parametrize("module,kernel", [("test_gpu_dw_planar", r"dw_planar_kernelI"), ("test_gpu_dw_gather", r"dw3x3_nhwc_tile4_dot4_kernelI.*ELb1EEEv")])
def test_depthwise_tensors_are_read_as_they_are(stub, tmp_path, module, kernel):
    """The cases of the two tests against the oracle take the kernels that those tests are for, in every form."""
    program = """
import os
sys.path.insert(0, %r)
import %s as m
for case in m.CASES:
    n, c, dm, h, w = case[:5]
    planar = m.__name__.endswith("planar")
    k, stride = (case[5], case[6]) if planar else (3, case[5])
    pad = case[8] if len(case) > 8 else (k // 2,) * 4
    for signed in (False, True):
        e = eden.make_requant_s8(0.02, 9, 0.004, 0, 0.1, -4) if signed else q
        desc = eden.conv_desc(n, c, h, w, c * dm, k, k, stride=(stride, stride), pad=pad, dm=dm, layout=(eden.NCHW if planar else eden.NHWC) | (eden.IO_SIGNED if signed else 0),
                              weight_layout=eden.W_OIHW | (eden.W_SIGNED if signed else 0))
        plan = eden.DwConvPlan(desc, buf(c * dm, 1, k, k), buf(c * dm, dtype=np.int32), e)
        ho, wo = (h + pad[0] + pad[1] - k) // stride + 1, (w + pad[2] + pad[3] - k) // stride + 1
        x, o = eden.DeviceBuffer(nbytes=n * c * h * w), eden.DeviceBuffer(nbytes=n * c * dm * ho * wo)
        for pairs in (False, True):
            if pairs:
                plan.set_perchannel(np.full(c * dm, 1 << 30), np.full(c * dm, -6))
            print("run", file=open(os.environ["HIP_STUB_LOG"], "a"))
            plan.run(x, o, e)
            print("end", file=open(os.environ["HIP_STUB_LOG"], "a"))
""" % (HERE, module)
    names, runs = [r[0] for r in launches(stub, tmp_path, program)], []
    while "run" in names:
        start, end = names.index("run"), names.index("end")
        runs.append(names[start + 1:end])
        names = names[end + 1:]
    assert len(runs) >= 40 and all(len(r) == 1 and re.search(kernel, r[0]) for r in runs), [r for r in runs if len(r) != 1 or not re.search(kernel, r[0])][:3]


@pytest.mark.parametrize("plan,in_bytes,out_bytes,direct", [
    # rows few enough for the few-row kernel: k to 2560
    ("fc(3, 2555, 798)", 3 * 2555, 3 * 798, True),
    ("fc(3, 3609, 798)", 3 * 3609, 3 * 798, False),
    ("fc(21, 3480, 294)", 21 * 3480, 21 * 294, True),
    # one round of tiles: k to 3500
    ("conv(1, 378, 9, 40, 3)", 378 * 81, 40 * 81, True),
    ("conv(1, 426, 13, 11, 3)", 426 * 169, 11 * 169, False),
    # two: k to 1024, one tap to 2208
    ("conv(4, 97, 42, 45, 3)", 4 * 97 * 1764, 4 * 45 * 1764, True),
    ("conv(4, 21, 42, 45, 7)", 4 * 21 * 1764, 4 * 45 * 1764, False),
    ("fc(637, 2204, 477)", 637 * 2204, 637 * 477, True),
    # four: one tap only
    ("conv(2, 238, 66, 42, 1)", 2 * 238 * 4356, 2 * 42 * 4356, True),
    ("conv(2, 50, 66, 42, 2)", 2 * 50 * 4356, 2 * 42 * 65 * 65, False),
    # planar: k to 576, one tap to 1152
    ("conv(1, 60, 20, 40, 3, eden.NCHW)", 60 * 400, 40 * 400, True),
    ("conv(1, 80, 20, 40, 3, eden.NCHW)", 80 * 400, 40 * 400, False),
    ("conv(4, 48, 48, 20, 3, eden.NCHW)", 4 * 48 * 2304, 4 * 20 * 2304, True),    # 288 tiles: to 432
    ("conv(4, 64, 48, 20, 3, eden.NCHW)", 4 * 64 * 2304, 4 * 20 * 2304, False),
    ("conv(1, 880, 20, 40, 1, eden.NCHW)", 880 * 400, 40 * 400, True),
    ("conv(1, 1168, 20, 40, 1, eden.NCHW)", 1168 * 400, 40 * 400, False),
])
def test_ragged_and_planar_tensors_are_read_as_they_are_where_that_is_faster(stub, tmp_path, plan, in_bytes, out_bytes, direct):
    program = """
bias = lambda n: buf(n, dtype=np.int32)
def fc(m, k, n):
    return eden.FcPlan(m, k, n, buf(n, k), bias(n), q)
def conv(n, c, h, cout, k, layout=eden.NHWC):
    return eden.ConvPlan(eden.conv_desc(n, c, h, h, cout, k, k, (1, 1), ((k - 1) // 2,) * 4, layout=layout), buf(cout, c, k, k), bias(cout), q)
plan = %s
import os
print("run", file=open(os.environ["HIP_STUB_LOG"], "a"))
plan.run(eden.DeviceBuffer(nbytes=%d), eden.DeviceBuffer(nbytes=%d), q)
""" % (plan, in_bytes, out_bytes)
    names = [r[0] for r in launches(stub, tmp_path, program)]
    names = names[names.index("run") + 1:]
    assert (len(names) == 1 and "few_tiles" in names[0]) if direct else len(names) > 1, names


IN_PLACE = """
import os
os.environ["HIP_STUB_COPIES"] = "1"
def in_place(plan, in_bytes, out_bytes):
    d = eden.DeviceBuffer(nbytes=in_bytes + out_bytes)
    for shift in (in_bytes, 0, in_bytes - 4):   # behind the input, on it, on its last word
        print("run", file=open(os.environ["HIP_STUB_LOG"], "a"))
        plan.run(d, eden.BufferView(d, shift), q)
"""


@pytest.mark.parametrize("plan,in_bytes,out_bytes", [
    ("eden.ConvPlan(eden.conv_desc(2, 21, 33, 33, 21, 3, 3, (1, 1), (1,) * 4, layout=eden.NHWC), buf(21, 21, 3, 3), bias(21), q)", 2 * 21 * 33 * 33, 2 * 21 * 33 * 33),
    ("eden.ConvPlan(eden.conv_desc(2, 21, 33, 33, 21, 3, 3, (1, 1), (1,) * 4, layout=eden.NCHW), buf(21, 21, 3, 3), bias(21), q)", 2 * 21 * 33 * 33, 2 * 21 * 33 * 33),
    ("eden.ConvPlan(eden.conv_desc(1, 64, 20, 20, 30, 1, 1, layout=eden.NCHW), buf(30, 64, 1, 1), bias(30), q)", 64 * 400, 30 * 400),
    ("eden.DeconvPlan(eden.conv_desc(2, 23, 15, 15, 17, 3, 3, (1, 1), (1,) * 4, layout=eden.NHWC, weight_layout=eden.W_IOHW), buf(23, 17, 3, 3), bias(17), q)", 2 * 23 * 225, 2 * 17 * 225),
    ("eden.FcPlan(97, 113, 113, buf(113, 113), bias(113), q)", 97 * 113, 97 * 113),
    ("eden.DwConvPlan(eden.conv_desc(2, 33, 21, 21, 33, 3, 3, (1, 1), (1,) * 4, dm=1, layout=eden.NHWC), buf(33, 1, 3, 3), bias(33), q)", 2 * 33 * 441, 2 * 33 * 441),
    ("eden.DwConvPlan(eden.conv_desc(2, 22, 21, 21, 44, 3, 3, (1, 1), (1,) * 4, dm=2, layout=eden.NHWC), buf(44, 1, 3, 3), bias(44), q)", 2 * 22 * 441, 2 * 44 * 441),
    ("eden.DwConvPlan(eden.conv_desc(2, 24, 21, 21, 24, 3, 3, (1, 1), (1,) * 4, dm=1, layout=eden.NCHW), buf(24, 1, 3, 3), bias(24), q)", 2 * 24 * 441, 2 * 24 * 441),
    ("eden.DwConvPlan(eden.conv_desc(2, 24, 21, 21, 24, 7, 7, (2, 2), (3,) * 4, dm=1, layout=eden.NCHW), buf(24, 1, 7, 7), bias(24), q)", 2 * 24 * 441, 2 * 24 * 121),
], ids=["ragged", "planar", "planar_whole_channels", "transposed", "fc", "depthwise_ragged", "depthwise_multiplier",
        "depthwise_planar", "depthwise_planar_7x7_stride_2"])
def test_an_output_on_its_input_reads_a_copy(stub, tmp_path, plan, in_bytes, out_bytes):
    program = "bias = lambda n: buf(n, dtype=np.int32)\n" + IN_PLACE + "in_place(%s, %d, %d)\n" % (plan, in_bytes, out_bytes)
    names = [r[0] for r in launches(stub, tmp_path, program)]
    at = [i for i, v in enumerate(names) if v == "run"] + [len(names)]
    apart, on, last_word = [names[at[i] + 1:at[i + 1]] for i in range(3)]
    assert len(apart) == 1 and len(on) > 1 and on[0].split("kernel")[0] not in apart[0] and on == last_word, (apart, on, last_word)
