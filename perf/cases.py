"""The work a user of this library has it do, as measurable cases.

`listed()` names representative cases, `draw(rng)` gives further ones of the same ranges, `prepare(case, seed)` makes
what a program holds before the call (device tensors, the operator's plan, an opened network), `run(state)` is one
pass through the public entry points and returns its outputs, `work(case)` states the bytes and operations a pass
cannot do without, `tolerance(case)` how far a correct result may be off: not at all, every output is whole bytes.

Kinds of case:
  fc          fully connected layer, [m, k] x [n, k] -> [m, n]
  conv        k x k convolution (first layers, 1x1, strided, atrous, grouped; channels-last or planar tensors)
  dw          depthwise convolution
  deconv      transposed convolution
  bottleneck  1x1 expansion, 3x3 depthwise, 1x1 projection, with the residual add where stride and channels allow it
  network     MobileNetV2 as one program: "device" replays the recorded operator plans on tensors that stay on the
              GPU, "host" opens an operator list with the userdriver and executes it on host buffers
`quant` says what the bytes are: "u8" = uint8 tensors and weights with one scale per tensor, "u8pc" = uint8 tensors
with int8 weights and one scale per output channel, "s8pc" = int8 tensors with such weights."""
import ctypes
import importlib
import math
import random

import numpy as np
import torch

eden = importlib.import_module("cl-eden-kernel_amd")
mobilenet = importlib.import_module("cl-eden-kernel_amd.mobilenet")
userdriver = importlib.import_module("cl-eden-kernel_amd.userdriver")

LIST_ID = 0xC5
MAX_MACS = 2e10      # of a drawn operator other than fc: well under the largest listed case
MAX_BYTES = 150e6


def fc(m, k, n, quant="u8"):
    return dict(kind="fc", m=m, k=k, n=n, quant=quant)


def conv(n, c, h, w, cout, k, stride=1, dil=1, groups=1, quant="u8", layout="nhwc", relu6=True):
    return dict(kind="conv", n=n, c=c, h=h, w=w, cout=cout, k=k, stride=stride, dil=dil, groups=groups, quant=quant, layout=layout, relu6=relu6)


def dw(n, c, h, w, k, stride=1, dil=1, dm=1, quant="u8", layout="nhwc"):
    return dict(kind="dw", n=n, c=c, h=h, w=w, k=k, stride=stride, dil=dil, dm=dm, quant=quant, layout=layout)


def deconv(n, c, h, w, cout, k, stride, quant="u8", layout="nhwc"):
    return dict(kind="deconv", n=n, c=c, h=h, w=w, cout=cout, k=k, stride=stride, quant=quant, layout=layout)


def bottleneck(n, cin, expanded, cout, h, w, stride, quant="u8"):
    return dict(kind="bottleneck", n=n, cin=cin, expanded=expanded, cout=cout, h=h, w=w, stride=stride, quant=quant)


def network(batch, image, data, per_channel=False, planar=False):
    return dict(kind="network", batch=batch, image=image, data=data, per_channel=per_channel, planar=planar)


def listed():
    return [
        # one row through a wide layer: a matrix-vector product, bound by latency and the weights' trip from memory
        dict(fc(1, 4096, 4096), name="fc_1x4096x4096"),
        # an ordinary batch through a wide layer
        dict(fc(256, 4096, 4096), name="fc_256x4096x4096"),
        # the largest operator: the same layer over 8192 rows (a dense layer at every pixel or token)
        dict(fc(8192, 4096, 4096), name="fc_8192x4096x4096"),
        # one image, one 3x3 layer of a residual stage: what a latency-bound program calls layer by layer
        dict(conv(1, 256, 14, 14, 256, 3), name="conv3x3_n1_256to256_14"),
        # a residual stage's 3x3 layer at a serving batch, int8 tensors, one scale per output channel
        dict(conv(32, 128, 28, 28, 128, 3, quant="s8pc"), name="conv3x3_s8pc_n32_128to128_28"),
        # a 21-class segmentation head on planar tensors of ragged extent: channels off every tile size
        dict(conv(3, 21, 65, 47, 21, 3, layout="nchw", relu6=False), name="conv3x3_nchw_n3_21to21_65x47"),
        # a wide-window depthwise layer at a training-sized batch
        dict(dw(64, 144, 56, 56, 5), name="dw5x5_n64_c144_56"),
        # upsampling in a decoder
        dict(deconv(8, 256, 32, 32, 128, 4, 2), name="deconv4x4s2_n8_256to128_32"),
        # the mobile block: 24 -> 144 expansion, 3x3 depthwise at stride 2, projection
        dict(bottleneck(32, 24, 144, 32, 56, 56, 2), name="bottleneck_n32_24x144to32_56s2"),
        # a whole network on one image handed over in host memory: latency of a request
        dict(network(1, 224, "host"), name="network_host_b1"),
        # ... on a planar batch in host memory, one scale per output channel: an offline or batched service
        dict(network(32, 224, "host", per_channel=True, planar=True), name="network_host_planar_pc_b32"),
        # ... on a batch that is on the GPU already: throughput
        dict(network(64, 224, "device"), name="network_device_b64"),
    ]


def log_between(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def channels(rng, lo, hi):
    """mostly whole multiples of eight, as networks have them; the rest anything"""
    c = log_between(rng, lo, hi)
    return max(8, (c + 4) // 8 * 8) if rng.random() < 0.75 else c


def draw(rng):
    while True:
        kind = rng.choice(["fc", "fc", "conv", "conv", "conv", "dw", "deconv", "bottleneck", "bottleneck", "network"])
        quant = rng.choice(["u8", "u8", "u8pc", "s8pc"])
        layout = "nhwc" if rng.random() < 0.75 else "nchw"
        n = log_between(rng, 1, 64)
        h = log_between(rng, 7, 112)
        w = h if rng.random() < 0.7 else max(7, min(112, h + rng.randint(-9, 9)))
        if kind == "fc":
            case = fc(log_between(rng, 1, 8192), log_between(rng, 64, 4096), log_between(rng, 10, 4096), rng.choice(["u8", "s8"]))
            if rng.random() < 0.6:   # layer widths are mostly round; the number of rows is what it is
                case["k"], case["n"] = max(64, case["k"] // 64 * 64), max(16, case["n"] // 16 * 16)
        elif kind == "conv":
            k, stride = rng.choice([1, 1, 3, 3, 3, 5, 7]), rng.choice([1, 1, 1, 2])
            dil = 2 if k == 3 and stride == 1 and rng.random() < 0.2 else 1
            c, cout = channels(rng, 8, 512), channels(rng, 8, 512)
            if rng.random() < 0.15:   # a first layer
                c, k, stride, dil, h = 3, rng.choice([3, 5, 7]), 2, 1, log_between(rng, 64, 224)
                w = h
            groups = rng.choice([2, 4, 8, 32])
            if c % groups or cout % groups or rng.random() < 0.85:
                groups = 1
            case = conv(n, c, h, w, cout, k, stride, dil, groups, quant, layout, rng.random() < 0.6)
        elif kind == "dw":
            k, stride = rng.choice([3, 3, 3, 5, 7]), rng.choice([1, 1, 2])
            case = dw(n, channels(rng, 16, 960), h, w, k, stride, 2 if k == 3 and stride == 1 and rng.random() < 0.2 else 1,
                      2 if rng.random() < 0.1 else 1, quant, layout)
        elif kind == "deconv":
            k, stride = rng.choice([(2, 2), (3, 2), (4, 2), (4, 2), (4, 4), (8, 4), (16, 8)])
            h, w = min(h, 64), min(w, 64)
            case = deconv(min(n, 16), channels(rng, 16, 256), h, w, channels(rng, 8, 128), k, stride, quant, layout)
        elif kind == "bottleneck":
            cin = max(8, log_between(rng, 16, 160) // 8 * 8)
            stride = rng.choice([1, 1, 2])
            case = bottleneck(n, cin, 6 * cin, cin if stride == 1 and rng.random() < 0.7 else max(8, log_between(rng, 16, 320) // 8 * 8),
                              h, w, stride, rng.choice(["u8", "u8pc"]))
        else:
            data = rng.choice(["host", "device"])
            # (a host batch crosses the bus as well: at most the listed one)
            case = network(log_between(rng, 1, 32 if data == "host" else 64), rng.choice([96, 128, 160, 192, 224]), data, rng.random() < 0.4,
                           data == "host" and rng.random() < 0.4)
        size = work(case)
        if kind in ("fc", "network") or (size["flops"] <= 2 * MAX_MACS and size["bytes"] <= MAX_BYTES):
            return case


# ---- sizes ----------------------------------------------------------------------

def out_extent(case, extent):
    if case["kind"] == "deconv":
        return (extent - 1) * case["stride"] + case["k"] - 2 * padding(case)
    return (extent + 2 * padding(case) - case.get("dil", 1) * (case["k"] - 1) - 1) // case["stride"] + 1


def padding(case):
    if case["kind"] == "deconv":
        return (case["k"] - case["stride"]) // 2
    return case.get("dil", 1) * (case["k"] - 1) // 2


def work(case):
    kind = case["kind"]
    if kind == "fc":
        m, k, n = case["m"], case["k"], case["n"]
        return dict(bytes=m * k + n * k + 4 * n + m * n, flops=2 * m * k * n)
    if kind == "network":
        tensors, ops = mobilenet.layers(case["image"])
        weights = 0
        for op in ops:
            if op["op"] in ("conv", "dw", "fc"):
                fan = 1 if op["op"] == "dw" else tensors[op["src"]]["c"]
                weights += op["cout"] * (fan * op.get("k", 1) ** 2 + 4)
        return dict(bytes=case["batch"] * (3 * case["image"] ** 2 + 1000) + weights, flops=2 * case["batch"] * mobilenet.macs_per_image(case["image"]))
    n, h, w = case["n"], case["h"], case["w"]
    if kind == "bottleneck":
        cin, mid, cout = case["cin"], case["expanded"], case["cout"]
        ho, wo = -(-h // case["stride"]), -(-w // case["stride"])
        weights = mid * cin + mid * 9 + cout * mid + 4 * (2 * mid + cout)
        return dict(bytes=n * h * w * cin + n * ho * wo * cout + weights, flops=2 * n * (h * w * cin * mid + ho * wo * mid * (9 + cout)))
    ho, wo, k2 = out_extent(case, h), out_extent(case, w), case["k"] ** 2
    if kind == "dw":
        c = case["c"] * case["dm"]
        return dict(bytes=n * h * w * case["c"] + n * ho * wo * c + c * (k2 + 4), flops=2 * n * ho * wo * c * k2)
    if kind == "deconv":
        return dict(bytes=n * (h * w * case["c"] + ho * wo * case["cout"]) + case["c"] * case["cout"] * k2 + 4 * case["cout"],
                    flops=2 * n * h * w * case["c"] * case["cout"] * k2)
    per_group = case["c"] // case["groups"]
    return dict(bytes=n * (h * w * case["c"] + ho * wo * case["cout"]) + case["cout"] * (per_group * k2 + 4), flops=2 * n * ho * wo * case["cout"] * per_group * k2)


def tolerance(case):
    return "exact"   # quantized bytes, integer arithmetic throughout


# ---- inputs, weights, quantization parameters -----------------------------------

class Mem:
    """A torch tensor's device memory as the plans take it (anything with a `ptr`)."""

    def __init__(self, tensor):
        self.tensor, self.ptr = tensor, ctypes.c_void_p(tensor.data_ptr())


class Alias:
    """Device memory that `owner` holds, for torch.as_tensor (the tensor keeps this object, and so the owner)."""

    def __init__(self, owner, pointer, shape):
        self.owner = owner
        self.__cuda_array_interface__ = dict(data=(pointer.value, False), shape=tuple(shape), typestr="|u1", version=2)


class Maker:
    def __init__(self, seed):
        self.rng = random.Random(seed)
        self.gen = torch.Generator(device="cuda")
        self.gen.manual_seed(seed)

    def bytes(self, shape, signed=False):
        """uniform over all byte values, as images and most feature maps around their zero point"""
        x = torch.randint(0, 256, shape, generator=self.gen, device="cuda", dtype=torch.uint8)
        return x.view(torch.int8) if signed else x

    def rectified(self, shape, signed=False):
        """a ReLU6 layer's output: half the values at the zero point, the rest up to the clamp"""
        x = torch.randn(shape, generator=self.gen, device="cuda").mul_(64).round_().clamp_(0, 255).to(torch.uint8)
        return x.bitwise_xor_(128).view(torch.int8) if signed else x

    def bias(self, count, reach=1000):
        return torch.randint(-reach, reach + 1, (count,), generator=self.gen, device="cuda", dtype=torch.int32)

    def weights(self, shape, quant):
        """(tensor, zero point, standard deviation around it): a normal field, over the whole byte range"""
        g = torch.randn(shape, generator=self.gen, device="cuda")
        if quant == "u8":
            zp = self.rng.randint(110, 140)
            return (g.mul_(40).round_().add_(zp).clamp_(0, 255)).to(torch.uint8), zp, 40.0
        return g.mul_(36).round_().clamp_(-127, 127).to(torch.int8), 0, 36.0


def requant(make, quant, cout, fan_in, in_zp, in_rms, w_zp, w_sd, relu6):
    """(Requant, (multipliers, shifts) or None) that spread a layer's outputs over the byte range: ReLU6 outputs have
    zero point 0 and scale 6 / 255, linear ones zero point 128 and about 35 steps of standard deviation."""
    acc_sd = math.sqrt(fan_in) * in_rms * w_sd
    signed = quant in ("s8", "s8pc")
    s_out, zp_out, out_sd = (6.0 / 255, 0, 64.0) if relu6 else (0.05, 128, 35.0)
    act = eden.ACT_RELU6 if relu6 else eden.ACT_NONE
    s_in = 0.02
    s_w = out_sd * s_out / (acc_sd * s_in)
    if signed:
        zp_out -= 128
    if not quant.endswith("pc"):
        return (eden.make_requant_s8 if signed else eden.make_requant)(s_in, in_zp, s_w, w_zp, s_out, zp_out, act, relu6), None
    scales = np.array([s_w * make.rng.uniform(0.6, 1.6) for _ in range(cout)], np.float32)
    q, mults, shifts = eden.make_requant_perchannel(s_in, in_zp, scales, s_out, zp_out, act, relu6)
    if signed:
        q.act_min, q.act_max = -128, 127   # (either clamp spans the bytes)
    return q, (mults, shifts)


def flags(quant):
    """(tensor flags, weight flags)"""
    return (eden.IO_SIGNED if quant in ("s8", "s8pc") else 0), (0 if quant == "u8" else eden.W_SIGNED)


# ---- prepare ----------------------------------------------------------------------

def prepare(case, seed):
    eden.init(0)
    return dict(fc=prepare_fc, conv=prepare_windowed, dw=prepare_windowed, deconv=prepare_windowed, bottleneck=prepare_bottleneck,
                network=prepare_network)[case["kind"]](case, seed)


def prepare_fc(case, seed):
    make = Maker(seed)
    m, k, n, quant = case["m"], case["k"], case["n"], case["quant"]
    io, wf = flags(quant)
    zp = make.rng.randint(0, 20) - (128 if io else 0)
    x = make.bytes((m, k), bool(io))
    w, w_zp, w_sd = make.weights((n, k), quant)
    q, _ = requant(make, quant, n, k, zp, 140.0, w_zp, w_sd, False)
    out = torch.zeros((m, n), dtype=x.dtype, device="cuda")
    plan = eden.FcPlan(m, k, n, Mem(w), Mem(make.bias(n)), q, flags=io | wf)
    return dict(kind="plan", plan=plan, x=Mem(x), out=Mem(out), q=q)


def prepare_windowed(case, seed):
    make = Maker(seed)
    kind, n, c, h, w, k, quant, layout = (case[f] for f in ("kind", "n", "c", "h", "w", "k", "quant", "layout"))
    io, wf = flags(quant)
    pad, ho, wo = padding(case), out_extent(case, h), out_extent(case, w)
    groups, dm = case.get("groups", 1), case.get("dm", 1)
    cout = c * dm if kind == "dw" else case["cout"]
    shape = (lambda ch, y, x: (n, y, x, ch)) if layout == "nhwc" else (lambda ch, y, x: (n, ch, y, x))
    rectified = kind == "dw"   # a depthwise layer follows an expansion with ReLU6
    zp = (0 if rectified else make.rng.randint(100, 150)) - (128 if io else 0)
    x = (make.rectified if rectified else make.bytes)(shape(c, h, w), bool(io))
    if kind == "deconv":
        w_shape, w_layout, fan_in = (c, cout, k, k), eden.W_IOHW, c * max(1, k // case["stride"]) ** 2
    elif kind == "dw":
        w_shape, w_layout, fan_in = (cout, 1, k, k), eden.W_OIHW, k * k
    else:
        w_shape, w_layout, fan_in = (cout, c // groups, k, k), eden.W_OIHW, c // groups * k * k
    wt, w_zp, w_sd = make.weights(w_shape, quant)
    q, pairs = requant(make, quant, cout, fan_in, zp, 45.0 if rectified else 75.0, w_zp, w_sd, kind == "dw" or case.get("relu6", False))
    desc = eden.conv_desc(n, c, h, w, cout, k, k, (case["stride"],) * 2, (pad,) * 4, (case.get("dil", 1),) * 2, groups, dm,
                          (eden.NHWC if layout == "nhwc" else eden.NCHW) | io, w_layout | wf)
    plan = dict(conv=eden.ConvPlan, dw=eden.DwConvPlan, deconv=eden.DeconvPlan)[kind](desc, Mem(wt), Mem(make.bias(cout)), q)
    if pairs:
        plan.set_perchannel(*pairs)
    out = torch.zeros(shape(cout, ho, wo), dtype=x.dtype, device="cuda")
    eden.sync()
    return dict(kind="plan", plan=plan, x=Mem(x), out=Mem(out), q=q)


def prepare_bottleneck(case, seed):
    make = Maker(seed)
    n, cin, mid, cout, h, w, stride, quant = (case[f] for f in ("n", "cin", "expanded", "cout", "h", "w", "stride", "quant"))
    ho, wo = -(-h // stride), -(-w // stride)
    _, wf = flags(quant)
    x = make.bytes((n, h, w, cin))

    def layer(plan_type, c, y, z, co, k, s, in_zp, in_rms, relu6):
        depthwise = plan_type is eden.DwConvPlan
        wt, w_zp, w_sd = make.weights((co, 1 if depthwise else c, k, k), quant)
        q, pairs = requant(make, quant, co, k * k * (1 if depthwise else c), in_zp, in_rms, w_zp, w_sd, relu6)
        desc = eden.conv_desc(n, c, y, z, co, k, k, (s, s), ((k - 1) // 2,) * 4, layout=eden.NHWC, weight_layout=eden.W_OIHW | wf)
        plan = plan_type(desc, Mem(wt), Mem(make.bias(co)), q)
        if pairs:
            plan.set_perchannel(*pairs)
        return plan, q

    expand, q_expand = layer(eden.ConvPlan, cin, h, w, mid, 1, 1, 128, 75.0, True)
    depth, q_depth = layer(eden.DwConvPlan, mid, h, w, mid, 3, stride, 0, 45.0, True)
    project, q_project = layer(eden.ConvPlan, mid, ho, wo, cout, 1, 1, 0, 45.0, False)
    one_launch = eden.conv_dw_block_preferred(expand, depth)
    state = dict(kind="bottleneck", expand=expand, depth=depth, project=project, q_expand=q_expand, q_depth=q_depth, q_project=q_project, one_launch=one_launch,
                 x=Mem(x), filtered=Mem(torch.zeros((n, ho, wo, mid), dtype=torch.uint8, device="cuda")), out=Mem(torch.zeros((n, ho, wo, cout), dtype=torch.uint8, device="cuda")))
    if not one_launch:
        state["expanded"] = Mem(torch.zeros((n, h, w, mid), dtype=torch.uint8, device="cuda"))
    if stride == 1 and cin == cout:
        state["q_add"] = eden.make_add_requant(0.05, 128, 0.05, 128, 0.07, 128)
    eden.sync()
    return state


def prepare_network(case, seed):
    batch, image = case["batch"], case["image"]
    x = np.random.default_rng(seed).integers(0, 256, (batch, image, image, 3), dtype=np.uint8)
    if case["data"] == "host":
        driver = userdriver.UserDriver(0)
        net, first, last, shape = mobilenet.operator_list(userdriver, LIST_ID, batch, image, per_channel=case["per_channel"], nchw=case["planar"])
        driver.open_subgraph(net)
        if case["planar"]:
            x = np.ascontiguousarray(x.transpose(0, 3, 1, 2))
        logits = np.zeros(shape, np.uint8)
        return dict(kind="host", driver=driver, buffers={first: x, last: logits}, logits=logits)
    # two chains of images side by side from 24 images on, expansions fused with their depthwise layers where preferred
    lanes = 2 if batch >= 24 and batch % 2 == 0 else 1
    net = mobilenet.MobileNetV2(eden, batch, image, fuse_add=True, per_channel=case["per_channel"], pooled=True, lanes=lanes, fuse_blocks="auto")
    net.set_input(x)
    stream = eden.Stream()
    graph = eden.Graph(stream, net.run)
    logits = torch.as_tensor(Alias(net, net.buffers[-1].ptr, (batch, 1000)), device="cuda")
    return dict(kind="device", net=net, stream=stream, graph=graph, logits=logits)


# ---- run ------------------------------------------------------------------------------

def run(state):
    kind = state["kind"]
    if kind == "plan":
        state["plan"].run(state["x"], state["out"], state["q"])
        return state["out"].tensor
    if kind == "bottleneck":
        x, filtered, out = state["x"], state["filtered"], state["out"]
        if state["one_launch"]:
            eden.conv_dw_block_run(state["expand"], state["depth"], x, filtered, state["q_expand"], state["q_depth"])
        else:
            state["expand"].run(x, state["expanded"], state["q_expand"])
            state["depth"].run(state["expanded"], filtered, state["q_depth"])
        if "q_add" in state:
            state["project"].run_add(filtered, x, out, state["q_project"], state["q_add"])
        else:
            state["project"].run(filtered, out, state["q_project"])
        return out.tensor
    if kind == "host":
        state["driver"].execute_subgraph(LIST_ID, state["buffers"])
        return state["logits"]
    state["graph"].launch(state["stream"])
    return state["logits"]
