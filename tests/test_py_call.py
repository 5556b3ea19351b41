"""The binding's operator calls (host/py_call.cpp) beside their ctypes form: whatever the arguments, both answer alike.  Plans
over no images compute nothing, so all but the last test run without a GPU."""
import ctypes as C
import sys

import numpy as np
import pytest

import oracle_lib as O
from harness import eden, synth, to_eh_requant

eden.load()
Q = eden.Requant(3, 4, 5, 1 << 30, -4, 0, 255)
BAD_Q = eden.Requant(3, 4, 5, 1 << 30, -99, 0, 255)   # shift out of range
AQ = eden.make_add_requant(0.1, 3, 0.2, 4, 0.3, 5)


class Mem:
    def __init__(self, ptr):
        self.ptr = ptr


class MemWithoutPtr:
    pass


class MemThatRaises:
    @property
    def ptr(self):
        raise KeyError("gone")


class Address(C.c_void_p):
    pass


def empty_plan():
    return eden.ConvPlan(eden.conv_desc(0, 16, 4, 4, 16, 1, 1, layout=eden.NHWC), Mem(None), None, Q)


def outcome(call):
    try:
        return "returned", call()
    except Exception as e:
        return type(e), str(e).replace("run_general", "run").replace("_conv_dw_block_run_general", "conv_dw_block_run")


A = Mem(C.c_void_p(4096))
RUN = {
    "positional": ((A, A, Q), {}),
    "stream none": ((A, A, Q, None), {}),
    "stream integer": ((A, A, Q, 0), {}),
    "stream handle": ((A, A, Q, C.c_void_p()), {}),
    "stream keyword": ((A, A, Q), dict(stream=None)),
    "all keywords": ((), dict(d_in=A, d_out=A, q=Q)),
    "null pointers": ((Mem(None), Mem(None), Q), {}),
    "null handles": ((Mem(C.c_void_p()), Mem(C.c_void_p()), Q), {}),
    "integer addresses": ((Mem(4096), Mem(8192), Q), {}),
    "derived handle": ((Mem(Address(4096)), A, Q), {}),
    "byref": ((A, A, C.byref(Q)), {}),
    "pointer": ((A, A, C.pointer(Q)), {}),
    "refused parameters": ((A, A, BAD_Q), {}),
    "refused parameters, keyword": ((A, A), dict(q=BAD_Q)),
    "other parameters": ((A, A, AQ), {}),
    "no parameters": ((A, A, None), {}),
    "text for an address": ((Mem("x"), A, Q), {}),
    "address too long": ((Mem(1 << 80), A, Q), {}),
    "no ptr": ((MemWithoutPtr(), A, Q), {}),
    "ptr raises": ((A, MemThatRaises(), Q), {}),
    "text for a stream": ((A, A, Q, "x"), {}),
    "too few": ((A, A), {}),
    "none": ((), {}),
    "too many": ((A, A, Q, None, None), {}),
    "unknown keyword": ((A, A, Q), dict(streams=None)),
}
ANSWERED = ("positional", "stream none", "stream integer", "stream handle", "stream keyword", "all keywords", "null pointers", "null handles", "integer addresses",
            "derived handle", "byref", "pointer", "text for an address", "address too long", "text for a stream")   # (ctypes takes text, and cuts integers)


def test_the_native_form_is_in_place():
    assert type(eden.ConvPlan.run).__name__ == "method_descriptor" and type(eden.ConvPlan.run_add).__name__ == "method_descriptor"
    assert eden.conv_dw_block_run is not eden._conv_dw_block_run_general


@pytest.mark.parametrize("form", RUN)
def test_run_takes_and_refuses_what_the_ctypes_form_does(form):
    args, kwargs = RUN[form]
    plan = empty_plan()
    native, general = outcome(lambda: plan.run(*args, **kwargs)), outcome(lambda: plan._run_general(*args, **kwargs))
    assert native == general
    assert (native == ("returned", None)) == (form in ANSWERED), native


@pytest.mark.parametrize("form", RUN)
def test_run_add_takes_and_refuses_what_the_ctypes_form_does(form):
    args, kwargs = RUN[form]
    plan = empty_plan()
    if len(args) >= 3:   # run_add's own order: input, residual, output, requant, add parameters[, stream]
        if isinstance(args[2], (type(C.byref(Q)), C._Pointer)):
            pytest.skip("run_add takes the structures themselves")
        args = (args[0], A, args[1], args[2], AQ) + args[3:]
    elif "d_in" in kwargs:
        kwargs = dict(d_in=A, d_residual=A, d_out=A, q=Q, aq=AQ)
    assert outcome(lambda: plan.run_add(*args, **kwargs)) == outcome(lambda: plan._run_add_general(*args, **kwargs))


@pytest.mark.parametrize("extra", [{}, dict(stream=None), dict(rows_per_tile=2), dict(tiles=1)], ids=str)
@pytest.mark.parametrize("args", [(A, A, Q, Q), (A, A, Q, BAD_Q), (Mem(None), A, Q, Q), (MemWithoutPtr(), A, Q, Q), (A, MemThatRaises(), Q, Q), (A, A, AQ, Q), (A, A, Q),
                                  (A, A, Q, Q, 0, 0, None), (A, A, Q, Q, 0, 0, None, 1)], ids=range(9))
def test_block_run_takes_and_refuses_what_the_ctypes_form_does(args, extra):
    conv = empty_plan()
    dw = eden.DwConvPlan.__new__(eden.DwConvPlan)   # (a plan that was never made: its handle is null)
    eden._Plan.__init__(dw)
    native = outcome(lambda: eden.conv_dw_block_run(conv, dw, *args, **extra))
    assert native == outcome(lambda: eden._conv_dw_block_run_general(conv, dw, *args, **extra))
    # (every call that reaches the library is refused there)
    assert native[0] != "returned"


def test_calls_hold_no_references():
    plan = empty_plan()
    count = lambda: [sys.getrefcount(o) for o in (A, A.ptr, Q, AQ, BAD_Q, plan, plan.handle)]
    before = count()
    for _ in range(200):
        plan.run(A, A, Q)
        plan.run(A, A, Q, None)
        plan.run(A, A, Q, stream=None)
        plan.run_add(A, A, A, Q, AQ)
        outcome(lambda: plan.run(A, A, BAD_Q))
        outcome(lambda: plan.run(A, MemThatRaises(), Q))
    assert count() == before


@pytest.mark.gpu
def test_every_form_of_a_call_computes():
    s = O.conv_shape(1, 32, 9, 9, 48, 1, 1)
    x, w = synth.fill_u8((1, 9, 9, 32), 71), synth.fill_u8((48, 32, 1, 1), 72)
    b = synth.fill_i32((48,), 73, -1000, 1000)
    oq = O.make_quant(0.02, 121, 0.005, 133, 0.05, 128)
    q = to_eh_requant(oq)
    want = O.conv2d(np.ascontiguousarray(x.transpose(0, 3, 1, 2)), w, b, s, oq).transpose(0, 2, 3, 1)
    d_x, d_w, d_b, d_o = eden.DeviceBuffer(host=x), eden.DeviceBuffer(host=w), eden.DeviceBuffer(host=b), eden.DeviceBuffer(nbytes=want.size)
    plan = eden.ConvPlan(eden.conv_desc(1, 32, 9, 9, 48, 1, 1, layout=eden.NHWC), d_w, d_b, q)
    stream = eden.Stream()
    as_int = lambda d: Mem(d.ptr.value)
    for args, kwargs in (((d_x, d_o, q), {}), ((d_x, d_o, q, stream.h), {}), ((d_x, d_o, q, stream.h.value), {}), ((d_x, d_o, q), dict(stream=stream.h)),
                         ((as_int(d_x), as_int(d_o), q), {}), ((), dict(d_in=d_x, d_out=d_o, q=q)), ((eden.BufferView(d_x, 0), d_o, C.byref(q)), {})):
        eden.check(eden.load().eh_memset(d_o.ptr, 0, want.size, None))
        eden.sync()
        plan.run(*args, **kwargs)
        stream.sync()
        assert np.array_equal(d_o.download(want.shape), want)
    with pytest.raises(eden.EdenHipError, match="null"):
        plan.run(Mem(None), d_o, q)
    with pytest.raises(eden.EdenHipError, match="null"):
        plan.run(d_x, Mem(0), q, stream.h)
