// The Python binding's operator calls as native methods: `plan.run`, `plan.run_add` and `conv_dw_block_run` go straight
// from the interpreter's argument vector to the C ABI (include/eden_hip.h).
//
// On a small layer the call itself is the time: the GPU takes the launches as fast as the host can write them, and every
// nanosecond of the host's adds to the pass.  A Python method that goes through ctypes costs 1.0 us per call (a frame,
// an argument object per pointer), this path 0.2 us.  It serves the usual argument types (objects with a `ptr` that is
// a c_void_p, an int or None, the binding's parameter structures, a stream handle, all by position); everything else,
// keywords included, goes to the ctypes form of the same call, which also raises what the arguments deserve.
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <cstdint>
#include <initializer_list>

#include "eden_hip.h"

namespace {

PyObject *pointer_type, *requant_type, *add_type;   // ctypes.c_void_p and the binding's structures
PyObject *check_status;                             // raises the library's error for a status
PyObject *block_general;                            // the ctypes form of conv_dw_block_run
PyObject *name_ptr, *name_handle, *name_entry, *name_run, *name_run_add;

// The bytes of a ctypes object, held for the call.
struct View {
    Py_buffer buffer;
    bool held = false;
    View() {}
    View(const View &) = delete;
    View &operator=(const View &) = delete;
    ~View() {
        if (held) PyBuffer_Release(&buffer);
    }
    void *of(PyObject *object, Py_ssize_t bytes) {
        if (PyObject_GetBuffer(object, &buffer, PyBUF_SIMPLE) != 0) return nullptr;
        held = true;
        return buffer.len == bytes ? buffer.buf : nullptr;
    }
};

// None, an integer or a c_void_p -> the address; false: some other form (an error may be set)
bool address_of(PyObject *object, void **out) {
    if (object == Py_None) {
        *out = nullptr;
        return true;
    }
    if (PyLong_CheckExact(object)) {
        *out = PyLong_AsVoidPtr(object);
        return !(*out == nullptr && PyErr_Occurred());
    }
    if ((PyObject *)Py_TYPE(object) != pointer_type) return false;
    View view;
    const void *bytes = view.of(object, sizeof(void *));
    if (!bytes) return false;
    *out = *(void *const *)bytes;
    return true;
}

bool member_address(PyObject *owner, PyObject *name, void **out) {
    PyObject *value = PyObject_GetAttr(owner, name);
    if (!value) return false;
    const bool ok = address_of(value, out);
    Py_DECREF(value);
    return ok;
}

template <class T>
const T *parameters(View &view, PyObject *object, PyObject *type) {
    return (PyObject *)Py_TYPE(object) == type ? (const T *)view.of(object, sizeof(T)) : nullptr;
}

PyObject *finish(int status) {
    if (status == EH_OK) Py_RETURN_NONE;
    return PyObject_CallFunction(check_status, "i", status);   // raises
}

PyObject *general(PyObject *self, PyObject *name, PyObject *const *args, Py_ssize_t nargs, PyObject *kwnames) {
    PyErr_Clear();
    PyObject *method = PyObject_GetAttr(self, name);
    if (!method) return nullptr;
    PyObject *result = PyObject_Vectorcall(method, args, (size_t)nargs, kwnames);
    Py_DECREF(method);
    return result;
}

using RunFn = int (*)(void *plan, const void *in, void *out, const eh_requant *q, void *stream);

PyObject *plan_run(PyObject *self, PyObject *const *args, Py_ssize_t nargs, PyObject *kwnames) {
    void *entry, *plan, *in, *out, *stream = nullptr;
    View view;
    const eh_requant *q;
    if (kwnames || nargs < 3 || nargs > 4 || !member_address(self, name_entry, &entry) || !entry || !member_address(self, name_handle, &plan) ||
        !member_address(args[0], name_ptr, &in) || !member_address(args[1], name_ptr, &out) || !(q = parameters<eh_requant>(view, args[2], requant_type)) ||
        (nargs == 4 && !address_of(args[3], &stream)))
        return general(self, name_run, args, nargs, kwnames);
    int status;
    Py_BEGIN_ALLOW_THREADS
    status = ((RunFn)entry)(plan, in, out, q, stream);
    Py_END_ALLOW_THREADS
    return finish(status);
}

PyObject *plan_run_add(PyObject *self, PyObject *const *args, Py_ssize_t nargs, PyObject *kwnames) {
    void *plan, *in, *residual, *out, *stream = nullptr;
    View view, add_view;
    const eh_requant *q;
    const eh_add_requant *aq;
    if (kwnames || nargs < 5 || nargs > 6 || !member_address(self, name_handle, &plan) || !member_address(args[0], name_ptr, &in) ||
        !member_address(args[1], name_ptr, &residual) || !member_address(args[2], name_ptr, &out) || !(q = parameters<eh_requant>(view, args[3], requant_type)) ||
        !(aq = parameters<eh_add_requant>(add_view, args[4], add_type)) || (nargs == 6 && !address_of(args[5], &stream)))
        return general(self, name_run_add, args, nargs, kwnames);
    int status;
    Py_BEGIN_ALLOW_THREADS
    status = eh_conv2d_u8_run_add((eh_conv_plan *)plan, in, residual, out, q, aq, stream);
    Py_END_ALLOW_THREADS
    return finish(status);
}

PyObject *block_run(PyObject *, PyObject *const *args, Py_ssize_t nargs, PyObject *kwnames) {
    void *pointwise, *depthwise, *in, *out;
    View view_p, view_d;
    const eh_requant *qp, *qd;
    // (explicit tile sizes and a stream are for the general form)
    if (kwnames || nargs != 6 || !member_address(args[0], name_handle, &pointwise) || !member_address(args[1], name_handle, &depthwise) ||
        !member_address(args[2], name_ptr, &in) || !member_address(args[3], name_ptr, &out) || !(qp = parameters<eh_requant>(view_p, args[4], requant_type)) ||
        !(qd = parameters<eh_requant>(view_d, args[5], requant_type))) {
        PyErr_Clear();
        return PyObject_Vectorcall(block_general, args, (size_t)nargs, kwnames);
    }
    int status;
    Py_BEGIN_ALLOW_THREADS
    status = eh_conv_dw_block_run((eh_conv_plan *)pointwise, (eh_dwconv_plan *)depthwise, in, out, qp, qd, 0, 0, nullptr);
    Py_END_ALLOW_THREADS
    return finish(status);
}

PyMethodDef run_method = {"run", (PyCFunction)(void (*)(void))plan_run, METH_FASTCALL | METH_KEYWORDS, "run($self, d_in, d_out, q, stream=None)\n--\n\nd_out = operator(d_in)"};
PyMethodDef run_add_method = {"run_add", (PyCFunction)(void (*)(void))plan_run_add, METH_FASTCALL | METH_KEYWORDS,
                              "run_add($self, d_in, d_residual, d_out, q, aq, stream=None)\n--\n\n"
                              "d_out = add(d_residual, convolution(d_in)) with the add parameters `aq` (the residual is the first operand)"};

// install(c_void_p, Requant, AddRequant, check, plan class, convolution plan class, conv_dw_block_run's general form):
// puts `run` and `run_add` on the classes
PyObject *install(PyObject *, PyObject *args) {
    PyObject *plan_class, *conv_class;
    if (!PyArg_ParseTuple(args, "OOOOO!O!O", &pointer_type, &requant_type, &add_type, &check_status, &PyType_Type, &plan_class, &PyType_Type, &conv_class, &block_general))
        return nullptr;
    for (PyObject *kept : {pointer_type, requant_type, add_type, check_status, block_general}) Py_INCREF(kept);
    PyObject *run = PyDescr_NewMethod((PyTypeObject *)plan_class, &run_method), *run_add = PyDescr_NewMethod((PyTypeObject *)conv_class, &run_add_method);
    const bool ok = run && run_add && PyObject_SetAttrString(plan_class, "run", run) == 0 && PyObject_SetAttrString(conv_class, "run_add", run_add) == 0;
    Py_XDECREF(run);
    Py_XDECREF(run_add);
    if (!ok) return nullptr;
    Py_RETURN_NONE;
}

PyMethodDef functions[] = {
    {"install", install, METH_VARARGS, nullptr},
    {"conv_dw_block_run", (PyCFunction)(void (*)(void))block_run, METH_FASTCALL | METH_KEYWORDS,
     "conv_dw_block_run(pointwise, depthwise, d_in, d_out, q_pointwise, q_depthwise, rows_per_tile=0, cols_per_tile=0, stream=None)\n--\n\n"
     "pointwise convolution + 3x3 depthwise convolution as one launch (the expanded tensor stays in LDS)"},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_call", nullptr, -1, functions, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__call(void) {
    name_ptr = PyUnicode_InternFromString("ptr");
    name_handle = PyUnicode_InternFromString("handle");
    name_entry = PyUnicode_InternFromString("_entry");
    name_run = PyUnicode_InternFromString("_run_general");
    name_run_add = PyUnicode_InternFromString("_run_add_general");
    if (!name_ptr || !name_handle || !name_entry || !name_run || !name_run_add) return nullptr;
    return PyModule_Create(&module);
}
