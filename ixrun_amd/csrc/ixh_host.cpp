// ixrun_amd._host: the host side of the calls whose kernels are shorter than Python's bookkeeping around them.
//
// A forward of one token spends 5 us on the GPU; checked, allocated and launched from Python through ctypes it took the
// host 8.  The same steps here: see the figures at each function.  Everything that is not the common case (other types,
// other devices, views, a scratch that has to grow, errors) is left to the caller: a function returns None and has done
// nothing, and the Python code behind it goes on.
#include <Python.h>
#include <structmember.h>

#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/ixhip.h"

namespace {

using LanesGemv = decltype(&ixh_lanes_gemv);
constexpr int kMaxRows = 16;

// The fused forward of one layer over its lane layout: an object called with the activations.
struct Forward {
    PyObject_HEAD
    vectorcallfunc call;
    LanesGemv gemv;
    const IxhLanes *lanes;
    const uint16_t *bias;
    int64_t in_f, out_f;
    long device;
    size_t workspace_bytes[kMaxRows + 1];
    PyObject *owner;       // keeps `lanes` and what it points at alive
    PyObject *workspaces;  // dict: device -> scratch tensor
    PyObject *device_key;
    PyObject *check;       // raises for a negative code
};

// A token of a layer of 2.4 M weights: 5 us of host time a call (8 us from Python).
PyObject *forward_call(PyObject *self_, PyObject *const *args, size_t nargsf, PyObject *kwnames) {
    HANDLE_TH_ERRORS
    Forward *self = reinterpret_cast<Forward *>(self_);
    if (PyVectorcall_NARGS(nargsf) != 1 || (kwnames && PyTuple_GET_SIZE(kwnames) != 0) || !THPVariable_CheckExact(args[0]))
        Py_RETURN_NONE;
    const at::Tensor &x = THPVariable_Unpack(args[0]);
    if (!x.is_cuda() || x.scalar_type() != at::kBFloat16 || x.dim() < 1 || x.size(-1) != self->in_f || x.get_device() != self->device ||
        !x.is_contiguous())
        Py_RETURN_NONE;
    const int64_t rows = x.numel() / self->in_f;
    if (rows < 1 || rows > kMaxRows) Py_RETURN_NONE;
    const size_t need = self->workspace_bytes[rows];
    void *scratch = nullptr;
    if (need) {
        PyObject *ws = PyDict_GetItemWithError(self->workspaces, self->device_key);
        if (!ws) {
            if (PyErr_Occurred()) return nullptr;
            Py_RETURN_NONE;
        }
        if (!THPVariable_Check(ws)) Py_RETURN_NONE;
        const at::Tensor &t = THPVariable_Unpack(ws);
        if (t.nbytes() < need) Py_RETURN_NONE;
        scratch = t.data_ptr();
    }
    c10::SmallVector<int64_t, 4> shape(x.sizes().begin(), x.sizes().end());
    shape.back() = self->out_f;
    at::Tensor y;
    int rc;
    {
        pybind11::gil_scoped_release without_gil;
        y = at::empty(shape, x.options());
        rc = self->gemv(self->lanes, static_cast<const uint16_t *>(x.const_data_ptr()), self->in_f, self->bias, (int32_t)rows,
                        static_cast<uint16_t *>(y.data_ptr()), self->out_f, scratch, need,
                        c10::hip::getCurrentHIPStream((c10::DeviceIndex)self->device).stream());
    }
    if (rc) {
        PyObject *r = PyObject_CallFunction(self->check, "i", rc);
        Py_XDECREF(r);
        if (!r) return nullptr;
    }
    return THPVariable_Wrap(std::move(y));
    END_HANDLE_TH_ERRORS
}

// Forward(gemv, lanes, bias, in_f, out_f, device, workspace_bytes, owner, workspaces, device_key, check); addresses as ints
int forward_init(PyObject *self_, PyObject *args, PyObject *) {
    Forward *self = reinterpret_cast<Forward *>(self_);
    unsigned long long gemv, lanes, bias;
    long long in_f, out_f;
    long device;
    PyObject *bytes, *owner, *workspaces, *key, *check;
    if (!PyArg_ParseTuple(args, "KKKLLlO!OO!OO", &gemv, &lanes, &bias, &in_f, &out_f, &device, &PyTuple_Type, &bytes, &owner,
                          &PyDict_Type, &workspaces, &key, &check))
        return -1;
    if (!gemv || !lanes || in_f < 1 || out_f < 1 || PyTuple_GET_SIZE(bytes) != kMaxRows + 1) {
        PyErr_SetString(PyExc_ValueError, "Forward: malformed arguments");
        return -1;
    }
    for (int i = 0; i <= kMaxRows; ++i) {
        self->workspace_bytes[i] = PyLong_AsSize_t(PyTuple_GET_ITEM(bytes, i));
        if (PyErr_Occurred()) return -1;
    }
    self->call = forward_call;
    self->gemv = reinterpret_cast<LanesGemv>(gemv);
    self->lanes = reinterpret_cast<const IxhLanes *>(lanes);
    self->bias = reinterpret_cast<const uint16_t *>(bias);
    self->in_f = in_f;
    self->out_f = out_f;
    self->device = device;
    PyObject **slots[] = {&self->owner, &self->workspaces, &self->device_key, &self->check};
    PyObject *values[] = {owner, workspaces, key, check};
    for (int i = 0; i < 4; ++i) {
        Py_INCREF(values[i]);
        Py_XSETREF(*slots[i], values[i]);
    }
    return 0;
}

// (called before __init__ has run, or on an object whose __init__ failed)
PyObject *forward_unset(PyObject *, PyObject *const *, size_t, PyObject *) {
    PyErr_SetString(PyExc_RuntimeError, "Forward is not initialised");
    return nullptr;
}

PyObject *forward_new(PyTypeObject *type, PyObject *, PyObject *) {
    PyObject *self = type->tp_alloc(type, 0);
    if (self) reinterpret_cast<Forward *>(self)->call = forward_unset;
    return self;
}

int forward_traverse(PyObject *self_, visitproc visit, void *arg) {
    Forward *self = reinterpret_cast<Forward *>(self_);
    Py_VISIT(self->owner);
    Py_VISIT(self->workspaces);
    Py_VISIT(self->device_key);
    Py_VISIT(self->check);
    return 0;
}

int forward_clear(PyObject *self_) {
    Forward *self = reinterpret_cast<Forward *>(self_);
    self->call = forward_unset;
    Py_CLEAR(self->owner);
    Py_CLEAR(self->workspaces);
    Py_CLEAR(self->device_key);
    Py_CLEAR(self->check);
    return 0;
}

void forward_dealloc(PyObject *self) {
    PyObject_GC_UnTrack(self);
    forward_clear(self);
    Py_TYPE(self)->tp_free(self);
}

PyTypeObject forward_type = {PyVarObject_HEAD_INIT(nullptr, 0)};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", "Host side of the short calls.", -1, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host() {
    forward_type.tp_name = "ixrun_amd._host.Forward";
    forward_type.tp_basicsize = sizeof(Forward);
    forward_type.tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_HAVE_GC | Py_TPFLAGS_HAVE_VECTORCALL;
    forward_type.tp_vectorcall_offset = offsetof(Forward, call);
    forward_type.tp_call = PyVectorcall_Call;
    forward_type.tp_new = forward_new;
    forward_type.tp_init = forward_init;
    forward_type.tp_traverse = forward_traverse;
    forward_type.tp_clear = forward_clear;
    forward_type.tp_dealloc = forward_dealloc;
    if (PyType_Ready(&forward_type) < 0) return nullptr;
    PyObject *m = PyModule_Create(&module);
    if (!m) return nullptr;
    Py_INCREF(&forward_type);
    if (PyModule_AddObject(m, "Forward", reinterpret_cast<PyObject *>(&forward_type)) < 0) {
        Py_DECREF(&forward_type);
        Py_DECREF(m);
        return nullptr;
    }
    return m;
}
