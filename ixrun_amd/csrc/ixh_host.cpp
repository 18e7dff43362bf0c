// ixrun_amd._host: the host side of the calls whose kernels are shorter than Python's bookkeeping around them.
//
// A forward of one token spends 5 us on the GPU; checked, allocated and launched from Python through ctypes it took the
// host 8.  The same steps here: see the figures at each function.  (Whole calls with the caller's own Python around them, with memory
// allocated through the dispatcher, plain calls found out in Python and the decoders' and the encoder's Python under a no_grad of its own / now: 1536 x
// 1536, one row 7.0 / 6.8 us; 1024 x 1024 at 40 rows 11.4 / 10.5; decode of 1408 x 672 9.3 / 6.5, with group scales of 640 x 1024 9.6 / 7.2; encode of
// 448 x 1024 39.3 / 36.2, of 2048 x 2500 40.0 / 37.3.)  Everything that is not the common case (other types,
// other devices than the current one, views, a scratch that has to grow, errors) is left to the caller: a function returns None and has done
// nothing, and the Python code behind it goes on.
#include <Python.h>
#include <structmember.h>

#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/autocast_mode.h>
#include <ATen/core/Tensor.h>
#include <ATen/hip/EmptyTensor.h>
#include <ATen/ops/empty.h>
#include <c10/core/GradMode.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/hip/HIPStream.h>
#include <vector>

#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/forward_grad.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/ixhip.h"

namespace {

using LanesGemv = decltype(&ixh_lanes_gemv);
constexpr int kMaxRows = 16;

// What this thread has on that looks at what goes through the dispatcher: modes, transforms, tracing.
c10::DispatchKeySet watching() { return c10::impl::tls_local_dispatch_key_set().included_ - c10::default_included_set; }

// Memory on the GPU, as at::empty gives it, which takes 0.3 us longer.
at::Tensor fresh(at::IntArrayRef size, at::ScalarType type, int64_t device) {
    const c10::Device on(c10::kCUDA, (c10::DeviceIndex)device);
    if (watching().empty()) return at::Tensor(at::detail::empty_cuda(size, type, on, std::nullopt));
    return at::empty(size, at::TensorOptions().device(on).dtype(type));
}

// Whether a product of `x`, an exact tensor, that is not torch's own is what the caller gets from F.linear: engine._plain_call, which takes 0.4 us.
bool plain_call(const at::Tensor &x) {
    return !(x.requires_grad() && c10::GradMode::is_enabled()) && !torch::autograd::ForwardADLevel::try_get_by_idx(0) &&
           !at::impl::torch_function_mode_enabled() &&
           !watching().has_any(c10::DispatchKeySet({c10::DispatchKey::FuncTorchDynamicLayerFrontMode, c10::DispatchKey::FuncTorchDynamicLayerBackMode})) &&
           (!at::autocast::is_autocast_enabled(at::kCUDA) || at::autocast::get_autocast_dtype(at::kCUDA) == at::kBFloat16);
}

// The fused forward of one layer over its lane layout: an object called with the activations.
struct Forward {
    PyObject_HEAD
    vectorcallfunc call;
    LanesGemv gemv;
    const IxhLanes *lanes;
    const uint16_t *bias;
    int64_t in_f, out_f;
    long device;
    decltype(&ixh_lanes_gemm) gemm;
    decltype(&ixh_lanes_gemm_workspace_bytes) gemm_workspace_bytes;
    long many_rows;  // rows up to which `many` takes a call; 0 until it is set
    long any_rows;  // more rows than these: plain calls only (no gradient, transform or other result type is asked for)
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
        !x.is_contiguous() || c10::hip::current_device() != self->device)
        Py_RETURN_NONE;
    const int64_t rows = x.numel() / self->in_f;
    if (rows < 1 || rows > kMaxRows) Py_RETURN_NONE;
    if (rows > self->any_rows && !plain_call(x)) Py_RETURN_NONE;
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
        y = fresh(shape, at::kBFloat16, self->device);
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

// many(x): 17 .. many_rows rows, plain calls only.  The slices' sums go through memory allocated for the call.  The host's way from
// Python and through ctypes took longer than the kernels of layers of up to some 2^24 weights: 20 to 21 us a call whatever the rows;
// now 2048 x 2048 at 17 / 100 / 192 rows 10.4 / 13.3 / 17.5, 4096 x 4096 (4 bits) at 32 rows 13.1, 5120 x 5120 at 32 rows 18.6, which
// are the kernels, and 512 x 768 10.6.
PyObject *forward_many(PyObject *self_, PyObject *arg) {
    HANDLE_TH_ERRORS
    Forward *self = reinterpret_cast<Forward *>(self_);
    if (self->call != forward_call || !THPVariable_CheckExact(arg)) Py_RETURN_NONE;
    const at::Tensor &x = THPVariable_Unpack(arg);
    if (!x.is_cuda() || x.scalar_type() != at::kBFloat16 || x.dim() < 1 || x.size(-1) != self->in_f || x.get_device() != self->device ||
        !x.is_contiguous() || c10::hip::current_device() != self->device)
        Py_RETURN_NONE;
    const int64_t rows = x.numel() / self->in_f;
    if (rows <= kMaxRows || rows > self->many_rows || (reinterpret_cast<uintptr_t>(x.const_data_ptr()) & 15u) != 0) Py_RETURN_NONE;
    if (!plain_call(x)) Py_RETURN_NONE;
    c10::SmallVector<int64_t, 4> shape(x.sizes().begin(), x.sizes().end());
    shape.back() = self->out_f;
    at::Tensor y, sums;
    int rc;
    try {
        pybind11::gil_scoped_release without_gil;
        y = fresh(shape, at::kBFloat16, self->device);
        const size_t need = self->gemm_workspace_bytes(self->lanes, (int32_t)rows);
        if (need) sums = fresh({(int64_t)need}, at::kByte, self->device);
        rc = self->gemm(self->lanes, static_cast<const uint16_t *>(x.const_data_ptr()), self->in_f, self->bias, (int32_t)rows,
                        static_cast<uint16_t *>(y.data_ptr()), self->out_f, need ? sums.data_ptr() : nullptr, need,
                        c10::hip::getCurrentHIPStream((c10::DeviceIndex)self->device).stream());
    } catch (const c10::OutOfMemoryError &) {
        Py_RETURN_NONE;  // nothing has been launched; the caller may have a way without the sums' memory
    }
    if (rc) {
        PyObject *r = PyObject_CallFunction(self->check, "i", rc);
        Py_XDECREF(r);
        if (!r) return nullptr;
    }
    return THPVariable_Wrap(std::move(y));
    END_HANDLE_TH_ERRORS
}

// Forward(gemv, lanes, bias, in_f, out_f, device, workspace_bytes, owner, workspaces, device_key, check, gemm,
// gemm_workspace_bytes); addresses as ints.  any_rows and many_rows are 0 until they are set.
int forward_init(PyObject *self_, PyObject *args, PyObject *) {
    Forward *self = reinterpret_cast<Forward *>(self_);
    unsigned long long gemv, lanes, bias, gemm, gemm_workspace_bytes;
    long long in_f, out_f;
    long device;
    PyObject *bytes, *owner, *workspaces, *key, *check;
    if (!PyArg_ParseTuple(args, "KKKLLlO!OO!OOKK", &gemv, &lanes, &bias, &in_f, &out_f, &device, &PyTuple_Type, &bytes, &owner,
                          &PyDict_Type, &workspaces, &key, &check, &gemm, &gemm_workspace_bytes))
        return -1;
    if (!gemv || !lanes || !gemm || !gemm_workspace_bytes || in_f < 1 || out_f < 1 || PyTuple_GET_SIZE(bytes) != kMaxRows + 1) {
        PyErr_SetString(PyExc_ValueError, "Forward: malformed arguments");
        return -1;
    }
    for (int i = 0; i <= kMaxRows; ++i) {
        self->workspace_bytes[i] = PyLong_AsSize_t(PyTuple_GET_ITEM(bytes, i));
        if (PyErr_Occurred()) return -1;
    }
    self->call = forward_call;
    self->gemv = reinterpret_cast<LanesGemv>(gemv);
    self->gemm = reinterpret_cast<decltype(self->gemm)>(gemm);
    self->gemm_workspace_bytes = reinterpret_cast<decltype(self->gemm_workspace_bytes)>(gemm_workspace_bytes);
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

// The library's entry points, as the Python side loaded them.
struct Library {
    decltype(&ixh_prefix_entries) prefix_entries;
    decltype(&ixh_prefix_workspace_bytes) prefix_workspace_bytes;
    decltype(&ixh_prefix_build_ws) prefix_build;
    decltype(&ixh_decode) decode;
    decltype(&ixh_decode_gs) decode_gs;
    decltype(&ixh_decode_unranked_takes) decode_unranked_takes;
    decltype(&ixh_decode_unranked_workspace_bytes) decode_unranked_workspace_bytes;
    decltype(&ixh_decode_unranked_ws) decode_unranked;
    decltype(&ixh_encode_workspace_bytes) encode_workspace_bytes;
    decltype(&ixh_encode_scan_counts) encode_scan;
    decltype(&ixh_encode_wait) encode_wait;
    decltype(&ixh_encode_pack) encode_pack;
    PyObject *check;
} library;

template <class F>
void entry(F &slot, PyObject *address) {
    slot = reinterpret_cast<F>(PyLong_AsUnsignedLongLong(address));
}

// raises what `check` makes of a negative code; false if it did
bool checked(int rc) {
    if (!rc) return true;
    PyObject *r = PyObject_CallFunction(library.check, "i", rc);
    Py_XDECREF(r);
    return r != nullptr;
}

// bind(prefix_entries, prefix_workspace_bytes, prefix_build_ws, decode, decode_gs, decode_unranked_takes, decode_unranked_workspace_bytes,
// decode_unranked_ws, encode_workspace_bytes, encode_scan_counts, encode_wait, encode_pack, check): addresses, and what raises for a negative code
PyObject *bind(PyObject *, PyObject *args) {
    PyObject *f[12], *check;
    if (!PyArg_ParseTuple(args, "OOOOOOOOOOOOO", &f[0], &f[1], &f[2], &f[3], &f[4], &f[5], &f[6], &f[7], &f[8], &f[9], &f[10], &f[11], &check)) return nullptr;
    entry(library.prefix_entries, f[0]);
    entry(library.prefix_workspace_bytes, f[1]);
    entry(library.prefix_build, f[2]);
    entry(library.decode, f[3]);
    entry(library.decode_gs, f[4]);
    entry(library.decode_unranked_takes, f[5]);
    entry(library.decode_unranked_workspace_bytes, f[6]);
    entry(library.decode_unranked, f[7]);
    entry(library.encode_workspace_bytes, f[8]);
    entry(library.encode_scan, f[9]);
    entry(library.encode_wait, f[10]);
    entry(library.encode_pack, f[11]);
    if (PyErr_Occurred()) return nullptr;
    Py_INCREF(check);
    Py_XSETREF(library.check, check);
    Py_RETURN_NONE;
}

// a contiguous tensor of this type on this device, or null
const at::Tensor *plain(PyObject *o, at::ScalarType type, int64_t device) {
    if (!THPVariable_CheckExact(o)) return nullptr;
    const at::Tensor &t = THPVariable_Unpack(o);
    return t.is_cuda() && t.scalar_type() == type && t.get_device() == device && t.is_contiguous() ? &t : nullptr;
}

// fills the descriptor of packed tensors on one device; false for anything that is not as it should be
bool describe(PyObject *level_bits, long long out_f, long long in_f, PyObject *bitmaps, PyObject *streams, PyObject *scale,
              int64_t device, IxhPacked *p) {
    if (!PyTuple_CheckExact(level_bits) || !PyList_CheckExact(bitmaps) || !PyList_CheckExact(streams) || out_f < 1 || in_f < 1)
        return false;
    const Py_ssize_t levels = PyTuple_GET_SIZE(level_bits);
    if (levels < 2 || levels > IXH_MAX_LEVELS || PyList_GET_SIZE(bitmaps) != levels - 1 || PyList_GET_SIZE(streams) != levels)
        return false;
    *p = IxhPacked{};
    p->n_levels = (int32_t)levels;
    p->out_f = out_f;
    p->in_f = in_f;
    for (Py_ssize_t i = 0; i < levels; ++i) {
        PyObject *b = PyTuple_GET_ITEM(level_bits, i);
        if (!PyLong_CheckExact(b)) return false;
        p->level_bits[i] = (int32_t)PyLong_AsLong(b);
        if (PyErr_Occurred()) {
            PyErr_Clear();
            return false;
        }
    }
    for (Py_ssize_t i = 0; i < levels - 1; ++i) {
        const at::Tensor *bm = plain(PyList_GET_ITEM(bitmaps, i), at::kInt, device);
        const at::Tensor *st = plain(PyList_GET_ITEM(streams, i), at::kInt, device);
        if (!bm || !st) return false;
        p->bitmap_words[i] = (uint64_t)bm->numel();
        p->stream_words[i] = (uint64_t)st->numel();
        p->bitmaps[i] = bm->numel() ? static_cast<const uint32_t *>(bm->const_data_ptr()) : nullptr;
        p->streams[i] = st->numel() ? static_cast<const uint32_t *>(st->const_data_ptr()) : nullptr;
    }
    const at::Tensor *last = plain(PyList_GET_ITEM(streams, levels - 1), at::kByte, device);
    if (!last) return false;
    p->last_bytes = (uint64_t)last->numel();
    p->last = last->numel() ? static_cast<const uint8_t *>(last->const_data_ptr()) : nullptr;
    if (scale != Py_None) {
        const at::Tensor *s = plain(scale, at::kBFloat16, device);
        if (!s || s->numel() != 1) return false;
        p->scale = static_cast<const uint16_t *>(s->const_data_ptr());
    }
    return true;
}

// decode(level_bits, out_f, in_f, bitmaps, streams, scale, table, group_scales, group_size): the bf16 weight, by units of
// 512; without a rank table small (3,5,8) tensors do without and for others one is built, with group scales (fp16, in place of `scale`) they are used.  Of tensors on the
// current device.
// 2048 x 2048 with a table: 6 us of host time (17 from Python).
PyObject *decode(PyObject *, PyObject *const *args, Py_ssize_t n_args) {
    HANDLE_TH_ERRORS
    constexpr int64_t kUnit = 512;
    if (n_args != 9 || !library.check) {
        PyErr_SetString(PyExc_TypeError, "decode: nine arguments, after bind");
        return nullptr;
    }
    const long long out_f = PyLong_AsLongLong(args[1]), in_f = PyLong_AsLongLong(args[2]), group = PyLong_AsLongLong(args[8]);
    if (PyErr_Occurred()) return nullptr;
    const int64_t device = c10::hip::current_device();
    IxhPacked p;
    if (!describe(args[0], out_f, in_f, args[3], args[4], args[5], device, &p) || out_f > (1ll << 31) / in_f) Py_RETURN_NONE;
    const int64_t n = out_f * in_f, entries = library.prefix_entries(n, kUnit), rows = p.n_levels - 1;
    const at::Tensor *scales = nullptr;
    if (args[7] != Py_None) {
        scales = plain(args[7], at::kHalf, device);
        if (!scales || group < 1 || scales->numel() < (n + group - 1) / group) Py_RETURN_NONE;
    } else if (!p.scale) {
        Py_RETURN_NONE;
    }
    const at::Tensor *given = nullptr;
    if (args[6] != Py_None) {
        given = plain(args[6], at::kInt, device);
        if (!given || given->numel() < rows * entries) Py_RETURN_NONE;
    }
    at::Tensor w, table;
    int rc = 0;
    {
        pybind11::gil_scoped_release without_gil;
        ixh_stream_t stream = c10::hip::getCurrentHIPStream((c10::DeviceIndex)device).stream();
        w = fresh({out_f, in_f}, at::kBFloat16, device);
        uint16_t *out = static_cast<uint16_t *>(w.data_ptr());
        const uint16_t *of_groups = scales ? static_cast<const uint16_t *>(scales->const_data_ptr()) : nullptr;
        const bool ranked = given || !library.decode_unranked_takes(&p, of_groups, group, out);
        if (!ranked) {
            const size_t bytes = library.decode_unranked_workspace_bytes(&p);
            if (bytes) table = fresh({(int64_t)bytes / 4}, at::kInt, device);
            rc = library.decode_unranked(&p, of_groups, group, out, bytes ? table.data_ptr() : nullptr, bytes, stream);
        } else if (!given) {
            const size_t bytes = library.prefix_workspace_bytes(n, kUnit, p.n_levels);
            table = fresh({rows * entries + (int64_t)bytes / 4}, at::kInt, device);  // and the scratch
            int32_t *ranks = static_cast<int32_t *>(table.data_ptr());
            rc = library.prefix_build(&p, kUnit, ranks, ranks + rows * entries, bytes, stream);
        }
        if (ranked && !rc) {
            const int32_t *ranks = static_cast<const int32_t *>((given ? *given : table).const_data_ptr());
            rc = scales ? library.decode_gs(&p, ranks, kUnit, of_groups, group, out, stream)
                        : library.decode(&p, ranks, kUnit, nullptr, out, stream);
        }
    }
    if (!checked(rc)) return nullptr;
    return THPVariable_Wrap(std::move(w));
    END_HANDLE_TH_ERRORS
}

// describe(address of an IxhPacked, level_bits, out_f, in_f, bitmaps, streams, scale): whether it was filled.  Of tensors on
// one device.
PyObject *describe_at(PyObject *, PyObject *const *args, Py_ssize_t n_args) {
    HANDLE_TH_ERRORS
    if (n_args != 7) {
        PyErr_SetString(PyExc_TypeError, "describe: seven arguments");
        return nullptr;
    }
    IxhPacked *p = reinterpret_cast<IxhPacked *>(PyLong_AsUnsignedLongLong(args[0]));
    const long long out_f = PyLong_AsLongLong(args[2]), in_f = PyLong_AsLongLong(args[3]);
    if (PyErr_Occurred()) return nullptr;
    if (!PyList_CheckExact(args[4]) || PyList_GET_SIZE(args[4]) == 0 || !THPVariable_CheckExact(PyList_GET_ITEM(args[4], 0)))
        Py_RETURN_FALSE;
    const at::Tensor &first = THPVariable_Unpack(PyList_GET_ITEM(args[4], 0));
    if (!first.is_cuda()) Py_RETURN_FALSE;
    IxhPacked filled;
    if (!describe(args[1], out_f, in_f, args[4], args[5], args[6], first.get_device(), &filled)) Py_RETURN_FALSE;
    *p = filled;
    Py_RETURN_TRUE;
    END_HANDLE_TH_ERRORS
}

// encode(weight, level_bits): (bitmaps, streams, scale, table, counts) of a contiguous bf16 matrix on the current device.
// Waits once, for the counts.  The host between the counts' arrival and the packing kernels is time that the GPU idles:
// 4 us (13 from Python).
PyObject *encode(PyObject *, PyObject *const *args, Py_ssize_t n_args) {
    HANDLE_TH_ERRORS
    if (n_args != 2 || !library.check) {
        PyErr_SetString(PyExc_TypeError, "encode: two arguments, after bind");
        return nullptr;
    }
    const int64_t device = c10::hip::current_device();
    const at::Tensor *w = plain(args[0], at::kBFloat16, device);
    if (!w || w->dim() != 2 || !PyTuple_CheckExact(args[1])) Py_RETURN_NONE;
    const int64_t out_f = w->size(0), in_f = w->size(1), n = w->numel();
    const int levels = (int)PyTuple_GET_SIZE(args[1]);
    if (n < 1 || levels < 2 || levels > IXH_MAX_LEVELS) Py_RETURN_NONE;
    IxhPacked p{};
    p.n_levels = levels;
    p.out_f = out_f;
    p.in_f = in_f;
    for (int i = 0; i < levels; ++i) {
        p.level_bits[i] = (int32_t)PyLong_AsLong(PyTuple_GET_ITEM(args[1], i));
        if (PyErr_Occurred()) return nullptr;
    }
    const size_t bytes = library.encode_workspace_bytes(out_f, in_f, levels);
    const int64_t entries = library.prefix_entries(n, 512);
    std::vector<at::Tensor> bitmaps(levels - 1), streams(levels);
    at::Tensor scale, table, arrived, scratch;
    int64_t counts[IXH_MAX_LEVELS];
    int rc;
    {
        pybind11::gil_scoped_release without_gil;
        ixh_stream_t stream = c10::hip::getCurrentHIPStream((c10::DeviceIndex)device).stream();
        const uint16_t *src = static_cast<const uint16_t *>(w->const_data_ptr());
        scratch = fresh({(int64_t)bytes}, at::kByte, device);
        scale = fresh({1}, at::kBFloat16, device);
        table = fresh({levels - 1, entries}, at::kInt, device);
        arrived = at::empty({levels - 1}, at::TensorOptions().dtype(at::kLong).pinned_memory(true));
        bitmaps[0] = fresh({(n + 31) / 32}, at::kInt, device);
        int32_t *ranks = static_cast<int32_t *>(table.data_ptr());
        int64_t *host = static_cast<int64_t *>(arrived.data_ptr());
        rc = library.encode_scan(src, out_f, in_f, levels, p.level_bits, static_cast<uint16_t *>(scale.data_ptr()), ranks,
                                 scratch.data_ptr(), bytes, host, stream);
        if (!rc) rc = library.encode_wait(host, levels - 1, stream);  // (nothing that throws in between: the kernel writes to `arrived`)
        if (!rc) {
            int64_t left = n;
            for (int i = 0; i < levels - 1; ++i) {
                counts[i] = host[i];
                if (i > 0) bitmaps[i] = fresh({(left + 31) / 32}, at::kInt, device);
                streams[i] = fresh({(counts[i] * p.level_bits[i] + 31) / 32}, at::kInt, device);
                p.bitmap_words[i] = (uint64_t)bitmaps[i].numel();
                p.stream_words[i] = (uint64_t)streams[i].numel();
                p.bitmaps[i] = bitmaps[i].numel() ? static_cast<const uint32_t *>(bitmaps[i].data_ptr()) : nullptr;
                p.streams[i] = streams[i].numel() ? static_cast<const uint32_t *>(streams[i].data_ptr()) : nullptr;
                left -= counts[i];
            }
            counts[levels - 1] = left;
            streams[levels - 1] = fresh({left}, at::kByte, device);
            p.last_bytes = (uint64_t)left;
            p.last = left ? static_cast<const uint8_t *>(streams[levels - 1].data_ptr()) : nullptr;
            p.scale = static_cast<const uint16_t *>(scale.data_ptr());
            rc = library.encode_pack(src, &p, ranks, stream);
        }
    }
    if (!checked(rc)) return nullptr;
    PyObject *bm = PyList_New(levels - 1), *st = PyList_New(levels), *cn = PyList_New(levels);
    bool ok = bm && st && cn;
    for (int i = 0; ok && i < levels; ++i) {
        PyObject *s = THPVariable_Wrap(streams[i]), *c = PyLong_FromLongLong(counts[i]);
        PyObject *b = i < levels - 1 ? THPVariable_Wrap(bitmaps[i]) : nullptr;
        ok = s && c && (b || i == levels - 1);
        if (s) PyList_SET_ITEM(st, i, s);
        if (c) PyList_SET_ITEM(cn, i, c);
        if (b) PyList_SET_ITEM(bm, i, b);
    }
    PyObject *result = ok ? Py_BuildValue("(OONNO)", bm, st, THPVariable_Wrap(scale), THPVariable_Wrap(table), cn) : nullptr;
    Py_XDECREF(bm);
    Py_XDECREF(st);
    Py_XDECREF(cn);
    return result;
    END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {
    {"bind", bind, METH_VARARGS, "The library's entry points."},
    {"decode", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(decode)), METH_FASTCALL, "The bf16 weight of packed tensors, or None."},
    {"describe", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(describe_at)), METH_FASTCALL, "Fills an IxhPacked."},
    {"encode", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(encode)), METH_FASTCALL, "Packed tensors of a bf16 weight, or None."},
    {nullptr, nullptr, 0, nullptr},
};

PyMemberDef forward_members[] = {
    {"any_rows", T_LONG, offsetof(Forward, any_rows), 0, "Rows up to which calls that are not plain are taken too."},
    {"many_rows", T_LONG, offsetof(Forward, many_rows), 0, "Rows up to which `many` takes a call."},
    {nullptr, 0, 0, 0, nullptr},
};

PyMethodDef forward_methods[] = {
    {"many", forward_many, METH_O, "The forward of more rows than a call takes, or None."},
    {nullptr, nullptr, 0, nullptr},
};

PyTypeObject forward_type = {PyVarObject_HEAD_INIT(nullptr, 0)};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", "Host side of the short calls.", -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit__host() {
    forward_type.tp_name = "ixrun_amd._host.Forward";
    forward_type.tp_basicsize = sizeof(Forward);
    forward_type.tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_HAVE_GC | Py_TPFLAGS_HAVE_VECTORCALL;
    forward_type.tp_vectorcall_offset = offsetof(Forward, call);
    forward_type.tp_call = PyVectorcall_Call;
    forward_type.tp_members = forward_members;
    forward_type.tp_methods = forward_methods;
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
