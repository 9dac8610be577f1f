// _ftcall: the call of a built plan, natively.
//
// A call checks its tensors (type, shape, place, contiguity, alignment), puts their addresses into the argument arrays of
// the plan's launches and hands these to ftr_launch_seq on torch's current stream. In Python that took 16 us a
// call (ctypes objects for every argument and descriptor, made anew each time), more than most kernels of a
// single layer: back to back, a 3x3 layer on 1x64x56x56 now takes its 5.1 us on the device instead of 15.7, a depthwise layer
// on 8x512x28x28 4.9 instead of 15.8. Everything but the addresses is laid out once, when the plan is built; a
// call's argument arrays are its own, so several threads may call one plan, and on several streams where the plan
// owns no buffers: its intermediates and workspaces exist once, and calls that use them must not overlap on the device.
//
// A call returns True when the work is enqueued and False when the tensors are not what the plan takes, begin at an
// address its kernels do not load from or are not plain tensors: the caller then goes the general way, which copies
// what is misplaced and says what is wrong.
#include "ftrocm.h"

#include <Python.h>
#include <c10/hip/HIPStream.h>
#include <c10/util/SmallVector.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <vector>

namespace {

typedef int (*launch_seq_t)(const ftr_launch_desc_t *, int, void *);
typedef const char *(*last_error_t)(void);

struct Buffer {
    c10::ScalarType dtype;
    std::vector<int64_t> shape;
    unsigned align;          // the address is a multiple of it
};

struct Arg {
    int tensor;              // index of the caller's tensor whose address it is, or -1: the value below
    unsigned long long value;
};

struct Call {
    PyObject_HEAD
    vectorcallfunc vectorcall;
    launch_seq_t launch_seq;
    last_error_t last_error;
    PyObject *error;                               // raised when a launch fails
    std::vector<Buffer> *bufs;
    std::vector<ftr_launch_desc_t> *launches;      // args: offset into `args` of the launch's first one
    std::vector<Arg> *args;
};

// a call's own arrays: on its stack up to these sizes (a few operators), on the heap for larger graphs
constexpr unsigned kInlineArgs = 64, kInlineLaunches = 16, kInlineBufs = 16;

bool fits(const at::Tensor &t, const Buffer &b) {
    const auto *impl = t.unsafeGetTensorImpl();
    return t.defined() && t.has_storage() && !impl->has_symbolic_sizes_strides() && t.scalar_type() == b.dtype &&
           t.is_cuda() && t.sizes() == c10::IntArrayRef(b.shape) && t.is_contiguous();
}

PyObject *call(PyObject *self_, PyObject *const *argv, size_t nargsf, PyObject *kwnames) {
    HANDLE_TH_ERRORS
    Call *self = reinterpret_cast<Call *>(self_);
    const size_t n = PyVectorcall_NARGS(nargsf);
    if (n != self->bufs->size() || (kwnames && PyTuple_GET_SIZE(kwnames))) Py_RETURN_FALSE;
    c10::SmallVector<void *, kInlineBufs> ptr(n);
    for (size_t i = 0; i < n; ++i) {
        if (!THPVariable_CheckExact(argv[i])) Py_RETURN_FALSE;
        const at::Tensor &t = THPVariable_Unpack(argv[i]);
        if (!fits(t, (*self->bufs)[i])) Py_RETURN_FALSE;
        ptr[i] = t.data_ptr();
        if (reinterpret_cast<uintptr_t>(ptr[i]) % (*self->bufs)[i].align) Py_RETURN_FALSE;
    }
    const std::vector<Arg> &args = *self->args;
    c10::SmallVector<unsigned long long, kInlineArgs> values(args.size());
    c10::SmallVector<void *, kInlineArgs> slots(args.size());
    for (size_t i = 0; i < args.size(); ++i) {
        values[i] = args[i].tensor < 0 ? args[i].value : reinterpret_cast<unsigned long long>(ptr[args[i].tensor]);
        slots[i] = &values[i];
    }
    c10::SmallVector<ftr_launch_desc_t, kInlineLaunches> seq(self->launches->begin(), self->launches->end());
    const int nl = static_cast<int>(seq.size());
    for (ftr_launch_desc_t &d : seq) d.args = slots.data() + reinterpret_cast<size_t>(d.args);
    void *stream = c10::hip::getCurrentHIPStream().stream();
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = self->launch_seq(seq.data(), nl, stream);
    Py_END_ALLOW_THREADS
    if (rc != 0) {
        PyErr_Format(self->error, "ftr_launch_seq: %s", self->last_error());
        return nullptr;
    }
    Py_RETURN_TRUE;
    END_HANDLE_TH_ERRORS
}

void dealloc(PyObject *self_) {
    Call *self = reinterpret_cast<Call *>(self_);
    Py_XDECREF(self->error);
    delete self->bufs;
    delete self->launches;
    delete self->args;
    Py_TYPE(self_)->tp_free(self_);
}

bool dtype_of(const char *name, c10::ScalarType &out) {
    const struct { const char *name; c10::ScalarType type; } known[] = {
        {"float32", c10::kFloat}, {"int8", c10::kChar}, {"int32", c10::kInt}, {"int64", c10::kLong}};
    for (const auto &k : known)
        if (!strcmp(name, k.name)) {
            out = k.type;
            return true;
        }
    return false;
}

// Call(launch_seq, last_error, error, [(dtype, shape, align)...], [(module, grid, block, lds_bytes, [(tensor, value)...])...]);
// raises ValueError for a type it does not know and for an argument that names no buffer
PyObject *create(PyTypeObject *type, PyObject *args, PyObject *) {
    unsigned long long launch_seq, last_error;
    PyObject *error, *bufs, *launches;
    if (!PyArg_ParseTuple(args, "KKOO!O!", &launch_seq, &last_error, &error, &PyList_Type, &bufs, &PyList_Type, &launches))
        return nullptr;
    Call *self = reinterpret_cast<Call *>(type->tp_alloc(type, 0));
    if (!self) return nullptr;
    self->vectorcall = call;
    self->launch_seq = reinterpret_cast<launch_seq_t>(launch_seq);
    self->last_error = reinterpret_cast<last_error_t>(last_error);
    Py_INCREF(error);
    self->error = error;
    self->bufs = new std::vector<Buffer>;
    self->launches = new std::vector<ftr_launch_desc_t>;
    self->args = new std::vector<Arg>;
    bool ok = true;
    for (Py_ssize_t i = 0; ok && i < PyList_GET_SIZE(bufs); ++i) {
        const char *name;
        PyObject *shape;
        Buffer b;
        ok = PyArg_ParseTuple(PyList_GET_ITEM(bufs, i), "sO!I", &name, &PyTuple_Type, &shape, &b.align) &&
             dtype_of(name, b.dtype) && b.align > 0;
        for (Py_ssize_t d = 0; ok && d < PyTuple_GET_SIZE(shape); ++d)
            b.shape.push_back(PyLong_AsLongLong(PyTuple_GET_ITEM(shape, d)));
        self->bufs->push_back(b);
    }
    for (Py_ssize_t i = 0; ok && i < PyList_GET_SIZE(launches); ++i) {
        unsigned long long mod;
        ftr_launch_desc_t d{};
        PyObject *list;
        ok = PyArg_ParseTuple(PyList_GET_ITEM(launches, i), "K(III)(III)IO!", &mod, &d.grid[0], &d.grid[1], &d.grid[2],
                              &d.block[0], &d.block[1], &d.block[2], &d.lds_bytes, &PyList_Type, &list);
        d.mod = reinterpret_cast<ftr_module_t>(mod);
        d.args = reinterpret_cast<void **>(self->args->size());
        for (Py_ssize_t a = 0; ok && a < PyList_GET_SIZE(list); ++a) {
            Arg arg;
            ok = PyArg_ParseTuple(PyList_GET_ITEM(list, a), "iK", &arg.tensor, &arg.value) &&
                 arg.tensor < static_cast<int>(self->bufs->size());
            self->args->push_back(arg);
        }
        self->launches->push_back(d);
    }
    if (!ok || PyErr_Occurred()) {
        if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "_ftcall.Call: unknown type or buffer index");
        Py_DECREF(self);
        return nullptr;
    }
    return reinterpret_cast<PyObject *>(self);
}

PyTypeObject CallType = {PyVarObject_HEAD_INIT(nullptr, 0)};
PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_ftcall", "Native call of a built plan.", -1, nullptr,
                          nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__ftcall(void) {
    CallType.tp_name = "_ftcall.Call";
    CallType.tp_basicsize = sizeof(Call);
    CallType.tp_dealloc = dealloc;
    CallType.tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_HAVE_VECTORCALL;
    CallType.tp_vectorcall_offset = offsetof(Call, vectorcall);
    CallType.tp_call = PyVectorcall_Call;
    CallType.tp_new = create;
    if (PyType_Ready(&CallType) < 0) return nullptr;
    PyObject *m = PyModule_Create(&module_def);
    if (!m) return nullptr;
    Py_INCREF(&CallType);
    if (PyModule_AddObject(m, "Call", reinterpret_cast<PyObject *>(&CallType)) < 0) {
        Py_DECREF(&CallType);
        Py_DECREF(m);
        return nullptr;
    }
    return m;
}
