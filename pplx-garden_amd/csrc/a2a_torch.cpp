// The operator's host path: tensors in, calls of the C ABI out.
//
// A step of eight ranks is sixteen operator calls (thirty-two through the split calls), and each has to
// look at six to eight tensors (shape, strides, type, address: some forty attributes) before one of them
// launches anything.  In Python that was 5.8 us a call, so that a decode step of 12 us on the GPU took 93;
// here a call that launches nothing is 0.2-0.3 us, most of it the interpreter's own way in and out (through a
// Python function in front of it 0.1 us more: call_without_a_frame below; 8 ranks x 1 token 11.3 -> 10.6 us a step).
//
// Plays the part of the reference's pyo3 classes (python-ext/src/py_p2p_all_to_all.rs:17-205) one level
// higher: it takes the tensors themselves and makes the checks of the reference's operator
// (python/pplx_garden/kernels/p2p_all_to_all.py:317-517).  CPython's C interface and torch's tensor
// class, nothing else: a tensor's fields are read in place and nothing is wrapped or converted.
#include <Python.h>

#include <ATen/core/Tensor.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstring>
#include <new>
#include <string>

#include "a2a.h"

namespace {

using at::ScalarType;
using at::Tensor;

// ---------------------------------------------------------------------------
// Context: the handle every user of one native context shares.  Closed by whoever destroys the context,
// so that a call made afterwards fails instead of using freed memory.  Also holds what the ranks of a
// collective have passed until the last of them calls.
// ---------------------------------------------------------------------------
constexpr int kKept = 8;   // tensors of one call that have to outlive it

template <typename Args>
struct Pending {
    Args args[A2A_MAX_WORLD_SIZE];
    uint32_t mode[A2A_MAX_WORLD_SIZE];               // what every rank has to pass alike
    PyObject *kept[A2A_MAX_WORLD_SIZE][kKept] = {};
    uint32_t posted = 0;                             // ranks that have called

    // Drops the references taken for the ranks in `ranks` (moved out of `kept` first: dropping one may run code).
    void release(uint32_t ranks) {
        for (int r = 0; r < A2A_MAX_WORLD_SIZE; ++r) {
            if (!(ranks >> r & 1)) continue;
            for (PyObject *&slot : kept[r]) {
                PyObject *old = slot;
                slot = nullptr;
                Py_XDECREF(old);
            }
        }
    }
};

struct Context {
    PyObject_HEAD
    a2a_ctx *ctx;
    uint32_t world;
    Pending<a2a_dispatch_args> *dispatch;
    Pending<a2a_combine_args> *combine;
};

PyObject *raise_last_error(a2a_ctx *ctx, const char *what, int rc) {
    const char *text = a2a_last_error(ctx);
    if (text != nullptr && text[0] != '\0') {
        PyErr_SetString(PyExc_RuntimeError, text);
    } else {
        PyErr_Format(PyExc_RuntimeError, "%s failed with code %d", what, rc);
    }
    return nullptr;
}

bool require_open(Context *c) {
    if (c->ctx != nullptr) return true;
    PyErr_SetString(PyExc_RuntimeError, "AllToAllContext has been destroyed");
    return false;
}

PyObject *context_new(PyTypeObject *type, PyObject *args, PyObject *) {
    unsigned long long handle;
    unsigned int world;
    if (!PyArg_ParseTuple(args, "KI", &handle, &world)) return nullptr;
    if (world < 1 || world > A2A_MAX_WORLD_SIZE) {
        PyErr_SetString(PyExc_ValueError, "world size out of range");
        return nullptr;
    }
    Context *c = reinterpret_cast<Context *>(type->tp_alloc(type, 0));
    if (c == nullptr) return nullptr;
    c->ctx = reinterpret_cast<a2a_ctx *>(handle);
    c->world = world;
    c->dispatch = new (std::nothrow) Pending<a2a_dispatch_args>();
    c->combine = new (std::nothrow) Pending<a2a_combine_args>();
    if (c->dispatch == nullptr || c->combine == nullptr) {
        Py_DECREF(c);
        return PyErr_NoMemory();
    }
    return reinterpret_cast<PyObject *>(c);
}

void context_dealloc(PyObject *self) {
    Context *c = reinterpret_cast<Context *>(self);
    if (c->dispatch != nullptr) c->dispatch->release(0xFFFFFFFFu);
    if (c->combine != nullptr) c->combine->release(0xFFFFFFFFu);
    delete c->dispatch;
    delete c->combine;
    Py_TYPE(self)->tp_free(self);
}

// Forgets the handle and what ranks have posted: from here on every call is refused.
PyObject *context_close(PyObject *self, PyObject *) {
    Context *c = reinterpret_cast<Context *>(self);
    c->ctx = nullptr;
    c->dispatch->posted = 0;
    c->combine->posted = 0;
    c->dispatch->release(0xFFFFFFFFu);
    c->combine->release(0xFFFFFFFFu);
    Py_RETURN_NONE;
}

// Ranks that wait in collective "dispatch" or "combine", as a bit mask.
PyObject *context_pending(PyObject *self, PyObject *kind) {
    Context *c = reinterpret_cast<Context *>(self);
    const char *name = PyUnicode_AsUTF8(kind);
    if (name == nullptr) return nullptr;
    if (strcmp(name, "dispatch") == 0) return PyLong_FromUnsignedLong(c->dispatch->posted);
    if (strcmp(name, "combine") == 0) return PyLong_FromUnsignedLong(c->combine->posted);
    return PyErr_Format(PyExc_ValueError, "no collective %s: \"dispatch\" or \"combine\"", name);
}

// The arguments of all ranks out of a C array (ctypes) of at least `world` structures.
template <typename Args>
bool array_of(PyObject *obj, uint32_t world, Py_buffer *view) {
    if (PyObject_GetBuffer(obj, view, PyBUF_SIMPLE) != 0) return false;
    const bool right_type = view->itemsize == (Py_ssize_t)sizeof(Args);
    if (right_type && view->len >= (Py_ssize_t)(sizeof(Args) * world)) return true;
    PyBuffer_Release(view);
    if (right_type) {
        PyErr_Format(PyExc_RuntimeError, "expected arguments of %u ranks", world);
    } else {
        PyErr_SetString(PyExc_TypeError, "an array of another call's arguments");
    }
    return false;
}

// A number as int() makes it (numpy's integers too), as the 32 bits of a C argument or as an address.
bool integer_of(PyObject *obj, uint32_t *out) {
    PyObject *number = PyNumber_Long(obj);
    if (number == nullptr) return false;
    *out = (uint32_t)PyLong_AsUnsignedLongMask(number);
    Py_DECREF(number);
    return !PyErr_Occurred();
}

bool address_of(PyObject *obj, void **out) {
    PyObject *number = PyNumber_Long(obj);
    if (number == nullptr) return false;
    *out = PyLong_AsVoidPtr(number);
    Py_DECREF(number);
    return !PyErr_Occurred();
}

// group_dispatch(array, quantize, stream)
PyObject *context_group_dispatch(PyObject *self, PyObject *const *args, Py_ssize_t n) {
    Context *c = reinterpret_cast<Context *>(self);
    if (n != 3) return PyErr_Format(PyExc_TypeError, "group_dispatch takes 3 arguments");
    uint32_t quantize;
    void *stream;
    if (!integer_of(args[1], &quantize) || !address_of(args[2], &stream)) return nullptr;
    Py_buffer view;
    if (!array_of<a2a_dispatch_args>(args[0], c->world, &view)) return nullptr;
    if (!require_open(c)) {
        PyBuffer_Release(&view);
        return nullptr;
    }
    a2a_ctx *const ctx = c->ctx;
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = a2a_dispatch(ctx, static_cast<const a2a_dispatch_args *>(view.buf), quantize, stream);
    Py_END_ALLOW_THREADS
    PyBuffer_Release(&view);
    if (rc != 0) return raise_last_error(ctx, "a2a_dispatch", rc);
    Py_RETURN_NONE;
}

// group_combine(array, expert_y type tag, accumulate, stream)
PyObject *context_group_combine(PyObject *self, PyObject *const *args, Py_ssize_t n) {
    Context *c = reinterpret_cast<Context *>(self);
    if (n != 4) return PyErr_Format(PyExc_TypeError, "group_combine takes 4 arguments");
    uint32_t tag;
    void *stream;
    if (!integer_of(args[1], &tag) || !address_of(args[3], &stream)) return nullptr;
    const int accumulate = PyObject_IsTrue(args[2]);
    if (accumulate < 0) return nullptr;
    Py_buffer view;
    if (!array_of<a2a_combine_args>(args[0], c->world, &view)) return nullptr;
    if (!require_open(c)) {
        PyBuffer_Release(&view);
        return nullptr;
    }
    a2a_ctx *const ctx = c->ctx;
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = a2a_combine(ctx, static_cast<const a2a_combine_args *>(view.buf), tag, (uint32_t)accumulate, stream);
    Py_END_ALLOW_THREADS
    PyBuffer_Release(&view);
    if (rc != 0) return raise_last_error(ctx, "a2a_combine", rc);
    Py_RETURN_NONE;
}

PyMethodDef context_methods[] = {
    {"close", context_close, METH_NOARGS, nullptr},
    {"pending", context_pending, METH_O, nullptr},
    {"group_dispatch", reinterpret_cast<PyCFunction>(reinterpret_cast<void *>(context_group_dispatch)), METH_FASTCALL,
     nullptr},
    {"group_combine", reinterpret_cast<PyCFunction>(reinterpret_cast<void *>(context_group_combine)), METH_FASTCALL,
     nullptr},
    {nullptr, nullptr, 0, nullptr},
};

PyTypeObject ContextType = {PyVarObject_HEAD_INIT(nullptr, 0)};

// ---------------------------------------------------------------------------
// Operator: one logical rank's dispatch() and combine().
// ---------------------------------------------------------------------------
struct Operator {
    PyObject_HEAD
    Context *context;
    uint32_t rank, world, dp_size;
    int64_t hidden_dim, hidden_dim_scale;   // hidden_dim_scale -1: rows carry no scales
    int64_t local_experts, topk;
    ScalarType in_dtype, out_dtype;
    bool has_scale_dtype;
    c10::DeviceIndex device;                // -1: the device that is current at the call
};

int tag_of(ScalarType t) {
    switch (t) {
        case ScalarType::Half: return A2A_F16;
        case ScalarType::BFloat16: return A2A_BF16;
        case ScalarType::Float: return A2A_F32;
        case ScalarType::Double: return A2A_F64;
        case ScalarType::Float8_e4m3fn: return A2A_F8_E4M3;
        case ScalarType::Float8_e5m2: return A2A_F8_E5M2;
        default: return -1;
    }
}

PyObject *operator_new(PyTypeObject *type, PyObject *args, PyObject *) {
    PyObject *context, *in_dtype, *out_dtype;
    unsigned int rank, dp_size;
    long long hidden, scale, local, topk;
    int has_scale_dtype, device;
    if (!PyArg_ParseTuple(args, "O!IILLLLO!O!pi", &ContextType, &context, &rank, &dp_size, &hidden, &scale, &local, &topk,
                          &THPDtypeType, &in_dtype, &THPDtypeType, &out_dtype, &has_scale_dtype, &device))
        return nullptr;
    Operator *op = reinterpret_cast<Operator *>(type->tp_alloc(type, 0));
    if (op == nullptr) return nullptr;
    Py_INCREF(context);
    op->context = reinterpret_cast<Context *>(context);
    op->rank = rank;
    op->world = op->context->world;
    op->dp_size = dp_size;
    op->hidden_dim = hidden;
    op->hidden_dim_scale = scale;
    op->local_experts = local;
    op->topk = topk;
    op->in_dtype = reinterpret_cast<THPDtype *>(in_dtype)->scalar_type;
    op->out_dtype = reinterpret_cast<THPDtype *>(out_dtype)->scalar_type;
    op->has_scale_dtype = has_scale_dtype != 0;
    op->device = (c10::DeviceIndex)device;
    if (rank >= op->world || dp_size < 1) {
        Py_DECREF(op);
        PyErr_SetString(PyExc_ValueError, "rank or dp_size out of range");
        return nullptr;
    }
    return reinterpret_cast<PyObject *>(op);
}

void operator_dealloc(PyObject *self) {
    Py_XDECREF(reinterpret_cast<Operator *>(self)->context);
    Py_TYPE(self)->tp_free(self);
}

// A condition of the operator's interface; like the reference's asserts, with the condition as the text.
#define A2A_REQUIRE(cond)                                  \
    do {                                                   \
        if (!(cond)) {                                     \
            PyErr_SetString(PyExc_AssertionError, #cond);  \
            return nullptr;                                \
        }                                                  \
    } while (0)

const Tensor *tensor_of(PyObject *obj, const char *name) {
    if (!THPVariable_Check(obj)) {
        PyErr_Format(PyExc_TypeError, "%s must be a torch.Tensor, got %s", name, Py_TYPE(obj)->tp_name);
        return nullptr;
    }
    return &THPVariable_Unpack(obj);
}

const Tensor *matrix_of(PyObject *obj, const char *name, PyObject *error) {
    const Tensor *t = tensor_of(obj, name);
    if (t != nullptr && t->dim() != 2) {
        PyErr_Format(error, "%s must have two dimensions, has %d", name, (int)t->dim());
        return nullptr;
    }
    return t;
}

// Scales: the strides of the first two dimensions are all that is read of their layout; further ones may follow.
const Tensor *scales_of(PyObject *obj, const char *name) {
    const Tensor *t = tensor_of(obj, name);
    if (t != nullptr && t->dim() < 2) {
        PyErr_Format(PyExc_IndexError, "%s must have at least two dimensions, has %d", name, (int)t->dim());
        return nullptr;
    }
    return t;
}

bool has_shape(const Tensor &t, int64_t rows, int64_t cols) { return t.size(0) == rows && t.size(1) == cols; }

uint64_t row_bytes(const Tensor &t) { return (uint64_t)t.stride(0) * t.element_size(); }

// Stands beside a rank's arguments until the collective runs.
void keep(PyObject *(&slots)[kKept], PyObject *const (&given)[kKept]) {
    for (int i = 0; i < kKept; ++i) {
        Py_XINCREF(given[i]);
        slots[i] = given[i];
    }
}

// Records the arguments of `rank`; returns 1 when it was the last one, 0 when others are missing, -1 on error.
template <typename Args>
int post(Pending<Args> &p, const char *kind, uint32_t rank, uint32_t world, const Args &args, uint32_t mode,
         PyObject *const (&given)[kKept]) {
    const uint32_t all = world >= 32 ? 0xFFFFFFFFu : (1u << world) - 1;
    if (p.posted >> rank & 1) {
        std::string missing;
        for (uint32_t r = 0; r < world; ++r) {
            if (!(p.posted >> r & 1)) missing += (missing.empty() ? "" : ", ") + std::to_string(r);
        }
        PyErr_Format(PyExc_RuntimeError,
                     "rank %u called %s() twice before ranks [%s] called it: in loopback "
                     "a collective runs when every logical rank has made the call",
                     rank, kind, missing.c_str());
        return -1;
    }
    p.args[rank] = args;
    p.mode[rank] = mode;
    keep(p.kept[rank], given);
    p.posted |= 1u << rank;
    return p.posted == all ? 1 : 0;
}

// The posted collective, taken out so that the next one can be posted while this one runs.
template <typename Args>
struct Taken {
    Pending<Args> &from;
    Args args[A2A_MAX_WORLD_SIZE];
    PyObject *kept[A2A_MAX_WORLD_SIZE][kKept];
    uint32_t world;
    bool alike = true;

    Taken(Pending<Args> &p, uint32_t n) : from(p), world(n) {
        for (uint32_t r = 0; r < n; ++r) {
            args[r] = p.args[r];
            if (p.mode[r] != p.mode[0]) alike = false;
            for (int i = 0; i < kKept; ++i) {
                kept[r][i] = p.kept[r][i];
                p.kept[r][i] = nullptr;
            }
        }
        p.posted = 0;
    }
    ~Taken() {
        for (uint32_t r = 0; r < world; ++r) {
            for (PyObject *o : kept[r]) Py_XDECREF(o);
        }
    }
};

void *current_stream(const Operator *op) { return c10::hip::getCurrentHIPStream(op->device).stream(); }

// The arguments of a call by position and by name, as a Python function with these parameters would take them: `a` comes
// in with the defaults (null where there is none) and goes out complete.
constexpr int kMostParameters = 10;

struct Parameters {
    const char *call;
    int count;
    const char *name[kMostParameters];
    PyObject *interned[kMostParameters];   // (names in a call are interned strings: found by address)
};

Parameters dispatch_parameters = {"dispatch", 10,
                                  {"out_expert_num_tokens", "out_expert_x", "out_expert_x_scale", "dp_x", "dp_x_scale",
                                   "indices", "weights", "bound_m", "do_send", "do_recv"}, {}};
Parameters combine_parameters = {"combine", 8,
                                 {"out_tokens", "indices", "weights", "expert_y", "bound_m", "do_send", "do_recv",
                                  "accumulate"}, {}};

bool intern_names(Parameters &p) {
    for (int i = 0; i < p.count; ++i) {
        p.interned[i] = PyUnicode_InternFromString(p.name[i]);
        if (p.interned[i] == nullptr) return false;
    }
    return true;
}

bool take_arguments(const Parameters &p, PyObject *const *args, Py_ssize_t n, PyObject *keywords, PyObject **a) {
    if (n > p.count) {
        PyErr_Format(PyExc_TypeError, "%s() takes %d arguments but %zd were given", p.call, p.count, n);
        return false;
    }
    for (Py_ssize_t i = 0; i < n; ++i) a[i] = args[i];
    uint32_t given = (1u << n) - 1;
    const Py_ssize_t named = keywords != nullptr ? PyTuple_GET_SIZE(keywords) : 0;
    for (Py_ssize_t i = 0; i < named; ++i) {
        PyObject *const key = PyTuple_GET_ITEM(keywords, i);
        int at = 0;
        while (at < p.count && p.interned[at] != key) ++at;
        if (at == p.count) {
            for (at = 0; at < p.count && PyUnicode_Compare(p.interned[at], key) != 0; ++at) {
            }
        }
        if (at == p.count) {
            PyErr_Format(PyExc_TypeError, "%s() got an unexpected keyword argument '%U'", p.call, key);
            return false;
        }
        if (given >> at & 1) {
            PyErr_Format(PyExc_TypeError, "%s() got multiple values for argument '%s'", p.call, p.name[at]);
            return false;
        }
        given |= 1u << at;
        a[at] = args[n + i];
    }
    for (int i = 0; i < p.count; ++i) {
        if (a[i] == nullptr) {
            PyErr_Format(PyExc_TypeError, "%s() missing required argument: '%s'", p.call, p.name[i]);
            return false;
        }
    }
    return true;
}

// dispatch(out_expert_num_tokens, out_expert_x, out_expert_x_scale, dp_x, dp_x_scale, indices, weights, bound_m=None,
//          do_send=True, do_recv=True)
PyObject *dispatch(Operator *op, PyObject *const *args, Py_ssize_t n, PyObject *keywords) {
    PyObject *a[kMostParameters] = {nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, Py_None, Py_True, Py_True};
    if (!take_arguments(dispatch_parameters, args, n, keywords, a)) return nullptr;
    const int do_send = PyObject_IsTrue(a[8]), do_recv = PyObject_IsTrue(a[9]);
    if (do_send < 0 || do_recv < 0) return nullptr;
    A2A_REQUIRE(do_send || do_recv);
    Context *const c = op->context;

    a2a_dispatch_args d;
    // Output count buffer (p2p_all_to_all.py:336-340).
    const Tensor *out_n = tensor_of(a[0], "out_expert_num_tokens");
    if (out_n == nullptr) return nullptr;
    A2A_REQUIRE(out_n->dim() == 1 && out_n->size(0) == op->local_experts);
    A2A_REQUIRE(out_n->stride(0) == 1);
    A2A_REQUIRE(out_n->scalar_type() == ScalarType::Int);
    // Output token buffer (p2p_all_to_all.py:342-348).
    const Tensor *out_x = matrix_of(a[1], "out_expert_x", PyExc_ValueError);
    if (out_x == nullptr) return nullptr;
    A2A_REQUIRE(out_x->size(1) == op->hidden_dim);
    A2A_REQUIRE(out_x->stride(1) == 1);
    A2A_REQUIRE(out_x->scalar_type() == op->in_dtype);
    // Output scale buffer (p2p_all_to_all.py:350-362).
    const Tensor *out_scale = nullptr;
    if (a[2] != Py_None) {
        out_scale = scales_of(a[2], "out_expert_x_scale");
        if (out_scale == nullptr) return nullptr;
        A2A_REQUIRE(op->has_scale_dtype && out_scale->scalar_type() == ScalarType::Float);
    }
    // Input tokens (p2p_all_to_all.py:364-369): rows of in_dtype, or bf16 rows that dispatch quantises.
    const Tensor *x = matrix_of(a[3], "dp_x", PyExc_ValueError);
    if (x == nullptr) return nullptr;
    const int64_t tokens = x->size(0);
    const bool quantize = a[4] == Py_None && x->scalar_type() == ScalarType::BFloat16 &&
                          op->in_dtype == ScalarType::Float8_e4m3fn && op->hidden_dim_scale >= 0;
    A2A_REQUIRE(x->size(1) == op->hidden_dim);
    A2A_REQUIRE(x->stride(1) == 1);
    if (quantize) {
        A2A_REQUIRE(op->hidden_dim % 128 == 0);
        A2A_REQUIRE(op->hidden_dim_scale == op->hidden_dim / 128);
        A2A_REQUIRE(op->has_scale_dtype);
        A2A_REQUIRE(out_scale != nullptr);
    } else {
        A2A_REQUIRE(x->scalar_type() == op->in_dtype);
    }
    // Input scales (p2p_all_to_all.py:371-388).
    const Tensor *x_scale = nullptr;
    if (a[4] != Py_None) {
        x_scale = scales_of(a[4], "dp_x_scale");
        if (x_scale == nullptr) return nullptr;
        A2A_REQUIRE(op->has_scale_dtype && op->hidden_dim_scale >= 0);
        A2A_REQUIRE(out_scale != nullptr);
        A2A_REQUIRE(x_scale->scalar_type() == ScalarType::Float);
    } else if (!quantize) {
        A2A_REQUIRE(!op->has_scale_dtype && op->hidden_dim_scale < 0);
    }
    // Indices and weights (p2p_all_to_all.py:390-402).
    const Tensor *indices = matrix_of(a[5], "indices", PyExc_AssertionError);
    if (indices == nullptr) return nullptr;
    A2A_REQUIRE(has_shape(*indices, tokens, op->topk));
    A2A_REQUIRE(indices->stride(1) == 1);
    A2A_REQUIRE(indices->scalar_type() == ScalarType::UInt32);
    const Tensor *weights = matrix_of(a[6], "weights", PyExc_AssertionError);
    if (weights == nullptr) return nullptr;
    A2A_REQUIRE(has_shape(*weights, tokens, op->topk));
    A2A_REQUIRE(weights->stride(1) == 1);
    A2A_REQUIRE(weights->scalar_type() == ScalarType::Float);
    // Dynamic bound on the number of tokens (p2p_all_to_all.py:404-411).
    d.bound_m = nullptr;
    if (a[7] != Py_None) {
        const Tensor *bound = tensor_of(a[7], "bound_m");
        if (bound == nullptr) return nullptr;
        A2A_REQUIRE(bound->numel() == 1);
        A2A_REQUIRE(bound->scalar_type() == ScalarType::Int);
        d.bound_m = static_cast<const int32_t *>(bound->data_ptr());
    }

    d.num_tokens = (uint64_t)tokens;
    d.x_ptr = x->data_ptr();
    d.x_stride = row_bytes(*x);
    d.x_scale_ptr = x_scale != nullptr ? static_cast<const float *>(x_scale->data_ptr()) : nullptr;
    d.x_scale_stride_elem = x_scale != nullptr ? (uint64_t)x_scale->stride(1) : 0;
    d.x_scale_stride_token = x_scale != nullptr ? (uint64_t)x_scale->stride(0) : 0;
    d.indices = static_cast<const int32_t *>(indices->data_ptr());
    d.indices_stride = (uint64_t)indices->stride(0);
    d.weights = static_cast<const float *>(weights->data_ptr());
    d.weights_stride = (uint64_t)weights->stride(0);
    d.out_num_tokens = static_cast<int32_t *>(out_n->data_ptr());
    d.out_x = out_x->data_ptr();
    d.out_x_stride = row_bytes(*out_x);
    d.out_x_rows = (uint64_t)out_x->size(0);
    d.out_x_scale = out_scale != nullptr ? static_cast<float *>(out_scale->data_ptr()) : nullptr;
    d.out_x_scale_stride_elem = out_scale != nullptr ? (uint64_t)out_scale->stride(1) : 0;
    d.out_x_scale_stride_token = out_scale != nullptr ? (uint64_t)out_scale->stride(0) : 0;

    if (do_send && do_recv) {
        PyObject *const given[kKept] = {a[0], a[1], a[2], a[3], a[4], a[5], a[6], a[7]};
        const int last = post(*c->dispatch, "dispatch", op->rank, op->world, d, (uint32_t)quantize, given);
        if (last < 0) return nullptr;
        if (last == 0) Py_RETURN_NONE;
        Taken<a2a_dispatch_args> step(*c->dispatch, op->world);
        if (!step.alike) {
            PyErr_SetString(PyExc_RuntimeError, "every rank must call dispatch() in the same mode");
            return nullptr;
        }
        if (!require_open(c)) return nullptr;
        a2a_ctx *const ctx = c->ctx;
        void *const stream = current_stream(op);
        int rc;
        Py_BEGIN_ALLOW_THREADS
        rc = a2a_dispatch(ctx, step.args, (uint32_t)quantize, stream);
        Py_END_ALLOW_THREADS
        if (rc != 0) return raise_last_error(ctx, "a2a_dispatch", rc);
        Py_RETURN_NONE;
    }

    if (!require_open(c)) return nullptr;
    a2a_ctx *const ctx = c->ctx;
    void *const stream = current_stream(op);
    int rc;
    Py_BEGIN_ALLOW_THREADS
    if (do_send) {
        rc = a2a_dispatch_send(ctx, op->rank, d.num_tokens, d.x_ptr, d.x_stride, (uint32_t)quantize, d.x_scale_ptr,
                               d.x_scale_stride_elem, d.x_scale_stride_token, d.indices, d.indices_stride, d.weights,
                               d.weights_stride, d.bound_m, stream);
    } else {
        rc = a2a_dispatch_recv(ctx, op->rank, d.out_num_tokens, d.out_x, d.out_x_stride, d.out_x_rows, d.out_x_scale,
                               d.out_x_scale_stride_elem, d.out_x_scale_stride_token, stream);
    }
    Py_END_ALLOW_THREADS
    if (rc != 0) return raise_last_error(ctx, do_send ? "a2a_dispatch_send" : "a2a_dispatch_recv", rc);
    Py_RETURN_NONE;
}

// combine(out_tokens, indices, weights, expert_y, bound_m=None, do_send=True, do_recv=True, accumulate=False)
PyObject *combine(Operator *op, PyObject *const *args, Py_ssize_t n, PyObject *keywords) {
    PyObject *a[kMostParameters] = {nullptr, nullptr, nullptr, nullptr, Py_None, Py_True, Py_True, Py_False};
    if (!take_arguments(combine_parameters, args, n, keywords, a)) return nullptr;
    const int do_send = PyObject_IsTrue(a[5]), do_recv = PyObject_IsTrue(a[6]), accumulate = PyObject_IsTrue(a[7]);
    if (do_send < 0 || do_recv < 0 || accumulate < 0) return nullptr;
    A2A_REQUIRE(do_send || do_recv);
    A2A_REQUIRE(!accumulate || op->dp_size == 1);
    Context *const c = op->context;

    // p2p_all_to_all.py:463-484
    const Tensor *out = matrix_of(a[0], "out_tokens", PyExc_AssertionError);
    const Tensor *indices = out != nullptr ? matrix_of(a[1], "indices", PyExc_ValueError) : nullptr;
    const Tensor *weights = indices != nullptr ? matrix_of(a[2], "weights", PyExc_AssertionError) : nullptr;
    const Tensor *y = weights != nullptr ? matrix_of(a[3], "expert_y", PyExc_ValueError) : nullptr;
    if (y == nullptr) return nullptr;
    const int64_t tokens = indices->size(0);
    A2A_REQUIRE(has_shape(*out, tokens, op->hidden_dim));
    A2A_REQUIRE(out->scalar_type() == op->out_dtype);
    A2A_REQUIRE(out->stride(1) == 1);
    A2A_REQUIRE(has_shape(*indices, tokens, op->topk));
    A2A_REQUIRE(indices->stride(1) == 1);
    A2A_REQUIRE(indices->scalar_type() == ScalarType::UInt32);
    A2A_REQUIRE(has_shape(*weights, tokens, op->topk));
    A2A_REQUIRE(weights->stride(1) == 1);
    A2A_REQUIRE(weights->scalar_type() == ScalarType::Float);
    A2A_REQUIRE(y->size(1) == op->hidden_dim);
    A2A_REQUIRE(y->stride(1) == 1);

    a2a_combine_args d;
    d.bound_m = nullptr;
    if (a[4] != Py_None) {
        const Tensor *bound = tensor_of(a[4], "bound_m");
        if (bound == nullptr) return nullptr;
        A2A_REQUIRE(bound->numel() == 1);
        A2A_REQUIRE(bound->scalar_type() == ScalarType::Int);
        d.bound_m = static_cast<const int32_t *>(bound->data_ptr());
    }
    d.expert_y = y->data_ptr();
    d.expert_y_stride = row_bytes(*y);
    d.expert_y_rows = (uint64_t)y->size(0);
    d.num_tokens = (uint64_t)tokens;
    d.out_tokens = out->data_ptr();
    d.out_tokens_stride = (uint64_t)out->stride(0);
    d.indices = static_cast<const int32_t *>(indices->data_ptr());
    d.indices_stride = (uint64_t)indices->stride(0);
    d.weights = static_cast<const float *>(weights->data_ptr());
    d.weights_stride = (uint64_t)weights->stride(0);
    const ScalarType y_dtype = y->scalar_type();
    const int y_tag = tag_of(y_dtype);

    if (do_send && do_recv) {
        PyObject *const given[kKept] = {a[0], a[1], a[2], a[3], a[4], nullptr, nullptr, nullptr};
        const int last = post(*c->combine, "combine", op->rank, op->world, d, (uint32_t)y_dtype << 1 | (uint32_t)accumulate,
                              given);
        if (last < 0) return nullptr;
        if (last == 0) Py_RETURN_NONE;
        Taken<a2a_combine_args> step(*c->combine, op->world);
        if (!step.alike) {
            PyErr_SetString(PyExc_RuntimeError,
                            "every rank must call combine() with the same expert_y dtype and accumulate");
            return nullptr;
        }
        if (!require_open(c)) return nullptr;
        if (y_tag < 0) return PyErr_Format(PyExc_RuntimeError, "unsupported expert_y dtype %s", c10::toString(y_dtype));
        a2a_ctx *const ctx = c->ctx;
        void *const stream = current_stream(op);
        int rc;
        Py_BEGIN_ALLOW_THREADS
        rc = a2a_combine(ctx, step.args, (uint32_t)y_tag, (uint32_t)accumulate, stream);
        Py_END_ALLOW_THREADS
        if (rc != 0) return raise_last_error(ctx, "a2a_combine", rc);
        Py_RETURN_NONE;
    }

    if (y->element_size() != (int64_t)c10::elementSize(op->out_dtype)) {
        // combine-send copies staging rows sized for out_dtype without knowing the type of expert_y (as the
        // reference's does, a2a_combine_send.cu:261); narrower rows would be over-read
        return PyErr_Format(PyExc_RuntimeError,
                            "split combine needs expert_y (%s) with the element size of out_dtype (%s); "
                            "call combine() with do_send and do_recv for mixed types",
                            c10::toString(y_dtype), c10::toString(op->out_dtype));
    }
    if (!require_open(c)) return nullptr;
    if (do_recv && y_tag < 0)
        return PyErr_Format(PyExc_RuntimeError, "unsupported expert_y dtype %s", c10::toString(y_dtype));
    a2a_ctx *const ctx = c->ctx;
    void *const stream = current_stream(op);
    int rc;
    Py_BEGIN_ALLOW_THREADS
    if (do_send) {
        rc = a2a_combine_send(ctx, op->rank, d.expert_y, d.expert_y_stride, d.expert_y_rows, stream);
    } else {
        rc = a2a_combine_recv(ctx, op->rank, d.num_tokens, d.expert_y_rows, (uint32_t)y_tag, d.out_tokens,
                              d.out_tokens_stride, d.indices, d.indices_stride, d.weights, d.weights_stride, d.bound_m,
                              (uint32_t)accumulate, stream);
    }
    Py_END_ALLOW_THREADS
    if (rc != 0) return raise_last_error(ctx, do_send ? "a2a_combine_send" : "a2a_combine_recv", rc);
    Py_RETURN_NONE;
}

// A torch call (data_ptr of a tensor without storage, say) may throw: no C++ exception enters the interpreter.
template <PyObject *(*CALL)(Operator *, PyObject *const *, Py_ssize_t, PyObject *)>
PyObject *guarded(PyObject *self, PyObject *const *args, Py_ssize_t n, PyObject *keywords) {
    try {
        return CALL(reinterpret_cast<Operator *>(self), args, n, keywords);
    } catch (python_error &e) {
        e.restore();
    } catch (const std::exception &e) {
        PyErr_SetString(PyExc_RuntimeError, e.what());
    }
    return nullptr;
}

PyMethodDef operator_methods[] = {
    {"dispatch", reinterpret_cast<PyCFunction>(reinterpret_cast<void *>(guarded<dispatch>)), METH_FASTCALL | METH_KEYWORDS,
     nullptr},
    {"combine", reinterpret_cast<PyCFunction>(reinterpret_cast<void *>(guarded<combine>)), METH_FASTCALL | METH_KEYWORDS,
     nullptr},
    {nullptr, nullptr, 0, nullptr},
};

PyTypeObject OperatorType = {PyVarObject_HEAD_INIT(nullptr, 0)};

// ---------------------------------------------------------------------------
// call_without_a_frame(function): calls of the Python function `f(self, ...)`, which hands its arguments to the method of the
// same name of `self._operator`, run that method without a Python frame in between.  The function stays the object it is, and
// with it whatever is looked up, bound, inspected or kept; only the way the interpreter enters it changes.  What is called
// is decided at the call: without a native operator in `_operator` (after `destroy()`, say) the function itself runs, and so
// it does under a profiler or debugger and once somebody has given it other code or defaults.
// ---------------------------------------------------------------------------
PyObject *operator_attribute;   // "_operator"

struct Frameless {
    const Parameters &parameters;
    PyObject *(*call)(PyObject *, PyObject *const *, Py_ssize_t, PyObject *);
    vectorcallfunc enter;           // how the interpreter enters the function itself
    PyObject *code, *defaults;      // the function's, when it was given the other entry
};

Frameless frameless_dispatch = {dispatch_parameters, guarded<dispatch>, nullptr, nullptr, nullptr};
Frameless frameless_combine = {combine_parameters, guarded<combine>, nullptr, nullptr, nullptr};

template <Frameless &F>
PyObject *enter_operator(PyObject *function, PyObject *const *args, size_t n, PyObject *keywords) {
    const PyThreadState *const thread = PyThreadState_Get();
    if (PyVectorcall_NARGS(n) > 0 && thread->c_tracefunc == nullptr && thread->c_profilefunc == nullptr &&
        PyFunction_GET_CODE(function) == F.code && PyFunction_GET_DEFAULTS(function) == F.defaults) {
        PyObject *const op = PyObject_GetAttr(args[0], operator_attribute);
        if (op == nullptr) {
            if (!PyErr_ExceptionMatches(PyExc_AttributeError)) return nullptr;
            PyErr_Clear();
        } else if (Py_TYPE(op) == &OperatorType) {
            PyObject *const result = F.call(op, args + 1, PyVectorcall_NARGS(n) - 1, keywords);
            Py_DECREF(op);
            return result;
        }
        Py_XDECREF(op);
    }
    return F.enter(function, args, n, keywords);
}

template <Frameless &F>
void set_entry(PyFunctionObject *f) {
    if (f->vectorcall == enter_operator<F>) return;
    F.enter = f->vectorcall;
    Py_XINCREF(f->func_code);
    Py_XINCREF(f->func_defaults);
    Py_XSETREF(F.code, f->func_code);
    Py_XSETREF(F.defaults, f->func_defaults);
    f->vectorcall = enter_operator<F>;
}

PyObject *call_without_a_frame(PyObject *, PyObject *function) {
    if (!PyFunction_Check(function)) return PyErr_Format(PyExc_TypeError, "a Python function is expected");
    PyFunctionObject *const f = reinterpret_cast<PyFunctionObject *>(function);
    if (PyUnicode_CompareWithASCIIString(f->func_name, frameless_dispatch.parameters.call) == 0) {
        set_entry<frameless_dispatch>(f);
    } else if (PyUnicode_CompareWithASCIIString(f->func_name, frameless_combine.parameters.call) == 0) {
        set_entry<frameless_combine>(f);
    } else {
        return PyErr_Format(PyExc_ValueError, "no call of the operator has the name %U", f->func_name);
    }
    Py_RETURN_NONE;
}

PyMethodDef module_methods[] = {
    {"call_without_a_frame", call_without_a_frame, METH_O, nullptr},
    {nullptr, nullptr, 0, nullptr},
};

PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_a2a_torch", nullptr, -1, module_methods, nullptr, nullptr, nullptr, nullptr};

bool add_type(PyObject *module, PyTypeObject &type, const char *name, const char *short_name, size_t size, newfunc make,
              destructor drop, PyMethodDef *methods) {
    type.tp_name = name;
    type.tp_basicsize = (Py_ssize_t)size;
    type.tp_flags = Py_TPFLAGS_DEFAULT;
    type.tp_new = make;
    type.tp_dealloc = drop;
    type.tp_methods = methods;
    if (PyType_Ready(&type) < 0) return false;
    Py_INCREF(&type);
    return PyModule_AddObject(module, short_name, reinterpret_cast<PyObject *>(&type)) == 0;
}

}  // namespace

PyMODINIT_FUNC PyInit__a2a_torch(void) {
    PyObject *m = PyModule_Create(&module_def);
    if (m == nullptr) return nullptr;
    operator_attribute = PyUnicode_InternFromString("_operator");
    if (operator_attribute == nullptr || !intern_names(dispatch_parameters) || !intern_names(combine_parameters)) {
        Py_DECREF(m);
        return nullptr;
    }
    if (!add_type(m, ContextType, "_a2a_torch.Context", "Context", sizeof(Context), context_new, context_dealloc,
                  context_methods) ||
        !add_type(m, OperatorType, "_a2a_torch.Operator", "Operator", sizeof(Operator), operator_new, operator_dealloc,
                  operator_methods)) {
        Py_DECREF(m);
        return nullptr;
    }
    return m;
}
