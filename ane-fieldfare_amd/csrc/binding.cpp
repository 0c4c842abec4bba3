// The Python binding's per-call work in native code: the compute methods of fieldfare_moe.Context and Matrix hand their
// tensors here, and one call reads their pointers and strides, takes torch's current stream, allocates what the method
// returns and calls the C ABI. A decode step makes four such calls for five launches of 31 us on the GPU; through ctypes
// (argument objects, a stream object and a Python-level torch.empty per output) a call took 7 to 11 us of host time, more than
// its kernels, and here it takes 1 to 2 us plus the launches. Nothing of the path's math is here; the C ABI does not
// know of it (Swift and C++ hosts call that directly).
#include <Python.h>

#include <ATen/core/Tensor.h>
#include <ATen/hip/EmptyTensor.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <dlfcn.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <algorithm>
#include <cstdlib>
#include <stdexcept>

#include "../../include/fieldfare_moe.h"

namespace {

PyObject *g_error = nullptr;      // fieldfare_moe.FieldfareError(code, message)

struct PythonError {};            // a Python exception is set

// the entry points, looked up in the library the package has loaded (bind)
#define FFMOE_CALLS(X)                                                                                                                 \
    X(ffmoe_matrix_gemv) X(ffmoe_matrix_rows) X(ffmoe_matrix_greedy) X(ffmoe_matrix_greedy_conf) X(ffmoe_router) X(ffmoe_verify)        \
    X(ffmoe_route_verify) X(ffmoe_route_verify_shared) X(ffmoe_verify_partials) X(ffmoe_reduce_token_major) X(ffmoe_prefill)           \
    X(ffmoe_dense_ffn) X(ffmoe_prefill_pairs) X(ffmoe_post_attn_setup) X(ffmoe_layer_tail) X(ffmoe_layer_tail_routed)                  \
    X(ffmoe_layer_tail_routed_shared) X(ffmoe_layer_tail_norms) X(ffmoe_rmsnorm) X(ffmoe_gelu_mul) X(ffmoe_argmax_rows)                 \
    X(ffmoe_sample_rows) X(ffmoe_gemv_int4_listed) X(ffmoe_gemv_int4)
#define FFMOE_POINTER(name) decltype(&::name) name = nullptr;
struct Calls {
    FFMOE_CALLS(FFMOE_POINTER)
} g_calls;
#undef FFMOE_POINTER

// While one lives the interpreter lock is given up: a launch that waits for room in its queue, a library's first use, an
// allocation that waits for the device do not hold up the program's other threads. Python objects are read before, results
// wrapped after.
struct Unlocked {
    PyThreadState *state = PyEval_SaveThread();
    ~Unlocked() { PyEval_RestoreThread(state); }
};

template <typename... P, typename... A>
int call(int (*f)(P...), A... args) {
    const Unlocked unlocked;
    return f(args...);
}

void check(int code, char *&err) {      // by reference: the call that fills it is the first argument
    if (code == FFMOE_OK) return;
    PyObject *args = Py_BuildValue("(is)", code, err ? err : "(no message)");
    free(err);
    if (args) {
        PyObject *e = PyObject_CallObject(g_error, args);
        Py_DECREF(args);
        if (e) {
            PyErr_SetObject(g_error, e);
            Py_DECREF(e);
        }
    }
    throw PythonError{};
}

// ---- arguments ---------------------------------------------------------------------------------------------------
const at::Tensor &tensor(PyObject *o) {
    if (!THPVariable_Check(o)) {
        PyErr_Format(PyExc_TypeError, "a tensor is wanted, got %.100s", Py_TYPE(o)->tp_name);
        throw PythonError{};
    }
    return THPVariable_Unpack(o);
}
template <typename T>
T *pointer(const at::Tensor &t) { return static_cast<T *>(t.data_ptr()); }
template <typename T>
T *pointer(PyObject *o) { return o == Py_None ? nullptr : pointer<T>(tensor(o)); }      // None: a null pointer
template <typename T>
T *handle(PyObject *o) {
    if (o == Py_None) return nullptr;
    void *p = PyLong_AsVoidPtr(o);
    if (!p && PyErr_Occurred()) throw PythonError{};
    return static_cast<T *>(p);
}
uint32_t u32(PyObject *o) {
    const unsigned long v = PyLong_AsUnsignedLongMask(o);
    if (v == (unsigned long)-1 && PyErr_Occurred()) throw PythonError{};
    return (uint32_t)v;
}
// the address `offset` bytes from a tensor's first; the offset has the pointer's width (a buffer that holds a model's weights is
// larger than 4 GiB) and, as in Python's own address arithmetic, is an int that may be negative
const uint8_t *address(PyObject *o, PyObject *offset) {
    if (!PyLong_Check(offset)) {
        PyErr_Format(PyExc_TypeError, "a byte offset is an int, got %.100s", Py_TYPE(offset)->tp_name);
        throw PythonError{};
    }
    const long long bytes = PyLong_AsLongLong(offset);
    if (bytes == -1 && PyErr_Occurred()) throw PythonError{};
    return reinterpret_cast<const uint8_t *>(reinterpret_cast<uintptr_t>(pointer<uint8_t>(o)) + (uintptr_t)bytes);
}
float f32(PyObject *o) {
    const double v = PyFloat_AsDouble(o);
    if (v == -1.0 && PyErr_Occurred()) throw PythonError{};
    return (float)v;
}
bool truth(PyObject *o) {
    const int v = PyObject_IsTrue(o);
    if (v < 0) throw PythonError{};
    return v != 0;
}
at::ScalarType dtype(PyObject *o) {
    if (!THPDtype_Check(o)) {
        PyErr_SetString(PyExc_TypeError, "a torch dtype is wanted");
        throw PythonError{};
    }
    return reinterpret_cast<THPDtype *>(o)->scalar_type;
}
void rank(const at::Tensor &t, int64_t dims) {      // where the shape is taken apart whole
    if (t.dim() == dims) return;
    PyErr_Format(PyExc_ValueError, "a tensor of %lld dimensions is wanted, got %lld", (long long)dims, (long long)t.dim());
    throw PythonError{};
}
uint32_t dim_of(const at::Tensor &t, int64_t dim) { return (uint32_t)t.size(dim); }
// row stride in elements; a single-row tensor may report any stride for its size-1 dimension
uint32_t row_stride(const at::Tensor &t) { return (uint32_t)(t.size(0) > 1 ? t.stride(0) : std::max(t.stride(0), t.size(1))); }
void *stream() { return c10::hip::getCurrentHIPStreamMasqueradingAsCUDA().stream(); }

at::Tensor allocate(const at::Tensor &like, at::ScalarType type, at::IntArrayRef sizes) {
    const at::Device device = like.device();
    const Unlocked unlocked;
    return at::detail::empty_cuda(sizes, type, device, std::nullopt);
}
at::Tensor fresh(const at::Tensor &like, at::ScalarType type, int64_t a) { return allocate(like, type, at::IntArrayRef{a}); }
at::Tensor fresh(const at::Tensor &like, at::ScalarType type, int64_t a, int64_t b) { return allocate(like, type, {a, b}); }
PyObject *wrap(at::Tensor t) { return THPVariable_Wrap(std::move(t)); }
// the caller's output tensor, or a new one
struct Out {
    at::Tensor t;
    PyObject *given = nullptr;
    PyObject *result() {
        if (given) {
            Py_INCREF(given);
            return given;
        }
        return wrap(std::move(t));
    }
};
Out output(PyObject *given, const at::Tensor &like, at::ScalarType type, int64_t a, int64_t b) {
    if (given != Py_None) return Out{tensor(given), given};
    return Out{fresh(like, type, a, b)};
}
PyObject *tuple(std::initializer_list<PyObject *> items) {
    PyObject *t = PyTuple_New((Py_ssize_t)items.size());
    Py_ssize_t i = 0;
    for (PyObject *o : items) PyTuple_SET_ITEM(t, i++, o);
    return t;
}

// ---- methods: args[0] is the context's (the matrix's) handle -------------------------------------------------------
using Args = PyObject *const *;

PyObject *matrix_gemv(Args a) {      // handle, x, m, act, f32_out, out
    const at::Tensor &x = tensor(a[1]);
    const bool wide = truth(a[4]);
    Out y = output(a[5], x, wide ? at::kFloat : dtype(a[3]), x.size(0), (int64_t)u32(a[2]));
    char *err = nullptr;
    check(call(g_calls.ffmoe_matrix_gemv, handle<ffmoe_matrix>(a[0]), stream(), pointer<uint16_t>(x), row_stride(x), dim_of(x, 0), y.t.data_ptr(),
               row_stride(y.t), wide, &err), err);
    return y.result();
}

PyObject *matrix_rows(Args a) {      // handle, ids (a tensor), out_scale, out (a tensor)
    const at::Tensor &ids = tensor(a[1]), &y = tensor(a[3]);
    char *err = nullptr;
    check(call(g_calls.ffmoe_matrix_rows, handle<ffmoe_matrix>(a[0]), stream(), pointer<uint32_t>(ids), dim_of(ids, 0), 0u, f32(a[2]),
               pointer<uint16_t>(y), row_stride(y), &err), err);
    Py_INCREF(a[3]);
    return a[3];
}

PyObject *matrix_greedy(Args a) {    // handle, x
    const at::Tensor &x = tensor(a[1]);
    at::Tensor out = fresh(x, at::kInt, x.size(0));
    char *err = nullptr;
    check(call(g_calls.ffmoe_matrix_greedy, handle<ffmoe_matrix>(a[0]), stream(), pointer<uint16_t>(x), row_stride(x), dim_of(x, 0),
               pointer<uint32_t>(out), &err), err);
    return wrap(out);
}

PyObject *matrix_greedy_conf(Args a) {      // handle, x, softcap
    const at::Tensor &x = tensor(a[1]);
    at::Tensor out = fresh(x, at::kInt, x.size(0)), conf = fresh(x, at::kFloat, x.size(0));
    char *err = nullptr;
    check(call(g_calls.ffmoe_matrix_greedy_conf, handle<ffmoe_matrix>(a[0]), stream(), pointer<uint16_t>(x), row_stride(x), dim_of(x, 0), f32(a[2]),
               pointer<uint32_t>(out), pointer<float>(conf), &err), err);
    return tuple({wrap(out), wrap(conf)});
}

PyObject *router(Args a) {           // handle, layer, router_x, act, top_k, n_experts, want_logits
    const at::Tensor &x = tensor(a[2]);
    const at::ScalarType act = dtype(a[3]);
    if (x.scalar_type() != act || !x.is_cuda() || x.stride(1) != 1) {
        PyErr_SetString(PyExc_AssertionError, "router rows: a CUDA tensor of the context's activation type with unit column stride");
        throw PythonError{};
    }
    const int64_t t = x.size(0), k = u32(a[4]);
    const bool want = truth(a[6]);
    at::Tensor idx = fresh(x, at::kInt, t, k), w = fresh(x, act, t, k), logits;
    if (want) logits = fresh(x, at::kFloat, t, (int64_t)u32(a[5]));
    char *err = nullptr;
    check(call(g_calls.ffmoe_router, handle<ffmoe_ctx>(a[0]), stream(), u32(a[1]), pointer<uint16_t>(x), row_stride(x), (uint32_t)t,
               pointer<uint32_t>(idx), pointer<uint16_t>(w), want ? pointer<float>(logits) : nullptr, &err), err);
    if (want) return tuple({wrap(idx), wrap(w), wrap(logits)});
    return tuple({wrap(idx), wrap(w)});
}

PyObject *verify(Args a) {           // handle, layer, x, idx, w, residual, out, act, d
    const at::Tensor &x = tensor(a[2]);
    Out y = output(a[6], x, dtype(a[7]), x.size(0), (int64_t)u32(a[8]));
    char *err = nullptr;
    check(call(g_calls.ffmoe_verify, handle<ffmoe_ctx>(a[0]), stream(), u32(a[1]), pointer<uint16_t>(x), row_stride(x), dim_of(x, 0),
               pointer<uint32_t>(a[3]), pointer<uint16_t>(a[4]), pointer<uint16_t>(a[5]), pointer<uint16_t>(y.t), &err), err);
    return y.result();
}

PyObject *route_verify(Args a) {     // handle, layer, router_x, x, residual, out, combine, act, top_k, d
    const at::Tensor &rx = tensor(a[2]), &x = tensor(a[3]);
    const int64_t t = x.size(0), k = u32(a[8]);
    const at::ScalarType act = dtype(a[7]);
    const bool combine = truth(a[6]);
    Out y;
    if (combine) y = output(a[5], x, act, t, (int64_t)u32(a[9]));
    at::Tensor idx = fresh(x, at::kInt, t, k), w = fresh(x, act, t, k);
    char *err = nullptr;
    check(call(g_calls.ffmoe_route_verify, handle<ffmoe_ctx>(a[0]), stream(), u32(a[1]), pointer<uint16_t>(rx), row_stride(rx), pointer<uint16_t>(x),
               row_stride(x), (uint32_t)t, pointer<uint16_t>(a[4]), combine ? pointer<uint16_t>(y.t) : nullptr,
               pointer<uint32_t>(idx), pointer<uint16_t>(w), &err), err);
    if (!combine) Py_INCREF(Py_None);
    return tuple({combine ? y.result() : Py_None, wrap(idx), wrap(w)});
}

PyObject *route_verify_shared(Args a) {     // handle, shared handle, layer, shared_layer, router_x, x, shared_x, act, top_k
    const at::Tensor &rx = tensor(a[4]), &x = tensor(a[5]), &sx = tensor(a[6]);
    const int64_t t = x.size(0), k = u32(a[8]);
    at::Tensor idx = fresh(x, at::kInt, t, k), w = fresh(x, dtype(a[7]), t, k);
    char *err = nullptr;
    check(call(g_calls.ffmoe_route_verify_shared, handle<ffmoe_ctx>(a[0]), handle<ffmoe_ctx>(a[1]), stream(), u32(a[2]), u32(a[3]),
               pointer<uint16_t>(rx), row_stride(rx), pointer<uint16_t>(x), row_stride(x), pointer<uint16_t>(sx),
               row_stride(sx), (uint32_t)t, pointer<uint32_t>(idx), pointer<uint16_t>(w), &err), err);
    return tuple({wrap(idx), wrap(w)});
}

PyObject *verify_partials(Args a) {  // handle, layer, x, idx, w, partials (a tensor)
    const at::Tensor &x = tensor(a[2]);
    char *err = nullptr;
    check(call(g_calls.ffmoe_verify_partials, handle<ffmoe_ctx>(a[0]), stream(), u32(a[1]), pointer<uint16_t>(x), row_stride(x), dim_of(x, 0),
               pointer<uint32_t>(a[3]), pointer<uint16_t>(a[4]), pointer<uint16_t>(a[5]), &err), err);
    Py_INCREF(a[5]);
    return a[5];
}

PyObject *reduce_token_major(Args a) {      // handle, partials, weights, act
    const at::Tensor &p = tensor(a[1]);
    rank(p, 3);
    at::Tensor h2 = fresh(p, dtype(a[3]), p.size(0), p.size(2));
    char *err = nullptr;
    check(call(g_calls.ffmoe_reduce_token_major, handle<ffmoe_ctx>(a[0]), stream(), pointer<uint16_t>(p), pointer<uint16_t>(a[2]),
               pointer<uint16_t>(h2), dim_of(p, 0), dim_of(p, 1), dim_of(p, 2), &err), err);
    return wrap(h2);
}

PyObject *prefill(Args a) {          // handle, layer, x, idx, w, out, act, d
    const at::Tensor &x = tensor(a[2]);
    Out y = output(a[5], x, dtype(a[6]), x.size(0), (int64_t)u32(a[7]));
    char *err = nullptr;
    check(call(g_calls.ffmoe_prefill, handle<ffmoe_ctx>(a[0]), stream(), u32(a[1]), pointer<uint16_t>(x), row_stride(x), dim_of(x, 0),
               pointer<uint32_t>(a[3]), pointer<uint16_t>(a[4]), pointer<uint16_t>(y.t), &err), err);
    return y.result();
}

PyObject *dense_ffn(Args a) {        // handle, layer, x, out, act, d
    const at::Tensor &x = tensor(a[2]);
    Out y = output(a[3], x, dtype(a[4]), x.size(0), (int64_t)u32(a[5]));
    char *err = nullptr;
    check(call(g_calls.ffmoe_dense_ffn, handle<ffmoe_ctx>(a[0]), stream(), u32(a[1]), pointer<uint16_t>(x), row_stride(x), dim_of(x, 0),
               pointer<uint16_t>(y.t), &err), err);
    return y.result();
}

PyObject *prefill_pairs(Args a) {    // handle, layer, x, sorted_pairs, t, partials (a tensor)
    const at::Tensor &x = tensor(a[2]), &pairs = tensor(a[3]);
    char *err = nullptr;
    check(call(g_calls.ffmoe_prefill_pairs, handle<ffmoe_ctx>(a[0]), stream(), u32(a[1]), pointer<uint16_t>(x), row_stride(x),
               pointer<ffmoe_pair>(pairs), dim_of(pairs, 0), u32(a[4]), pointer<uint16_t>(a[5]), &err), err);
    Py_INCREF(a[5]);
    return a[5];
}

PyObject *post_attn_setup(Args a) {  // handle, hidden, attn, w_post_attn, w_pre_ffn, w_pre_ffn2, eps, d, out, act
    const at::Tensor &hidden = tensor(a[1]), &attn = tensor(a[2]);
    const int64_t t = hidden.size(0), d = u32(a[7]);
    at::Tensor outs[3];
    PyObject *given = a[8] == Py_None ? nullptr : a[8];
    for (int i = 0; i < 3; ++i) {
        if (given) {
            // given[i]: three tensors in a sequence, or one of [3, t, >= d]
            PyObject *index = PyLong_FromLong(i), *item = index ? PyObject_GetItem(given, index) : nullptr;
            Py_XDECREF(index);
            if (!item) throw PythonError{};
            outs[i] = THPVariable_Check(item) ? THPVariable_Unpack(item) : at::Tensor();
            if (!THPVariable_Check(item)) PyErr_SetString(PyExc_TypeError, "out holds three tensors");
            Py_DECREF(item);
            if (PyErr_Occurred()) throw PythonError{};
        } else {
            outs[i] = fresh(hidden, dtype(a[9]), t, d);
        }
    }
    char *err = nullptr;
    check(call(g_calls.ffmoe_post_attn_setup, handle<ffmoe_ctx>(a[0]), stream(), pointer<uint16_t>(hidden), row_stride(hidden), pointer<uint16_t>(attn),
               row_stride(attn), pointer<uint16_t>(outs[0]), row_stride(outs[0]), pointer<uint16_t>(outs[1]),
               row_stride(outs[1]), pointer<uint16_t>(outs[2]), row_stride(outs[2]), pointer<uint16_t>(a[3]),
               pointer<uint16_t>(a[4]), pointer<uint16_t>(a[5]), (uint32_t)t, (uint32_t)d, f32(a[6]), &err), err);
    if (given) {
        Py_INCREF(given);
        return given;
    }
    return tuple({wrap(outs[0]), wrap(outs[1]), wrap(outs[2])});
}

PyObject *layer_tail(Args a) {       // handle, h2, h1, hidden, w_postffn2, w_postffn, layer_scalar, eps, d
    const at::Tensor &h2 = tensor(a[1]), &h1 = tensor(a[2]), &hidden = tensor(a[3]);
    char *err = nullptr;
    check(call(g_calls.ffmoe_layer_tail, handle<ffmoe_ctx>(a[0]), stream(), pointer<uint16_t>(h2), row_stride(h2), pointer<uint16_t>(h1), row_stride(h1),
               pointer<uint16_t>(hidden), row_stride(hidden), pointer<uint16_t>(a[4]), pointer<uint16_t>(a[5]),
               dim_of(hidden, 0), u32(a[8]), f32(a[7]), f32(a[6]), &err), err);
    Py_INCREF(a[3]);
    return a[3];
}

PyObject *layer_tail_routed(Args a) {       // handle, route_w, h1, hidden, w_postffn2, w_postffn, layer_scalar, eps
    const at::Tensor &h1 = tensor(a[2]), &hidden = tensor(a[3]);
    char *err = nullptr;
    check(call(g_calls.ffmoe_layer_tail_routed, handle<ffmoe_ctx>(a[0]), stream(), pointer<uint16_t>(a[1]), pointer<uint16_t>(h1), row_stride(h1),
               pointer<uint16_t>(hidden), row_stride(hidden), pointer<uint16_t>(a[4]), pointer<uint16_t>(a[5]),
               dim_of(hidden, 0), f32(a[7]), f32(a[6]), &err), err);
    Py_INCREF(a[3]);
    return a[3];
}

PyObject *layer_tail_routed_shared(Args a) {       // handle, shared handle, route_w, hidden, w_postffn2, w_postffn, layer_scalar, eps
    const at::Tensor &hidden = tensor(a[3]);
    char *err = nullptr;
    check(call(g_calls.ffmoe_layer_tail_routed_shared, handle<ffmoe_ctx>(a[0]), handle<ffmoe_ctx>(a[1]), stream(), pointer<uint16_t>(a[2]),
               pointer<uint16_t>(hidden), row_stride(hidden), pointer<uint16_t>(a[4]),
               pointer<uint16_t>(a[5]), dim_of(hidden, 0), f32(a[7]), f32(a[6]), &err), err);
    Py_INCREF(a[3]);
    return a[3];
}

PyObject *layer_tail_norms(Args a) { // handle, h2, h1, hidden, w_postffn1, w_postffn2, w_postffn, layer_scalar, w_next, eps, d, act
    const at::Tensor &h2 = tensor(a[1]), &h1 = tensor(a[2]), &hidden = tensor(a[3]);
    const uint32_t d = u32(a[10]);
    at::Tensor normed;
    if (a[8] != Py_None) normed = fresh(hidden, dtype(a[11]), hidden.size(0), d);
    char *err = nullptr;
    check(call(g_calls.ffmoe_layer_tail_norms, handle<ffmoe_ctx>(a[0]), stream(), pointer<uint16_t>(h2), row_stride(h2), pointer<uint16_t>(h1),
               row_stride(h1), pointer<uint16_t>(hidden), row_stride(hidden), pointer<uint16_t>(a[4]),
               pointer<uint16_t>(a[5]), pointer<uint16_t>(a[6]), pointer<uint16_t>(a[8]),
               normed.defined() ? pointer<uint16_t>(normed) : nullptr, d, dim_of(hidden, 0), d, f32(a[9]), f32(a[7]),
               &err), err);
    if (normed.defined()) return wrap(normed);
    Py_RETURN_NONE;
}

PyObject *rmsnorm(Args a) {          // handle, x, w, eps, d, out, act
    const at::Tensor &x = tensor(a[1]);
    const uint32_t d = u32(a[4]);
    Out y = output(a[5], x, dtype(a[6]), x.size(0), d);
    char *err = nullptr;
    check(call(g_calls.ffmoe_rmsnorm, handle<ffmoe_ctx>(a[0]), stream(), pointer<uint16_t>(x), row_stride(x), pointer<uint16_t>(a[2]),
               pointer<uint16_t>(y.t), row_stride(y.t), dim_of(x, 0), d, f32(a[3]), &err), err);
    return y.result();
}

PyObject *gelu_mul(Args a) {         // handle, gate, up, out
    const at::Tensor &gate = tensor(a[1]), &up = tensor(a[2]);
    rank(gate, 2);
    Out y = output(a[3], gate, gate.scalar_type(), gate.size(0), gate.size(1));
    char *err = nullptr;
    check(call(g_calls.ffmoe_gelu_mul, handle<ffmoe_ctx>(a[0]), stream(), pointer<uint16_t>(gate), row_stride(gate), pointer<uint16_t>(up),
               row_stride(up), pointer<uint16_t>(y.t), row_stride(y.t), dim_of(gate, 0), dim_of(gate, 1), &err), err);
    return y.result();
}

PyObject *argmax_rows(Args a) {      // handle, logits, count (0: the whole row), softcap, want_conf
    const at::Tensor &l = tensor(a[1]);
    const uint32_t count = u32(a[2]);
    const bool want = truth(a[4]);
    at::Tensor out = fresh(l, at::kInt, l.size(0)), conf;
    if (want) conf = fresh(l, at::kFloat, l.size(0));
    char *err = nullptr;
    check(call(g_calls.ffmoe_argmax_rows, handle<ffmoe_ctx>(a[0]), stream(), pointer<float>(l), row_stride(l), dim_of(l, 0), count ? count : dim_of(l, 1),
               f32(a[3]), pointer<uint32_t>(out), want ? pointer<float>(conf) : nullptr, &err), err);
    if (want) return tuple({wrap(out), wrap(conf)});
    return wrap(out);
}

PyObject *sample_rows(Args a) {      // handle, logits, temperature, softcap, seed, key_base, top_k, top_p, ids, key_offset, count (0: the whole row)
    const at::Tensor &l = tensor(a[1]);
    const uint32_t count = u32(a[10]);
    const unsigned long long seed = PyLong_AsUnsignedLongLongMask(a[4]);
    if (seed == (unsigned long long)-1 && PyErr_Occurred()) throw PythonError{};
    const ffmoe_sampling rule{f32(a[2]), f32(a[7]), u32(a[6]), u32(a[5]), f32(a[3]), (uint64_t)seed};
    at::Tensor out = fresh(l, at::kInt, l.size(0)), prob = fresh(l, at::kFloat, l.size(0));
    char *err = nullptr;
    check(call(g_calls.ffmoe_sample_rows, handle<ffmoe_ctx>(a[0]), stream(), pointer<float>(l), row_stride(l), dim_of(l, 0), count ? count : dim_of(l, 1),
               pointer<uint32_t>(a[8]), &rule, pointer<uint32_t>(a[9]), pointer<uint32_t>(out), pointer<float>(prob),
               &err), err);
    return tuple({wrap(out), wrap(prob)});
}

PyObject *gemv_int4_listed(Args a) { // handle, W, S, B, ids, x
    const at::Tensor &s = tensor(a[2]), &ids = tensor(a[4]), &x = tensor(a[5]);
    const uint32_t m = dim_of(ids, 0), n = dim_of(s, 1) * FFMOE_GROUP;
    at::Tensor y = fresh(x, at::kFloat, x.size(0), m);
    char *err = nullptr;
    check(call(g_calls.ffmoe_gemv_int4_listed, handle<ffmoe_ctx>(a[0]), stream(), pointer<uint8_t>(a[1]), pointer<uint16_t>(s), pointer<uint16_t>(a[3]),
               pointer<uint32_t>(ids), pointer<uint16_t>(x), pointer<float>(y), m, n, dim_of(x, 0), row_stride(x), m,
               &err), err);
    return wrap(y);
}

PyObject *gemv_int4(Args a) {        // handle, W, S, B, x, f32_out, w_byte_offset, act
    const at::Tensor &s = tensor(a[2]), &x = tensor(a[4]);
    const uint32_t m = dim_of(s, 0), n = dim_of(s, 1) * FFMOE_GROUP;
    const bool wide = truth(a[5]);
    const uint8_t *w = address(a[1], a[6]);
    at::Tensor y = fresh(x, wide ? at::kFloat : dtype(a[7]), x.size(0), m);
    char *err = nullptr;
    check(call(g_calls.ffmoe_gemv_int4, handle<ffmoe_ctx>(a[0]), stream(), w, pointer<uint16_t>(s),
               pointer<uint16_t>(a[3]), pointer<uint16_t>(x), y.data_ptr(), m, n, dim_of(x, 0), row_stride(x), m, wide, &err), err);
    return wrap(y);
}

template <PyObject *(*F)(Args), int N>
PyObject *method(PyObject *, PyObject *const *args, Py_ssize_t n) {
    if (n != N) {
        PyErr_Format(PyExc_TypeError, "%d arguments are wanted, got %zd", N, n);
        return nullptr;
    }
    // what torch throws arrives as from torch's own calls (torch.OutOfMemoryError from an allocation, IndexError, ...)
    HANDLE_TH_ERRORS
    try {
        return F(args);
    } catch (const PythonError &) {
        return nullptr;
    }
    END_HANDLE_TH_ERRORS
}

// bind(path of the loaded library, exception class)
PyObject *bind(PyObject *, PyObject *args) {
    const char *path;
    PyObject *error;
    if (!PyArg_ParseTuple(args, "sO", &path, &error)) return nullptr;
    void *lib = dlopen(path, RTLD_NOW | RTLD_NOLOAD);
    if (!lib) {
        PyErr_Format(PyExc_RuntimeError, "%s is not loaded", path);
        return nullptr;
    }
#define FFMOE_LOOK_UP(name)                                                       \
    g_calls.name = reinterpret_cast<decltype(&::name)>(dlsym(lib, #name));        \
    if (!g_calls.name) {                                                          \
        PyErr_SetString(PyExc_RuntimeError, "the library has no " #name);         \
        return nullptr;                                                           \
    }
    FFMOE_CALLS(FFMOE_LOOK_UP)
#undef FFMOE_LOOK_UP
    Py_INCREF(error);
    Py_XSETREF(g_error, error);
    Py_RETURN_NONE;
}

#define FFMOE_METHOD(name, n) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(method<name, n>)), METH_FASTCALL, nullptr}
PyMethodDef g_methods[] = {
    {"bind", bind, METH_VARARGS, nullptr},
    FFMOE_METHOD(matrix_gemv, 6),
    FFMOE_METHOD(matrix_rows, 4),
    FFMOE_METHOD(matrix_greedy, 2),
    FFMOE_METHOD(matrix_greedy_conf, 3),
    FFMOE_METHOD(router, 7),
    FFMOE_METHOD(verify, 9),
    FFMOE_METHOD(route_verify, 10),
    FFMOE_METHOD(route_verify_shared, 9),
    FFMOE_METHOD(verify_partials, 6),
    FFMOE_METHOD(reduce_token_major, 4),
    FFMOE_METHOD(prefill, 8),
    FFMOE_METHOD(dense_ffn, 6),
    FFMOE_METHOD(prefill_pairs, 6),
    FFMOE_METHOD(post_attn_setup, 10),
    FFMOE_METHOD(layer_tail, 9),
    FFMOE_METHOD(layer_tail_routed, 8),
    FFMOE_METHOD(layer_tail_routed_shared, 8),
    FFMOE_METHOD(layer_tail_norms, 12),
    FFMOE_METHOD(rmsnorm, 7),
    FFMOE_METHOD(gelu_mul, 4),
    FFMOE_METHOD(argmax_rows, 5),
    FFMOE_METHOD(sample_rows, 11),
    FFMOE_METHOD(gemv_int4_listed, 6),
    FFMOE_METHOD(gemv_int4, 8),
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "ffmoe_binding", "Per-call work of fieldfare_moe in native code.", -1, g_methods, nullptr,
                        nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_ffmoe_binding(void) { return PyModule_Create(&g_module); }
