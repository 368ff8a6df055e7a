// Python entry points of the short launches (a layer at a few images), where
// the host's time per call is what a caller waits for: the checks, the output
// tensor, the stream and the C ABI call in one native function.  Every
// function returns None for a call it does not take (other layouts, dtypes,
// tensor types, large launches, any error): the caller then runs its Python
// path, which takes or refuses the call.  One layer at one row, host time per
// call: 10.4 us through ctypes, 4.5 us here.
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstring>

#include "../../include/rpfq.h"

namespace {

// Launches of at least this many operations are left to the Python path,
// which chooses between more kernels; the host is not what bounds them.
constexpr double kMostOps = 1.5e9;

// The C ABI as the library that _native.load() opened exports it: this module
// links none, so that another build of the library (RPFQ_LIBRARY) serves these
// calls too.  Null until bind().
#define RPFQ_HOST_CALLS(X)                                                                              \
    X(rpfq_wide_linear_kernel) X(rpfq_row_scales) X(rpfq_wide_linear_scaled)                            \
    X(rpfq_layer_norm_wide_linear_fusable) X(rpfq_layer_norm_wide_linear) X(rpfq_act_quant_wide_linear) \
    X(rpfq_attention)
struct Api {
#define X(f) decltype(&::f) f;
    RPFQ_HOST_CALLS(X)
#undef X
} api = {};
constexpr const char* kCalls[] = {
#define X(f) #f,
    RPFQ_HOST_CALLS(X)
#undef X
};
constexpr Py_ssize_t kNumCalls = sizeof(kCalls) / sizeof(kCalls[0]);
static_assert(sizeof(Api) == kNumCalls * sizeof(void*), "one pointer per call");

int dtype_code(at::ScalarType t) {
    switch (t) {
        case at::kFloat: return RPFQ_F32;
        case at::kHalf: return RPFQ_F16;
        case at::kBFloat16: return RPFQ_BF16;
        default: return -1;
    }
}

// A plain strided device tensor (no subclass), or NULL.
const at::Tensor* plain(PyObject* o) {
    if (!THPVariable_CheckExact(o)) return nullptr;
    const at::Tensor& t = THPVariable_Unpack(o);
    return t.is_cuda() && t.layout() == at::kStrided && !t.is_neg() && !t.is_conj() ? &t : nullptr;
}

bool rows16(const at::Tensor& t) {
    return t.is_contiguous() && reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0;
}

// None or a contiguous float32 device vector of n values.
bool vec(PyObject* o, int64_t n, const float** p) {
    *p = nullptr;
    if (o == Py_None) return true;
    const at::Tensor* t = plain(o);
    if (!t || t->scalar_type() != at::kFloat || !t->is_contiguous() || t->numel() != n) return false;
    *p = t->const_data_ptr<float>();
    return true;
}

// The numbers of a call: false where o is not one (the Python error goes).
bool number(PyObject* o, int64_t* v) {
    *v = PyLong_AsLongLong(o);
    if (!PyErr_Occurred()) return true;
    PyErr_Clear();
    return false;
}
bool number(PyObject* o, float* v) {
    *v = (float)PyFloat_AsDouble(o);
    if (!PyErr_Occurred()) return true;
    PyErr_Clear();
    return false;
}

struct Call {
    const rpfq_wide_desc* d;
    const at::Tensor *blob, *x;
    const void* res = nullptr;
    int64_t m = 0;
    int xdt = 0, ydt = 0;
    at::ScalarType yt{};
    c10::SmallVector<int64_t, 6> shape;
    at::Tensor y;
    void* stream = nullptr;
    // the output and the stream, once it is known that the call is taken here
    void take() {
        y = at::empty(shape, x->options().dtype(yt));
        stream = c10::hip::getCurrentHIPStream(x->device().index()).stream();
    }
};

// The operands the layer calls share: desc address, blob, x, residual, the
// output's dtype (None: x's).
bool layer(PyObject* desc, PyObject* blob, PyObject* x, PyObject* residual, PyObject* out_dtype, Call& c) {
    int64_t at;
    if (!api.rpfq_attention || !number(desc, &at)) return false;
    c.d = reinterpret_cast<const rpfq_wide_desc*>(at);
    c.blob = plain(blob);
    c.x = plain(x);
    if (!c.d || !c.blob || !c.x || c.x->dim() < 1) return false;
    const int64_t in = 2 * c.d->k_complex, out = 2 * c.d->n_complex;
    if (c.x->size(-1) != in || !rows16(*c.x)) return false;
    c.m = c.x->numel() / in;
    c.yt = c.x->scalar_type();
    if (out_dtype != Py_None) {
        if (!THPDtype_Check(out_dtype)) return false;
        c.yt = reinterpret_cast<THPDtype*>(out_dtype)->scalar_type;
    }
    c.xdt = dtype_code(c.x->scalar_type());
    c.ydt = dtype_code(c.yt);
    if (c.m < 1 || c.xdt < 0 || c.ydt < 0 || 2.0 * (double)c.m * (double)in * (double)out >= kMostOps) return false;
    c.shape.assign(c.x->sizes().begin(), c.x->sizes().end());
    c.shape.back() = out;
    if (residual != Py_None) {
        const at::Tensor* r = plain(residual);
        if (!r || r->scalar_type() != c.yt || r->sizes() != at::IntArrayRef(c.shape) || !rows16(*r)) return false;
        c.res = r->data_ptr();
    }
    return true;
}

// Allocations and launches run without the interpreter lock, as through torch
// and ctypes: one that waits for memory or for room in the queue must not hold
// up the other threads, or a host function in that queue that needs the lock.
struct Unlocked {
    PyThreadState* state = PyEval_SaveThread();
    Unlocked() = default;
    Unlocked(const Unlocked&) = delete;
    ~Unlocked() { PyEval_RestoreThread(state); }
};

PyObject* done(int rc, const at::Tensor& y) {
    if (rc != RPFQ_OK) Py_RETURN_NONE;
    return THPVariable_Wrap(y);
}

// linear(desc, blob, x, bias, residual, out_dtype, flags, guard): guard bit 0:
// float32 / bf16 rows get their prescales, bit 1: rows that go to the DMA
// kernel as prescaled fp16 (many rows) are left to the Python path.
PyObject* linear(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    Call c;
    const float* bias;
    int64_t flags, guard;
    if (n != 8 || !number(a[6], &flags) || !number(a[7], &guard) || !layer(a[0], a[1], a[2], a[4], a[5], c) ||
        !vec(a[3], 2 * c.d->n_complex, &bias))
        Py_RETURN_NONE;
    const int64_t in = 2 * c.d->k_complex;
    const bool scaled = c.xdt != RPFQ_F16 && (guard & 1);
    int kernel = -1;
    if (scaled && (guard & 2) && in <= 4096 &&
        api.rpfq_wide_linear_kernel(c.d, c.m, RPFQ_F16, c.ydt, (int)flags, &kernel) == RPFQ_OK && kernel == RPFQ_KERNEL_DMA)
        Py_RETURN_NONE;
    int rc = RPFQ_OK;
    {
        Unlocked u;
        c.take();
        at::Tensor s;
        if (scaled) {
            s = at::empty({c.m}, c.x->options().dtype(at::kFloat));
            rc = api.rpfq_row_scales(c.x->data_ptr(), c.xdt, c.m, in, s.data_ptr<float>(), c.stream);
        }
        if (rc == RPFQ_OK)
            rc = api.rpfq_wide_linear_scaled(c.d, c.blob->data_ptr(), c.blob->nbytes(), c.x->data_ptr(), c.xdt, c.m,
                                             scaled ? s.const_data_ptr<float>() : nullptr, bias, c.res, c.y.data_ptr(),
                                             c.ydt, (int)flags, c.stream);
    }
    return done(rc, c.y);
    END_HANDLE_TH_ERRORS
}

// layer_norm_linear(desc, blob, x, ln_weight, ln_bias, eps, bias, out_dtype, flags)
// where the launch takes the LayerNorm in its prologue.
PyObject* layer_norm_linear(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    Call c;
    const float *w, *b, *bias;
    float eps;
    int64_t flags;
    int fusable = 0;
    if (n != 9 || !number(a[5], &eps) || !number(a[8], &flags) || !layer(a[0], a[1], a[2], Py_None, a[7], c)) Py_RETURN_NONE;
    const int64_t in = 2 * c.d->k_complex;
    if (!vec(a[3], in, &w) || !vec(a[4], in, &b) || !vec(a[6], 2 * c.d->n_complex, &bias) ||
        api.rpfq_layer_norm_wide_linear_fusable(c.d, c.m, c.xdt, c.ydt, &fusable) != RPFQ_OK || !fusable)
        Py_RETURN_NONE;
    int rc;
    {
        Unlocked u;
        c.take();
        rc = api.rpfq_layer_norm_wide_linear(c.d, c.blob->data_ptr(), c.blob->nbytes(), c.x->data_ptr(), c.xdt, c.m, w, b,
                                             eps, bias, c.y.data_ptr(), c.ydt, (int)flags, c.stream);
    }
    return done(rc, c.y);
    END_HANDLE_TH_ERRORS
}

// act_quant_linear(desc, blob, x, bits, bias, residual, out_dtype, flags) where
// the launch takes the act quant in its prologue.
PyObject* act_quant_linear(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    Call c;
    const float* bias;
    int64_t bits, flags;
    int fusable = 0;
    if (n != 8 || !number(a[3], &bits) || !number(a[7], &flags) || !layer(a[0], a[1], a[2], a[5], a[6], c) || !vec(a[4], 2 * c.d->n_complex, &bias) ||
        api.rpfq_layer_norm_wide_linear_fusable(c.d, c.m, c.xdt, c.ydt, &fusable) != RPFQ_OK || !fusable)
        Py_RETURN_NONE;
    int rc;
    {
        Unlocked u;
        c.take();
        rc = api.rpfq_act_quant_wide_linear(c.d, c.blob->data_ptr(), c.blob->nbytes(), c.x->data_ptr(), c.xdt, c.m,
                                            (int)bits, 0, nullptr, nullptr, 0.0f, bias, c.res, c.y.data_ptr(), c.ydt,
                                            (int)flags, c.stream);
    }
    return done(rc, c.y);
    END_HANDLE_TH_ERRORS
}

// attention(qkv, heads, scale)
PyObject* attention(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    int64_t h;
    float scale;
    if (n != 3 || !number(a[1], &h) || !number(a[2], &scale)) Py_RETURN_NONE;
    const at::Tensor* q = api.rpfq_attention ? plain(a[0]) : nullptr;
    if (!q || q->dim() != 3 || h < 1 || q->size(2) != 192 * h ||
        q->numel() == 0 || !rows16(*q))
        Py_RETURN_NONE;
    at::Tensor y;
    int rc;
    {
        Unlocked u;
        y = at::empty({q->size(0), q->size(1), 64 * h}, q->options());
        rc = api.rpfq_attention(q->data_ptr(), dtype_code(q->scalar_type()), q->size(0), q->size(1), h, 64, scale,
                                y.data_ptr(), c10::hip::getCurrentHIPStream(q->device().index()).stream());
    }
    return done(rc, y);
    END_HANDLE_TH_ERRORS
}

// bind(addresses): the functions named by CALLS, in that order.
PyObject* bind(PyObject*, PyObject* addresses) {
    Api next;
    if (!PyTuple_Check(addresses) || PyTuple_GET_SIZE(addresses) != kNumCalls) {
        PyErr_SetString(PyExc_ValueError, "bind takes a tuple of one address per name in CALLS");
        return nullptr;
    }
    for (Py_ssize_t i = 0; i < kNumCalls; ++i) {
        void* f = PyLong_AsVoidPtr(PyTuple_GET_ITEM(addresses, i));
        if (!f) {
            if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "bind: a null address");
            return nullptr;
        }
        std::memcpy(reinterpret_cast<char*>(&next) + i * sizeof(void*), &f, sizeof(f));
    }
    api = next;
    Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"bind", bind, METH_O, nullptr},
    {"linear", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(linear)), METH_FASTCALL, nullptr},
    {"layer_norm_linear", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(layer_norm_linear)), METH_FASTCALL, nullptr},
    {"act_quant_linear", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(act_quant_linear)), METH_FASTCALL, nullptr},
    {"attention", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(attention)), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host(void) {
    PyObject* m = PyModule_Create(&module);
    PyObject* names = m ? PyTuple_New(kNumCalls) : nullptr;
    for (Py_ssize_t i = 0; names && i < kNumCalls; ++i) {
        PyObject* name = PyUnicode_FromString(kCalls[i]);
        if (!name) Py_CLEAR(names);
        else PyTuple_SET_ITEM(names, i, name);
    }
    if (!names || PyModule_AddObject(m, "CALLS", names) < 0) {
        Py_XDECREF(names);
        Py_XDECREF(m);
        return nullptr;
    }
    return m;
}
