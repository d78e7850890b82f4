// The host side of one call, natively: what rumus_amd/ops.py does around an entry point of librumus_hip.so (checks,
// the result tensor, the current stream, the call itself), for the entry points that a serving loop makes thousands of
// times a second.
//
// Why: at few rows the host is what bounds a call.  1 x 4096 x 4096 takes 3.7 us on the GPU and took 12.2 us of Python
// per call on the host (2.8 of them torch.cuda.current_stream(), 1.7 torch.empty, 1.5 the checks of five tensors, about
// 1 reading shapes, 0.8 ctypes), so the GPU stood idle for two thirds of the time.
//
// Every function here takes only the plain case: ordinary torch tensors on the device, contiguous, of the right type and
// large enough, no mode or transform around the call.  For anything else it returns None before anything is queued, and
// the general path in ops.py then gives its answer or raises its error.  A failed call raises RumusError, as it does there.
#include <Python.h>

#include <ATen/core/TensorBody.h>
#include <ATen/ops/empty.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <ATen/PythonTorchFunctionTLS.h>

#include "rumus_hip.h"

namespace {

using at::ScalarType;
using at::Tensor;

// A tensor that the general path would use as it is: exact type (a subclass may have its own idea of every operation), on
// the device, no wrapper of a transform, strided memory of its own.
bool ordinary(PyObject* o, ScalarType dtype, const Tensor*& out) {
    if (!THPVariable_CheckExact(o)) return false;
    const Tensor& t = THPVariable_Unpack(o);
    static const c10::DispatchKeySet wrappers({c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper,
                                               c10::DispatchKey::Functionalize, c10::DispatchKey::Python});
    if (!t.defined() || !t.is_cuda() || t.layout() != c10::kStrided || !t.has_storage() || t.scalar_type() != dtype ||
        t.key_set().has_any(wrappers))
        return false;
    out = &t;
    return true;
}

bool plain(PyObject* o, ScalarType dtype, const Tensor*& out) { return ordinary(o, dtype, out) && out->is_contiguous(); }

// None, or a plain tensor of at least `least` elements
bool plain_or_none(PyObject* o, ScalarType dtype, uint64_t least, const Tensor*& out) {
    out = nullptr;
    return o == Py_None || (plain(o, dtype, out) && (uint64_t)out->numel() >= least);
}

bool small(PyObject* o, uint32_t& out) {          // a whole number that a size argument holds
    if (!PyLong_CheckExact(o)) return false;
    const long long v = PyLong_AsLongLong(o);
    if (v == -1 && PyErr_Occurred()) {
        PyErr_Clear();
        return false;
    }
    if (v < 0 || v > 0x7fffffff) return false;
    out = (uint32_t)v;
    return true;
}

bool fits(int64_t v) { return v > 0 && v <= 0x7fffffff; }

// a mode that wants to see torch's own calls (torch.empty among them) keeps the general path
bool watched() { return at::impl::torch_function_mode_enabled() || c10::impl::TorchDispatchModeTLS::any_modes_set(); }

void* stream() { return c10::hip::getCurrentHIPStream().stream(); }      // of the current device

template <typename T>
T* ptr(const Tensor* t) { return t ? static_cast<T*>(t->data_ptr()) : nullptr; }

Tensor make(at::IntArrayRef shape, const Tensor& like, ScalarType dtype) {
    return at::empty(shape, at::TensorOptions().dtype(dtype).device(like.device()));
}

PyObject* result(int rc, const Tensor& y) {
    if (rc == 0) return THPVariable_Wrap(y);
    PyObject* module = PyImport_ImportModule("rumus_amd._lib");
    PyObject* type = module ? PyObject_GetAttrString(module, "RumusError") : nullptr;
    PyObject* value = type ? PyObject_CallFunction(type, "is", rc, rumus_hip_last_error()) : nullptr;
    if (value) PyErr_SetObject(type, value);
    Py_XDECREF(value);
    Py_XDECREF(type);
    Py_XDECREF(module);
    return nullptr;
}

// `f` with the interpreter free for other threads, as ctypes leaves it
template <typename F>
int unlocked(F f) {
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = f();
    Py_END_ALLOW_THREADS
    return rc;
}

// packed, scales and zero-points as large as the geometry needs
struct W4 {
    const Tensor *packed, *scales, *zp;
    uint32_t k, n, padded_k, group, groups;
    bool read(PyObject* p, PyObject* s, PyObject* z, PyObject* k_, PyObject* g_) {
        if (!plain(p, at::kInt, packed) || !plain(s, at::kFloat, scales) || !plain(z, at::kFloat, zp) || !small(k_, k) ||
            !small(g_, group) || k == 0 || group == 0 || packed->dim() != 2 || !fits(packed->size(1)))
            return false;
        n = (uint32_t)packed->size(1);
        const uint64_t count = ((uint64_t)k + group - 1) / group, padded = count * group;
        if (padded > 0x7fffffff) return false;
        groups = (uint32_t)count;
        padded_k = (uint32_t)padded;
        const uint64_t rows = padded / 8 ? padded / 8 : 1;
        return (uint64_t)packed->numel() >= rows * n && (uint64_t)scales->numel() >= count * n && (uint64_t)zp->numel() >= count * n;
    }
};

// the caller's result tensor if it is the right one, a new one for None
bool output(PyObject* o, int64_t rows, int64_t cols, ScalarType dtype, const Tensor& like, Tensor& y) {
    if (o == Py_None) {
        y = make({rows, cols}, like, dtype);
        return true;
    }
    const Tensor* t;
    if (!plain(o, dtype, t) || t->dim() != 2 || t->size(0) != rows || t->size(1) != cols) return false;
    y = *t;
    return true;
}

#define RUMUS_PLAIN(cond) \
    do {                  \
        if (!(cond)) Py_RETURN_NONE; \
    } while (0)

// (x, packed, scales, zero_points, bias, index, k, group_size, out)
template <typename Act, ScalarType DTYPE, auto FN>
PyObject* w4_matmul(PyObject*, PyObject* const* a, Py_ssize_t count) {
    HANDLE_TH_ERRORS
    const Tensor *x, *bias, *index;
    W4 w;
    RUMUS_PLAIN(count == 9 && !watched() && plain(a[0], DTYPE, x) && w.read(a[1], a[2], a[3], a[6], a[7]));
    RUMUS_PLAIN(x->dim() == 2 && x->size(1) == w.k && fits(x->size(0)));
    RUMUS_PLAIN(plain_or_none(a[4], at::kFloat, w.n, bias) && plain_or_none(a[5], at::kInt, w.k, index));
    const uint32_t m = (uint32_t)x->size(0);
    Tensor y;
    RUMUS_PLAIN(output(a[8], m, w.n, DTYPE, *x, y));
    void* s = stream();
    const int rc = unlocked([&] {
        return FN(ptr<const Act>(x), ptr<const uint32_t>(w.packed), ptr<const float>(w.scales), ptr<const float>(w.zp),
                  ptr<const float>(bias), ptr<const int32_t>(index), ptr<Act>(&y), m, w.k, w.n, w.padded_k, w.group, w.groups, s);
    });
    return result(rc, y);
    END_HANDLE_TH_ERRORS
}

// (a, packed, scales, zero_points, k, group_size, out)
PyObject* w4_matmul_t(PyObject*, PyObject* const* a, Py_ssize_t count) {
    HANDLE_TH_ERRORS
    const Tensor* g;
    W4 w;
    RUMUS_PLAIN(count == 7 && !watched() && plain(a[0], at::kFloat, g) && w.read(a[1], a[2], a[3], a[4], a[5]));
    RUMUS_PLAIN(g->dim() == 2 && g->size(1) == w.n && fits(g->size(0)));
    const uint32_t m = (uint32_t)g->size(0);
    Tensor y;
    RUMUS_PLAIN(output(a[6], m, w.k, at::kFloat, *g, y));
    void* s = stream();
    const int rc = unlocked([&] {
        return rumus_hip_qmatmul_int4_t(ptr<const float>(g), ptr<const uint32_t>(w.packed), ptr<const float>(w.scales),
                                        ptr<const float>(w.zp), ptr<float>(&y), m, w.k, w.n, w.padded_k, w.group, w.groups, s);
    });
    return result(rc, y);
    END_HANDLE_TH_ERRORS
}

// (x, packed, scales, zero_points, k, group_size, norm_weight, eps, swiglu, bias, residual, out)
PyObject* w4_decode_block(PyObject*, PyObject* const* a, Py_ssize_t count) {
    HANDLE_TH_ERRORS
    const Tensor *x, *norm, *bias, *residual;
    W4 w;
    RUMUS_PLAIN(count == 12 && !watched() && plain(a[0], at::kFloat, x) && w.read(a[1], a[2], a[3], a[4], a[5]));
    RUMUS_PLAIN(PyFloat_CheckExact(a[7]) && PyBool_Check(a[8]));
    const bool swiglu = a[8] == Py_True;
    RUMUS_PLAIN(x->dim() == 2 && x->size(1) == (swiglu ? 2 : 1) * (int64_t)w.k && fits(x->size(0)));
    const uint32_t m = (uint32_t)x->size(0);
    RUMUS_PLAIN(plain_or_none(a[6], at::kFloat, w.k, norm) && plain_or_none(a[9], at::kFloat, w.n, bias) &&
                plain_or_none(a[10], at::kFloat, 0, residual));
    RUMUS_PLAIN(!residual || (residual->dim() == 2 && residual->size(0) == m && residual->size(1) == w.n));
    Tensor y;
    RUMUS_PLAIN(output(a[11], m, w.n, at::kFloat, *x, y));
    void* s = stream();
    const float eps = (float)PyFloat_AS_DOUBLE(a[7]);
    const int rc = unlocked([&] {
        return rumus_hip_qmatmul_int4_decode_block(ptr<const float>(x), ptr<const float>(norm), eps, swiglu ? 1 : 0,
                                                   ptr<const uint32_t>(w.packed), ptr<const float>(w.scales), ptr<const float>(w.zp),
                                                   ptr<const float>(bias), ptr<const float>(residual), ptr<float>(&y), m, w.k, w.n,
                                                   w.padded_k, w.group, w.groups, s);
    });
    return result(rc, y);
    END_HANDLE_TH_ERRORS
}

// (a, words, k, n, block_size)
template <typename Act, ScalarType DTYPE, auto FN>
PyObject* q8_matmul(PyObject*, PyObject* const* a, Py_ssize_t count) {
    HANDLE_TH_ERRORS
    const Tensor *x, *words;
    uint32_t k, n, block;
    RUMUS_PLAIN(count == 5 && !watched() && plain(a[0], DTYPE, x) && plain(a[1], at::kInt, words) && small(a[2], k) &&
                small(a[3], n) && small(a[4], block) && k && n && block);
    RUMUS_PLAIN(x->dim() == 2 && x->size(1) == k && fits(x->size(0)));
    // whole blocks per column, a header word in front of each (ops.matmul_q8 has the reason)
    RUMUS_PLAIN((uint64_t)words->numel() >= (uint64_t)n * ((k + (uint64_t)block - 1) / block) * (((uint64_t)block + 7) / 4));
    const uint32_t m = (uint32_t)x->size(0);
    const Tensor y = make({m, n}, *x, DTYPE);
    void* s = stream();
    const int rc = unlocked([&] { return FN(ptr<const Act>(x), ptr<const uint32_t>(words), ptr<Act>(&y), m, k, n, block, s); });
    return result(rc, y);
    END_HANDLE_TH_ERRORS
}

// (x, wq, sw, bias): rows quantized, then the integer product
PyObject* int8_linear(PyObject*, PyObject* const* a, Py_ssize_t count) {
    HANDLE_TH_ERRORS
    const Tensor *x, *wq, *sw, *bias;
    RUMUS_PLAIN(count == 4 && !watched() && plain(a[0], at::kFloat, x) && plain(a[1], at::kChar, wq) && plain(a[2], at::kFloat, sw));
    RUMUS_PLAIN(x->dim() == 2 && wq->dim() == 2 && x->size(1) == wq->size(1) && fits(x->size(0)) && fits(x->size(1)) && fits(wq->size(0)));
    const uint32_t m = (uint32_t)x->size(0), k = (uint32_t)x->size(1), n = (uint32_t)wq->size(0);
    RUMUS_PLAIN((uint64_t)sw->numel() >= n && plain_or_none(a[3], at::kFloat, n, bias));
    const uint64_t bytes = rumus_hip_i8_linear_scratch_size(m, k, n);
    Tensor scratch;                                            // quantized rows, where they go through memory
    if (bytes) scratch = make({(int64_t)bytes}, *x, at::kChar);
    const Tensor y = make({m, n}, *x, at::kFloat);
    void* const mem = bytes ? ptr<void>(&scratch) : nullptr;
    void* s = stream();
    const int rc = unlocked([&] {
        return rumus_hip_i8_linear(ptr<const float>(x), ptr<const int8_t>(wq), ptr<const float>(sw), ptr<const float>(bias), mem, ptr<float>(&y), m,
                                   k, n, s);
    });
    return result(rc, y);
    END_HANDLE_TH_ERRORS
}

// (q, k_new, v_new, k_cache, v_cache, pos): [B, 1, H, d] and [B, T, H, d], any strides with the last dim contiguous
PyObject* attention_decode_append(PyObject*, PyObject* const* a, Py_ssize_t count) {
    HANDLE_TH_ERRORS
    const Tensor* t[6];
    uint32_t pos;
    RUMUS_PLAIN(count == 6 && !watched() && small(a[5], pos));
    for (int i = 0; i < 5; i++) RUMUS_PLAIN(ordinary(a[i], at::kFloat, t[i]) && t[i]->dim() == 4 && t[i]->stride(3) == 1);
    const int64_t b = t[0]->size(0), h = t[0]->size(2), d = t[0]->size(3), positions = t[3]->size(1);
    RUMUS_PLAIN(fits(b) && fits(h) && fits(d) && fits(positions));
    for (int i = 0; i < 5; i++)
        RUMUS_PLAIN(t[i]->size(0) == b && t[i]->size(1) == (i < 3 ? 1 : positions) && t[i]->size(2) == h && t[i]->size(3) == d);
    const Tensor o = make({b, 1, h, d}, *t[0], at::kFloat);
    t[5] = &o;
    uint64_t strides[18];
    for (int i = 0; i < 6; i++) {
        strides[3 * i] = (uint64_t)t[i]->stride(0);
        strides[3 * i + 1] = (uint64_t)t[i]->stride(2);
        strides[3 * i + 2] = (uint64_t)t[i]->stride(1);
    }
    void* s = stream();
    const int rc = unlocked([&] {
        return rumus_hip_attention_decode_append(ptr<const float>(t[0]), ptr<const float>(t[1]), ptr<const float>(t[2]), ptr<float>(t[3]),
                                                 ptr<float>(t[4]), ptr<float>(&o), (uint32_t)b, (uint32_t)h, (uint32_t)d, pos,
                                                 (uint32_t)positions, strides, s);
    });
    return result(rc, o);
    END_HANDLE_TH_ERRORS
}

template <typename F>
PyCFunction fast(F f) { return reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(f)); }

PyMethodDef methods[] = {
    {"rumus_hip_qmatmul_int4", fast(w4_matmul<float, at::kFloat, rumus_hip_qmatmul_int4>), METH_FASTCALL, nullptr},
    {"rumus_hip_qmatmul_int4_f16", fast(w4_matmul<uint16_t, at::kHalf, rumus_hip_qmatmul_int4_f16>), METH_FASTCALL, nullptr},
    {"rumus_hip_qmatmul_int4_perm", fast(w4_matmul<float, at::kFloat, rumus_hip_qmatmul_int4_perm>), METH_FASTCALL, nullptr},
    {"rumus_hip_qmatmul_int4_perm_static", fast(w4_matmul<float, at::kFloat, rumus_hip_qmatmul_int4_perm_static>), METH_FASTCALL, nullptr},
    {"rumus_hip_qmatmul_int4_decode", fast(w4_matmul<float, at::kFloat, rumus_hip_qmatmul_int4_decode>), METH_FASTCALL, nullptr},
    {"qmatmul_int4_t", fast(w4_matmul_t), METH_FASTCALL, nullptr},
    {"qmatmul_int4_decode_block", fast(w4_decode_block), METH_FASTCALL, nullptr},
    {"matmul_q8", fast(q8_matmul<float, at::kFloat, rumus_hip_matmul_q8>), METH_FASTCALL, nullptr},
    {"matmul_q8_f16", fast(q8_matmul<uint16_t, at::kHalf, rumus_hip_matmul_q8_f16>), METH_FASTCALL, nullptr},
    {"int8_linear", fast(int8_linear), METH_FASTCALL, nullptr},
    {"attention_decode_append", fast(attention_decode_append), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr},
};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host_calls", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host_calls() { return PyModule_Create(&module); }
