// Python binding of the per-call entry points over torch tensors (module
// candle_moe._fast): reads the tensors' descriptors through torch's C++
// interface and calls the C ABI.
//
// The ctypes route (candle_moe/__init__.py) spends 1.3 us of Python per tensor
// and call, half of the host's time for a call of three launches, and small
// batches are bound by the host. A call, ctypes / here (repeated eager calls):
// topk-softmax [64, 128] 9.7 / 3.8 us, [32768, 128] 9.7 / 7.4 (the kernel);
// router_topk T=1 H=2048 E=128 11.0 / 8.4; FusedMoE.forward T=2 H=128 I=64 E=8
// 20.4 / 13.0, its host time alone 20.2 / 11.1. This module serves the calls whose tensors are plain, strided and
// of the dtypes, shapes and devices the entry points take; for anything else it
// returns None and the ctypes route runs instead, which raises what it always
// raised. It keeps nothing between calls: no descriptor, pointer or output.
#include <Python.h>

#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/version.h>

#include <exception>

#include "../../include/candle_moe.h"

namespace {

// C ABI entry points of the loaded library, given by address (bind()).
decltype(&candle_moe_apply_topk_softmax_inplace) g_topk;
decltype(&candle_moe_fused_moe_forward) g_forward;
decltype(&candle_moe_router_topk) g_router;
decltype(&candle_moe_fused_moe_fp8) g_fp8;
decltype(&candle_moe_fused_moe_packed) g_packed;
PyObject* g_raw_stream;  // torch._C._cuda_getCurrentRawStream

int dtype_code(at::ScalarType t) {
    switch (t) {
        case at::kHalf: return CM_DT_F16;
        case at::kBFloat16: return CM_DT_BF16;
        case at::kFloat: return CM_DT_F32;
        // int32 index tensors are taken as u32 bit patterns
        case at::kInt:
        case at::kUInt32: return CM_DT_U32;
        case at::kLong: return CM_DT_I64;
        case at::kDouble: return CM_DT_F64;
        case at::kByte: return CM_DT_U8;
        default: return -1;
    }
}

// The tensor of a Python object, or null where the general route has to see it
// (subclasses, tensors without storage or strides).
const at::Tensor* plain(PyObject* o) {
    if (!THPVariable_CheckExact(o)) return nullptr;
    const at::Tensor& t = THPVariable_Unpack(o);
    if (!t.defined() || t.layout() != at::kStrided || !t.has_storage() || t.unsafeGetTensorImpl()->is_python_dispatch())
        return nullptr;
    return &t;
}

bool describe(PyObject* o, cm_tensor_t& d) {
    const at::Tensor* t = plain(o);
    if (!t || t->dim() > CM_MAX_RANK) return false;
    d = cm_tensor_t{};
    d.dtype = dtype_code(t->scalar_type());
    if (d.dtype < 0) return false;
    d.rank = (int32_t)t->dim();
    for (int i = 0; i < d.rank; ++i) {
        d.dims[i] = t->size(i);
        d.strides[i] = t->stride(i);
    }
    d.data = t->numel() ? t->data_ptr() : nullptr;
    d.device = t->is_cuda() ? (int32_t)t->get_device() : -1;
    return t->is_cuda() || t->is_cpu();
}

// Current stream of the tensor's device (null for host tensors, which the
// entry points reject); false with a Python error set.
bool stream_of(const at::Tensor& t, void** s) {
    *s = nullptr;
    if (!t.is_cuda()) return true;
    PyObject* dev = PyLong_FromLong(t.get_device());
    if (!dev) return false;
    PyObject* r = PyObject_CallOneArg(g_raw_stream, dev);
    Py_DECREF(dev);
    if (!r) return false;
    *s = PyLong_AsVoidPtr(r);
    Py_DECREF(r);
    return !PyErr_Occurred();
}

// t is contiguous, of this dtype, on the device and of these sizes.
bool is(const at::Tensor* t, at::ScalarType ty, const at::Device& dev, at::IntArrayRef sizes) {
    return t && t->scalar_type() == ty && t->device() == dev && t->is_contiguous() && t->sizes() == sizes;
}
bool is_index(const at::Tensor* t, const at::Device& dev, at::IntArrayRef sizes) {
    return is(t, at::kInt, dev, sizes) || is(t, at::kUInt32, dev, sizes);
}

// The status of f(), called without the interpreter lock. f calls the C ABI only
// (tensors are read before: they may raise, which takes the lock).
template <class F>
int unlocked(F&& f) {
    struct Unlock {
        PyThreadState* state = PyEval_SaveThread();
        ~Unlock() { PyEval_RestoreThread(state); }
    } unlock;
    return f();
}
template <class F>
PyObject* call(F&& f) {
    return PyLong_FromLong(unlocked(f));
}

template <class F>
PyObject* guarded(F&& f) {
    try {
        return f();
    } catch (const std::exception& e) {
        PyErr_SetString(PyExc_RuntimeError, e.what());
        return nullptr;
    }
}

// v[i] = the integers among the arguments; false (no error set) where one is
// not an int in range: the general route converts or rejects it.
bool ints(PyObject* const* a, int n, long long* v) {
    for (int i = 0; i < n; ++i) {
        if (!PyLong_Check(a[i])) return false;
        v[i] = PyLong_AsLongLong(a[i]);
        if (v[i] == -1 && PyErr_Occurred()) {
            PyErr_Clear();
            return false;
        }
    }
    return true;
}

bool argc(Py_ssize_t n, Py_ssize_t want) {
    if (n == want) return true;
    PyErr_Format(PyExc_TypeError, "expected %zd arguments, got %zd", want, n);
    return false;
}

// bind(topk, forward, router, fp8, packed, raw_stream): entry point addresses
PyObject* py_bind(PyObject*, PyObject* const* a, Py_ssize_t n) {
    if (!argc(n, 6)) return nullptr;
    void* p[5];
    for (int i = 0; i < 5; ++i) {
        p[i] = PyLong_AsVoidPtr(a[i]);
        if (PyErr_Occurred()) return nullptr;
    }
    g_topk = reinterpret_cast<decltype(g_topk)>(p[0]);
    g_forward = reinterpret_cast<decltype(g_forward)>(p[1]);
    g_router = reinterpret_cast<decltype(g_router)>(p[2]);
    g_fp8 = reinterpret_cast<decltype(g_fp8)>(p[3]);
    g_packed = reinterpret_cast<decltype(g_packed)>(p[4]);
    Py_INCREF(a[5]);
    Py_XSETREF(g_raw_stream, a[5]);
    Py_RETURN_NONE;
}

// topk(gating, weight, indices, token_expert_indices) -> status or None
PyObject* py_topk(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return guarded([&]() -> PyObject* {
        if (!argc(n, 4)) return nullptr;
        cm_tensor_t d[4];
        for (int i = 0; i < 4; ++i)
            if (!describe(a[i], d[i])) Py_RETURN_NONE;
        void* s;
        if (!stream_of(*plain(a[0]), &s)) return nullptr;
        return call([&] { return g_topk(&d[0], &d[1], &d[2], &d[3], s); });
    });
}

// forward(E, k, act, input, gate, up, down or None, weights, indices,
// moe_type) -> the output tensor, a failing call's status, or None
PyObject* py_forward(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return guarded([&]() -> PyObject* {
        if (!argc(n, 10)) return nullptr;
        long long v[3], moe_type;
        if (!ints(a, 3, v) || !ints(a + 9, 1, &moe_type) || moe_type < 0 || moe_type > 1 || v[2] < 0 || v[2] > 2)
            Py_RETURN_NONE;
        cm_fused_moe_t m;
        m.num_experts = v[0];
        m.num_selected_experts = v[1];
        m.activation = (int32_t)v[2];
        const bool has_down = a[6] != Py_None;
        cm_tensor_t d[6], od;
        for (int i = 0; i < 6; ++i)
            if ((i != 3 || has_down) && !describe(a[3 + i], d[i])) Py_RETURN_NONE;
        const at::Tensor& x = *plain(a[3]);
        if (x.dim() != 2 || !x.is_cuda()) Py_RETURN_NONE;
        void* s;
        if (!stream_of(x, &s)) return nullptr;
        at::Tensor out = at::empty(x.sizes(), at::TensorOptions().dtype(x.scalar_type()).device(x.device()));
        if (!out.has_storage() || out.unsafeGetTensorImpl()->is_python_dispatch()) Py_RETURN_NONE;
        od = d[0];
        od.data = out.numel() ? out.data_ptr() : nullptr;
        od.strides[0] = out.stride(0);
        od.strides[1] = out.stride(1);
        const int rc = unlocked([&] {
            return g_forward(&m, &d[0], &d[1], &d[2], has_down ? &d[3] : nullptr, &d[4], &d[5], (uint32_t)moe_type, &od,
                             s);
        });
        return rc == CANDLE_MOE_OK ? THPVariable_Wrap(std::move(out)) : PyLong_FromLong(rc);
    });
}

// router(hidden, router_weight, weight, indices, token_expert_indices) -> status or None
PyObject* py_router(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return guarded([&]() -> PyObject* {
        if (!argc(n, 5)) return nullptr;
        const at::Tensor* t[5];
        for (int i = 0; i < 5; ++i)
            if (!(t[i] = plain(a[i]))) Py_RETURN_NONE;
        const at::Tensor &x = *t[0], &w = *t[1];
        const int code = dtype_code(x.scalar_type());
        if (!x.is_cuda() || x.dim() != 2 || w.dim() != 2 || t[2]->dim() != 2 || code < 0 || code > CM_DT_F32 ||
            !x.is_contiguous())
            Py_RETURN_NONE;
        const long long T = x.size(0), H = x.size(1), E = w.size(0), k = t[2]->size(1);
        const at::Device dev = x.device();
        const int64_t tk[2] = {T, k};
        if (!is(&w, x.scalar_type(), dev, {E, H}) || !is(t[2], at::kFloat, dev, tk) || !is_index(t[3], dev, tk) ||
            !is_index(t[4], dev, tk) || T > INT_MAX || H > INT_MAX || E > INT_MAX)
            Py_RETURN_NONE;
        void* s;
        if (!stream_of(x, &s)) return nullptr;
        void* p[5];
        for (int i = 0; i < 5; ++i) p[i] = t[i]->data_ptr();
        return call([&] {
            return g_router(p[0], p[1], p[2], p[3], p[4], (int)T, (int)H, (int)E, (int)k, (uint32_t)code, s);
        });
    });
}

// The MoE calls over prepared weights (fp8 codes with scales, pre-packed):
// input, gate, up, down or None, (gate, up, down scales,) weights, indices,
// output, E, k, act, moe_type -> status or None
PyObject* prepared(PyObject* const* a, Py_ssize_t n, bool fp8) {
    return guarded([&]() -> PyObject* {
        const int ns = fp8 ? 3 : 0;
        if (!argc(n, 11 + ns)) return nullptr;
        long long v[4];
        if (!ints(a + 7 + ns, 4, v)) Py_RETURN_NONE;
        const long long E = v[0], k = v[1];
        if (v[3] < 0 || v[3] > 1 || v[2] < 0 || v[2] > 2 || E < 1 || k < 1 || E > INT_MAX || k > INT_MAX)
            Py_RETURN_NONE;
        const bool qwen3 = v[3] == 0;
        const at::Tensor* x = plain(a[0]);
        const at::Tensor* gate = plain(a[1]);
        if (!x || !gate || !x->is_cuda() || x->dim() != 2 || gate->dim() != 3 || !x->is_contiguous() ||
            (x->scalar_type() != at::kHalf && x->scalar_type() != at::kBFloat16))
            Py_RETURN_NONE;
        const int64_t T = x->size(0), H = x->size(1), I = gate->size(1);
        if (T > INT_MAX || H > INT_MAX || I > INT_MAX) Py_RETURN_NONE;
        const at::Device dev = x->device();
        const at::ScalarType ty = x->scalar_type(), wt = fp8 ? at::kByte : ty;
        const int64_t in[3] = {E, I, H}, out_s[3] = {E, H, I}, tk[2] = {T, k}, th[2] = {T, H};
        const at::Tensor* up = plain(a[2]);
        const at::Tensor* down = a[3] == Py_None ? nullptr : plain(a[3]);
        if (!is(gate, wt, dev, in) || !is(up, wt, dev, qwen3 ? at::IntArrayRef(in) : at::IntArrayRef(out_s)) ||
            (qwen3 ? !is(down, wt, dev, out_s) : a[3] != Py_None))
            Py_RETURN_NONE;
        const at::Tensor* sc[3] = {nullptr, nullptr, nullptr};
        if (fp8) {
            const int64_t si[2] = {E, I}, sh[2] = {E, H};
            for (int i = 0; i < 3; ++i) sc[i] = a[4 + i] == Py_None ? nullptr : plain(a[4 + i]);
            if (!is(sc[0], at::kFloat, dev, si) ||
                !is(sc[1], at::kFloat, dev, qwen3 ? at::IntArrayRef(si) : at::IntArrayRef(sh)) ||
                (qwen3 ? !is(sc[2], at::kFloat, dev, sh) : a[6] != Py_None))
                Py_RETURN_NONE;
        }
        const at::Tensor *rw = plain(a[4 + ns]), *idx = plain(a[5 + ns]), *out = plain(a[6 + ns]);
        if (!is(rw, at::kFloat, dev, tk) || !is_index(idx, dev, tk) || !is(out, ty, dev, th)) Py_RETURN_NONE;
        void* s;
        if (!stream_of(*x, &s)) return nullptr;
        const uint32_t code = (uint32_t)dtype_code(ty);
        const at::Tensor* all[10] = {x, gate, up, down, rw, idx, out, sc[0], sc[1], sc[2]};
        void* p[10];
        for (int i = 0; i < 10; ++i) p[i] = all[i] ? all[i]->data_ptr() : nullptr;
        return call([&] {
            if (fp8)
                return g_fp8(p[0], p[1], p[2], p[3], static_cast<const float*>(p[7]), static_cast<const float*>(p[8]),
                             static_cast<const float*>(p[9]), p[4], p[5], p[6], (int)T, (int)H, (int)I, (int)E, (int)k,
                             (int)v[2], (uint32_t)v[3], code, s);
            return g_packed(p[0], p[1], p[2], p[3], p[4], p[5], p[6], (int)T, (int)H, (int)I, (int)E, (int)k, (int)v[2],
                            (uint32_t)v[3], code, s);
        });
    });
}
PyObject* py_fp8(PyObject*, PyObject* const* a, Py_ssize_t n) { return prepared(a, n, true); }
PyObject* py_packed(PyObject*, PyObject* const* a, Py_ssize_t n) { return prepared(a, n, false); }

#define CM_METHOD(name) {#name, (PyCFunction)(void (*)(void))py_##name, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {CM_METHOD(bind), CM_METHOD(topk),   CM_METHOD(forward),          CM_METHOD(router),
                         CM_METHOD(fp8),  CM_METHOD(packed), {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_fast", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__fast(void) {
    PyObject* m = PyModule_Create(&module);
    // the torch it was built for: another one's objects are laid out differently
    if (m && PyModule_AddStringConstant(m, "torch_version", TORCH_VERSION) < 0) Py_CLEAR(m);
    return m;
}
