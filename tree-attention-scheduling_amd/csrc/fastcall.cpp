// fastcall.cpp -- Python entry of the per-layer calls (module _fastcall, host only).
//
// A decode step calls attention_matrix and decode_append once per layer, and a
// small layer runs for 9-20 us.  With the checks, the device context, the stream
// query and the ctypes call in Python, the host took 13 us for attention_matrix,
// 30 us for decode_append and attention_matrix, and 34 us with the tails' update
// before them, and the GPU waited; from here it takes 9, 15 and 18 us, most of it
// the launches (two, three and four), and the layers run at their device time.
//
// Each function covers the ordinary call -- contiguous tensors of the plan's
// shapes and dtype on the current device -- and does nothing for any other: it
// then returns None and the caller (kernels.py) runs the general path, which
// converts, names what is wrong, or switches the device.  Nothing is kept from
// one call for the next.
#include <torch/csrc/autograd/python_variable.h>

#include <ATen/ATen.h>

#include "tree_attn.h"

namespace {

// The library's functions (_native.load binds them) and torch's current-stream query.
struct Bound {
    decltype(&ta_attention_matrix) attention_matrix = nullptr;
    decltype(&ta_attention_tokens) attention_tokens = nullptr;
    decltype(&ta_decode_append) decode_append = nullptr;
    decltype(&ta_fill_lengths) fill_lengths = nullptr;
    PyObject *raw_stream = nullptr;      // torch._C._cuda_getCurrentRawStream
    PyObject *current_device = nullptr;  // torch._C._cuda_getDevice
} bound;

// The current stream of `device`, which has to be the current device.
bool stream_of(int device, void **stream) {
    PyObject *cur = PyObject_CallNoArgs(bound.current_device);
    if (!cur) return false;
    const long index = PyLong_AsLong(cur);
    Py_DECREF(cur);
    if (index != device) {
        PyErr_Clear();
        return false;
    }
    PyObject *arg = PyLong_FromLong(device);
    PyObject *raw = arg ? PyObject_CallOneArg(bound.raw_stream, arg) : nullptr;
    Py_XDECREF(arg);
    if (!raw) return false;
    *stream = PyLong_AsVoidPtr(raw);
    Py_DECREF(raw);
    return !PyErr_Occurred();
}

bool is_half(at::ScalarType t) { return t == at::kBFloat16 || t == at::kHalf; }
int ta_dtype(at::ScalarType t) { return t == at::kHalf ? TA_FP16 : TA_BF16; }

// A contiguous tensor in the memory of GPU `device`.
bool plain(const at::Tensor &t, at::ScalarType dtype, int device) {
    return t.defined() && t.layout() == at::kStrided && t.is_cuda() && t.get_device() == device &&
           t.scalar_type() == dtype && t.is_contiguous();
}

bool sizes(const at::Tensor &t, int64_t a, int64_t b, int64_t c) {
    return t.dim() == 3 && t.size(0) == a && t.size(1) == b && t.size(2) == c;
}

template <int N>
bool tensors(PyObject *const *args, const at::Tensor *(&out)[N]) {
    for (int i = 0; i < N; ++i) {
        if (!THPVariable_Check(args[i])) return false;
        out[i] = &THPVariable_Unpack(args[i]);
    }
    return true;
}

// Runs f without the GIL, as a ctypes call would; its code as a Python int.
template <class F>
PyObject *unlocked(F &&f) {
    int rc;
    Py_BEGIN_ALLOW_THREADS;
    rc = f();
    Py_END_ALLOW_THREADS;
    return PyLong_FromLong(rc);
}

// None (the general path), after dropping what an unusual tensor raised.
PyObject *general() {
    PyErr_Clear();
    Py_RETURN_NONE;
}

// attention(q, kp, vp, plan address, out, token_major): the library's return code, or None
PyObject *attention(PyObject *, PyObject *const *args, Py_ssize_t n) {
    try {
        if (n != 6 || !bound.attention_matrix) return general();
        const at::Tensor *t[3], *o[1];
        if (!tensors(args, t) || !tensors(args + 4, o)) return general();
        const ta_plan *plan = static_cast<const ta_plan *>(PyLong_AsVoidPtr(args[3]));
        const int tokens = PyObject_IsTrue(args[5]);
        if (!plan || tokens < 0) return general();
        const at::Tensor &q = *t[0], &k = *t[1], &v = *t[2];
        const at::ScalarType dtype = q.scalar_type();
        if (!is_half(dtype) || ta_dtype(dtype) != plan->dtype || !q.is_cuda()) return general();
        const int device = (int)q.get_device();
        if (!plain(q, dtype, device) || !plain(k, dtype, device) || !plain(v, dtype, device) ||
            !sizes(q, plan->nreq, plan->hq, plan->d) || k.dim() != 3)
            return general();
        const int64_t cap = k.size(tokens ? 0 : 2);
        if (cap <= 0 || cap > INT32_MAX) return general();
        if (tokens) {
            if (!sizes(k, cap, plan->hk, plan->d) || !sizes(v, cap, plan->hk, plan->d)) return general();
            // (a view may start anywhere; a packed copy would not)
            if ((uintptr_t)k.data_ptr() % 16 || (uintptr_t)v.data_ptr() % 16) return general();
        } else if (!sizes(k, plan->hk, plan->d, cap) || !sizes(v, plan->hk, cap, plan->d)) {
            return general();
        }
        if (plan->xtail && cap % 8) return general();  // PreparedPlan.for_capacity
        void *stream;
        if (!stream_of(device, &stream)) return general();
        const void *qp = q.data_ptr(), *kp = k.data_ptr(), *vp = v.data_ptr();
        void *out = o[0]->data_ptr();
        const auto fn = tokens ? bound.attention_tokens : bound.attention_matrix;
        return unlocked([&] { return fn(qp, kp, vp, (int32_t)cap, plan, out, stream); });
    } catch (...) {
        return general();
    }
}

// decode_append(q, k, v, cos, sin, slots, kp, vp): the rotated q, the library's return code if
// that is not 0, or None
PyObject *append(PyObject *, PyObject *const *args, Py_ssize_t n) {
    try {
        if (n != 8 || !bound.decode_append) return general();
        const at::Tensor *t[8];
        if (!tensors(args, t)) return general();
        const at::Tensor &q = *t[0], &k = *t[1], &v = *t[2], &cos = *t[3], &sin = *t[4], &slots = *t[5], &kp = *t[6],
                         &vp = *t[7];
        const at::ScalarType dtype = q.scalar_type();
        if (!is_half(dtype) || !q.is_cuda() || q.dim() < 2) return general();
        const int device = (int)q.get_device();
        for (const at::Tensor *x : {&q, &k, &v, &cos, &sin, &kp, &vp})
            if (!plain(*x, dtype, device)) return general();
        const int64_t nreq = q.size(0), d = q.size(-1);
        if (!plain(slots, at::kInt, device) || slots.numel() != nreq || nreq <= 0 || d <= 0 || nreq > INT32_MAX)
            return general();
        if (q.numel() % (nreq * d) || k.numel() % (nreq * d) || k.dim() < 2 || v.dim() < 2 || k.size(0) != nreq ||
            v.size(0) != nreq || k.size(-1) != d || v.size(-1) != d || v.numel() != k.numel())
            return general();
        const int64_t hq = q.numel() / (nreq * d), hk = k.numel() / (nreq * d);
        if (kp.dim() != 3) return general();
        const int64_t cap = kp.size(2);
        if (hq <= 0 || hk <= 0 || cap <= 0 || cap > INT32_MAX || !sizes(kp, hk, d, cap) || !sizes(vp, hk, cap, d))
            return general();
        const int64_t rope = cos.numel();  // one row of d values for all requests, or one each
        if (sin.numel() != rope || (rope != d && rope != nreq * d) || cos.size(-1) != d || sin.size(-1) != d)
            return general();
        void *stream;
        if (!stream_of(device, &stream)) return general();
        at::Tensor out = at::empty({nreq, hq, d}, q.options());
        const void *p[5] = {q.data_ptr(), k.data_ptr(), v.data_ptr(), cos.data_ptr(), sin.data_ptr()};
        const int32_t *at_slots = static_cast<const int32_t *>(slots.data_ptr());
        void *kpp = kp.data_ptr(), *vpp = vp.data_ptr(), *op = out.data_ptr();
        int rc;
        Py_BEGIN_ALLOW_THREADS;
        rc = bound.decode_append(p[0], p[1], p[2], p[3], p[4], rope == nreq * d ? (int32_t)d : 0, at_slots, kpp, vpp,
                                 op, (int32_t)nreq, (int32_t)hq, (int32_t)hk, (int32_t)d, (int32_t)cap,
                                 ta_dtype(dtype), stream);
        Py_END_ALLOW_THREADS;
        if (rc) return PyLong_FromLong(rc);
        return THPVariable_Wrap(std::move(out));
    } catch (...) {
        return general();
    }
}

// fill(metadata int32, offsets int64, value): the library's return code, or None
PyObject *fill(PyObject *, PyObject *const *args, Py_ssize_t n) {
    try {
        if (n != 3 || !bound.fill_lengths) return general();
        const at::Tensor *t[2];
        if (!tensors(args, t)) return general();
        const long value = PyLong_AsLong(args[2]);
        if (PyErr_Occurred() || value < 0 || value > INT32_MAX || !t[0]->is_cuda()) return general();
        const int device = (int)t[0]->get_device();
        if (!plain(*t[0], at::kInt, device) || !plain(*t[1], at::kLong, device) || t[1]->numel() > INT32_MAX)
            return general();
        void *stream;
        if (!stream_of(device, &stream)) return general();
        int32_t *meta = static_cast<int32_t *>(t[0]->data_ptr());
        const int64_t *offs = static_cast<const int64_t *>(t[1]->data_ptr());
        const int32_t count = (int32_t)t[1]->numel();
        return unlocked([&] { return bound.fill_lengths(meta, offs, count, (int32_t)value, stream); });
    } catch (...) {
        return general();
    }
}

// bind(addresses of ta_attention_matrix, ta_attention_tokens, ta_decode_append, ta_fill_lengths,
//      torch._C._cuda_getCurrentRawStream, torch._C._cuda_getDevice)
PyObject *bind(PyObject *, PyObject *const *args, Py_ssize_t n) {
    if (n != 6) {
        PyErr_SetString(PyExc_TypeError, "bind takes four addresses and two functions");
        return nullptr;
    }
    Bound b;
    b.attention_matrix = reinterpret_cast<decltype(b.attention_matrix)>(PyLong_AsVoidPtr(args[0]));
    b.attention_tokens = reinterpret_cast<decltype(b.attention_tokens)>(PyLong_AsVoidPtr(args[1]));
    b.decode_append = reinterpret_cast<decltype(b.decode_append)>(PyLong_AsVoidPtr(args[2]));
    b.fill_lengths = reinterpret_cast<decltype(b.fill_lengths)>(PyLong_AsVoidPtr(args[3]));
    if (PyErr_Occurred()) return nullptr;
    Py_INCREF(args[4]);
    Py_INCREF(args[5]);
    b.raw_stream = args[4];
    b.current_device = args[5];
    std::swap(bound, b);
    Py_XDECREF(b.raw_stream);
    Py_XDECREF(b.current_device);
    Py_RETURN_NONE;
}

#define TA_FAST(NAME, FN) {NAME, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(FN)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {TA_FAST("attention", attention), TA_FAST("decode_append", append), TA_FAST("fill", fill),
                         TA_FAST("bind", bind), {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_fastcall", nullptr, -1, methods};

}  // namespace

// BUILT_FOR names the Python and the torch whose object layouts the module was compiled with;
// _native uses it with no other.
PyMODINIT_FUNC PyInit__fastcall(void) {
    PyObject *m = PyModule_Create(&module);
    if (m && PyModule_AddStringConstant(m, "BUILT_FOR", TA_BUILT_FOR) < 0) {
        Py_DECREF(m);
        return nullptr;
    }
    return m;
}
