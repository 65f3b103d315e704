// CPython extension `kvhip._step`: one attention call of a layer -- `attentionWithCacheUpdate`, with or without the rotary
// positions in front -- from its tensors to the C entry point in one native call.  A short decode step takes the device less
// time than the interpreter took to look the tensors' shapes, types and addresses up and to convert twenty arguments
// (16 layers over 512 keys of one sequence: 149 us a pass, 130 from here).  Handles the ordinary form of the call; for
// everything else (other masks, arrays that are not contiguous, shapes or types that do not go together, numbers that are
// none) it returns None before anything is done, and the Python methods, which check and report, take the call.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include "kvhip.h"

namespace {

PyObject *g_tensor_type, *g_rope_type;           // torch.Tensor, kvhip.RoPE
PyObject *g_dtypes[3], *g_device, *g_raw_stream;  // float16, bfloat16, float32; the current device and its stream
PyObject *s_is_contiguous, *s_is_cuda, *s_dtype, *s_shape, *s_data_ptr, *s_new_empty, *s_dims, *s_traditional, *s_base, *s_scale, *s_freqs;

struct Array {
    long long n[4];
    int dtype;  // kvhip_dtype
    void *p;
};

bool take_int(PyObject *o, long long &v) {
    v = PyLong_AsLongLong(o);
    return !(v == -1 && PyErr_Occurred());
}
bool is_true(PyObject *o) {  // steals o
    const bool t = o == Py_True;
    Py_XDECREF(o);
    return t;
}
// the tensor as the library reads it; false (perhaps with an exception set): not of the ordinary form
bool take(PyObject *t, Array &a) {
    if (reinterpret_cast<PyObject *>(Py_TYPE(t)) != g_tensor_type) return false;
    if (!is_true(PyObject_GetAttr(t, s_is_cuda)) || !is_true(PyObject_CallMethodNoArgs(t, s_is_contiguous))) return false;
    PyObject *dt = PyObject_GetAttr(t, s_dtype);
    a.dtype = -1;
    for (int i = 0; i < 3; ++i)
        if (dt == g_dtypes[i]) a.dtype = i;
    Py_XDECREF(dt);
    if (a.dtype < 0) return false;
    PyObject *shape = PyObject_GetAttr(t, s_shape);
    bool ok = shape && PyTuple_Check(shape) && PyTuple_GET_SIZE(shape) == 4;
    for (int i = 0; ok && i < 4; ++i) ok = take_int(PyTuple_GET_ITEM(shape, i), a.n[i]) && a.n[i] > 0 && a.n[i] <= INT32_MAX;
    Py_XDECREF(shape);
    if (!ok) return false;
    PyObject *ptr = PyObject_CallMethodNoArgs(t, s_data_ptr);
    a.p = ptr ? PyLong_AsVoidPtr(ptr) : nullptr;
    Py_XDECREF(ptr);
    return a.p != nullptr;
}
PyObject *none() {  // (an interrupt or an exit is not a form of the call)
    if (PyErr_Occurred()) {
        if (!PyErr_ExceptionMatches(PyExc_Exception)) return nullptr;
        PyErr_Clear();
    }
    Py_RETURN_NONE;
}

// attend(entry, handle, shape, q, k, v, scale, mask, rope, keep)
//   entry    address of kvhip_cache_update_attend, or of kvhip_cache_update_attend_rope if `rope` is not None
//   shape    (B, kv heads, key size, value size, dtype) of what the cache holds
//   mask     address of a kvhip_mask
//   keep     largest rotated queries, in bytes, for which the cache's own buffer is to be used
// Returns the output tensor, None (not handled, nothing done) or the status of a call that failed.
PyObject *attend(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
    if (nargs != 10) {
        PyErr_SetString(PyExc_TypeError, "attend takes 10 arguments");
        return nullptr;
    }
    Array q, k, v;
    if (!take(args[3], q) || !take(args[4], k) || !take(args[5], v)) return none();
    const long long B = q.n[0], Hq = q.n[1], L = q.n[2], Dk = q.n[3], Hkv = k.n[1], Dv = v.n[3];
    if (k.n[0] != B || v.n[0] != B || k.n[2] != L || v.n[2] != L || k.n[3] != Dk || v.n[1] != Hkv || q.dtype != k.dtype || v.dtype != k.dtype) return none();
    PyObject *held = args[2];
    if (!PyTuple_Check(held) || PyTuple_GET_SIZE(held) != 5 || PyTuple_GET_ITEM(held, 4) != g_dtypes[k.dtype]) return none();
    const long long want[4] = {B, Hkv, Dk, Dv};
    for (int i = 0; i < 4; ++i) {
        long long n;
        if (!take_int(PyTuple_GET_ITEM(held, i), n) || n != want[i]) return none();
    }
    PyObject *rope = args[8];
    kvhip_rope r{};
    PyObject *freqs = nullptr;
    if (rope != Py_None) {
        long long keep;
        if (reinterpret_cast<PyObject *>(Py_TYPE(rope)) != g_rope_type) return none();
        if (!take_int(args[9], keep) || B * Hq * L * Dk * (k.dtype == KVHIP_F32 ? 4 : 2) > keep) return none();
        PyObject *dims = PyObject_GetAttr(rope, s_dims), *trad = PyObject_GetAttr(rope, s_traditional), *base = PyObject_GetAttr(rope, s_base),
                 *scale = PyObject_GetAttr(rope, s_scale);
        freqs = PyObject_GetAttr(rope, s_freqs);
        if (dims && trad && base && scale && freqs) {
            r.dims = (int32_t)PyLong_AsLong(dims);
            r.traditional = PyObject_IsTrue(trad) == 1;
            r.base = (float)PyFloat_AsDouble(base);
            r.scale = (float)PyFloat_AsDouble(scale);
            if (freqs != Py_None) {
                PyObject *ptr = PyObject_CallMethodNoArgs(freqs, s_data_ptr);
                r.freqs = ptr ? static_cast<const float *>(PyLong_AsVoidPtr(ptr)) : nullptr;
                Py_XDECREF(ptr);
            }
        }
        Py_XDECREF(dims);
        Py_XDECREF(trad);
        Py_XDECREF(base);
        Py_XDECREF(scale);
    }
    const float scale = (float)PyFloat_AsDouble(args[6]);
    auto *cache = static_cast<kvhip_cache *>(PyLong_AsVoidPtr(args[1]));
    const auto *mask = static_cast<const kvhip_mask *>(PyLong_AsVoidPtr(args[7]));
    void *entry = PyLong_AsVoidPtr(args[0]);
    if (PyErr_Occurred() || !cache || !mask || !entry) {
        Py_XDECREF(freqs);
        return none();
    }
    PyObject *size = Py_BuildValue("(LLLL)", B, Hq, L, Dv);
    PyObject *out = size ? PyObject_CallMethodOneArg(args[3], s_new_empty, size) : nullptr;
    Py_XDECREF(size);
    PyObject *device = out ? PyObject_CallNoArgs(g_device) : nullptr;
    PyObject *stream = device ? PyObject_CallOneArg(g_raw_stream, device) : nullptr;
    PyObject *ptr = stream ? PyObject_CallMethodNoArgs(out, s_data_ptr) : nullptr;
    void *dst = ptr ? PyLong_AsVoidPtr(ptr) : nullptr, *st = stream ? PyLong_AsVoidPtr(stream) : nullptr;
    Py_XDECREF(ptr);
    Py_XDECREF(device);
    Py_XDECREF(stream);
    if (PyErr_Occurred()) {
        Py_XDECREF(out);
        Py_XDECREF(freqs);
        return nullptr;
    }
    kvhip_status status;
    Py_BEGIN_ALLOW_THREADS
    if (rope == Py_None)
        status = reinterpret_cast<decltype(&kvhip_cache_update_attend)>(entry)(cache, q.p, k.p, v.p, (int32_t)B, (int32_t)Hq, (int32_t)Hkv, (int32_t)L,
                                                                               (int32_t)Dk, (int32_t)Dv, k.dtype, scale, mask, dst, st);
    else
        status = reinterpret_cast<decltype(&kvhip_cache_update_attend_rope)>(entry)(cache, &r, nullptr, q.p, k.p, v.p, (int32_t)B, (int32_t)Hq, (int32_t)Hkv,
                                                                                    (int32_t)L, (int32_t)Dk, (int32_t)Dv, k.dtype, scale, mask, nullptr, dst, st);
    Py_END_ALLOW_THREADS
    Py_XDECREF(freqs);
    if (status >= KVHIP_OK) return out;
    Py_DECREF(out);
    return PyLong_FromLong(status);
}

// bind(Tensor, RoPE, (float16, bfloat16, float32), current device, its raw stream)
PyObject *bind(PyObject *, PyObject *args) {
    PyObject *types;
    if (!PyArg_ParseTuple(args, "OOO!OO", &g_tensor_type, &g_rope_type, &PyTuple_Type, &types, &g_device, &g_raw_stream)) return nullptr;
    if (PyTuple_GET_SIZE(types) != 3) {
        PyErr_SetString(PyExc_TypeError, "three dtypes");
        return nullptr;
    }
    Py_INCREF(g_tensor_type);
    Py_INCREF(g_rope_type);
    Py_INCREF(g_device);
    Py_INCREF(g_raw_stream);
    for (int i = 0; i < 3; ++i) {
        g_dtypes[i] = PyTuple_GET_ITEM(types, i);
        Py_INCREF(g_dtypes[i]);
    }
    Py_RETURN_NONE;
}

PyMethodDef g_methods[] = {{"attend", reinterpret_cast<PyCFunction>(reinterpret_cast<void *>(attend)), METH_FASTCALL, nullptr},
                           {"bind", bind, METH_VARARGS, nullptr},
                           {nullptr, nullptr, 0, nullptr}};
PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "_step", nullptr, -1, g_methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__step() {
    const struct {
        PyObject **to;
        const char *name;
    } names[] = {{&s_is_contiguous, "is_contiguous"}, {&s_is_cuda, "is_cuda"}, {&s_dtype, "dtype"}, {&s_shape, "shape"}, {&s_data_ptr, "data_ptr"},
                 {&s_new_empty, "new_empty"}, {&s_dims, "dims"}, {&s_traditional, "traditional"}, {&s_base, "base"}, {&s_scale, "scale"}, {&s_freqs, "freqs"}};
    for (const auto &n : names)
        if (!(*n.to = PyUnicode_InternFromString(n.name))) return nullptr;
    return PyModule_Create(&g_module);
}
