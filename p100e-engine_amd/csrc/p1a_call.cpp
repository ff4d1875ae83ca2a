// The Python side of a call in native code: arguments -> the C ABI of include/p1a_attn.h. A one-row step of a small model is
// bound by what the host does around its three launches, and half of what was not the launches was the ctypes call: 19
// arguments converted one by one, a descriptor built field by field, a stream looked up from Python. The calls a step is made of
// come here instead; arguments are taken as ctypes takes them (whole numbers cut to 32 bits, floats, ctypes numbers of the parameter's
// type, what _as_parameter_ stands for, None for a null pointer, anything with data_ptr() as a device pointer), and the GIL is released around the call. One token of 4 heads of 64, prep and decode from Python:
// 18.1 us with ctypes, 15.6 so (7.7 of them the C calls, 3.5 the caller's own indexing); two layers of 24 / 4 heads of 96 34.4 -> 29.2.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <cstdint>
#include <cstring>

#include "p1a_attn.h"

namespace {

PyObject * s_data_ptr, * s_struct, * s_value, * s_as_parameter, * s_field[11];
const char * const FIELDS[11] = {"type", "n_ctx", "Hkv", "D", "k", "v", "pt", "rtab", "psh", "pstride", "_pt_off"};
enum { INT, UINT, SIZE, FLOAT, POINTER, DESC, NCLASS };

// A module's state (a process may load the binding more than once), set by bind()
struct calls {
    // the library's entry points, the class whose fields are read directly, and how the current stream is found
    decltype(&p1a_attn_prep) f_prep;
    decltype(&p1a_attn_decode_a16) f_decode;
    decltype(&p1a_attn_prefill) f_prefill;
    decltype(&p1a_kv_append) f_append;
    PyObject * kv_class, * stream_of;
    PyObject * classes[NCLASS];   // ctypes' c_int, c_uint32, c_size_t, c_float, c_void_p, and the descriptor's Structure

    // (each reader does nothing once an error is set, so that the callers test for one at the end)
    // The value of a ctypes number, for a parameter of just that type; else null. of: its class (c_int, c_float, ...)
    PyObject * plain(PyObject * o, int of) {
        if (PyErr_Occurred()) return nullptr;
        const int is = PyObject_IsInstance(o, classes[of]);
        return is == 1 ? PyObject_GetAttr(o, s_value) : nullptr;
    }
    // what an argument says it stands for, or null (and the error there was stays)
    PyObject * stand_in(PyObject * o, bool argument) {
        if (!argument || !PyErr_ExceptionMatches(PyExc_TypeError)) return nullptr;
        PyObject * t, * v, * tb;
        PyErr_Fetch(&t, &v, &tb);
        PyObject * r = PyObject_GetAttr(o, s_as_parameter);
        if (!r) { PyErr_Clear(); PyErr_Restore(t, v, tb); return nullptr; }
        Py_XDECREF(t); Py_XDECREF(v); Py_XDECREF(tb);
        return r;
    }
    uint64_t whole(PyObject * o, int of, bool argument = true) {
        if (PyErr_Occurred()) return 0;
        if (PyLong_CheckExact(o)) return (uint64_t) PyLong_AsUnsignedLongMask(o);
        uint64_t r = 0;
        if (PyObject * v = plain(o, of)) { r = whole(v, of, false); Py_DECREF(v); return r; }
        if (PyErr_Occurred()) return 0;
        if (PyFloat_Check(o)) PyErr_SetString(PyExc_TypeError, "int expected instead of float instance");
        else r = (uint64_t) PyLong_AsUnsignedLongMask(o);
        if (PyErr_Occurred())
            if (PyObject * v = stand_in(o, argument)) { r = Py_EnterRecursiveCall(" in a call's argument") ? 0 : (r = whole(v, of), Py_LeaveRecursiveCall(), r); Py_DECREF(v); }
        return r;
    }
    int as_int(PyObject * o) { return (int) (uint32_t) whole(o, INT); }
    size_t as_size(PyObject * o) { return (size_t) whole(o, SIZE); }
    float as_float(PyObject * o) {
        if (PyErr_Occurred()) return 0.f;
        if (PyFloat_CheckExact(o)) return (float) PyFloat_AS_DOUBLE(o);
        float r = 0.f;
        if (PyObject * v = plain(o, FLOAT)) { r = as_float(v); Py_DECREF(v); return r; }
        if (PyErr_Occurred()) return 0.f;
        r = (float) PyFloat_AsDouble(o);
        if (PyErr_Occurred())
            if (PyObject * v = stand_in(o, true)) { r = Py_EnterRecursiveCall(" in a call's argument") ? 0.f : (r = as_float(v), Py_LeaveRecursiveCall(), r); Py_DECREF(v); }
        return r;
    }
    // a pointer: None, a Python int, a c_void_p
    void * address(PyObject * o) {
        if (PyErr_Occurred() || o == Py_None) return nullptr;
        if (PyLong_Check(o)) return (void *) (uintptr_t) PyLong_AsUnsignedLongMask(o);
        void * r = nullptr;
        if (PyObject * v = plain(o, POINTER)) { r = address(v); Py_DECREF(v); }
        else if (!PyErr_Occurred()) PyErr_Format(PyExc_TypeError, "address expected instead of %s instance", Py_TYPE(o)->tp_name);
        return r;
    }
    PyObject * data_ptr_of(PyObject * t) { return PyErr_Occurred() ? nullptr : PyObject_CallMethodNoArgs(t, s_data_ptr); }
    void * data_ptr(PyObject * t) {
        if (PyErr_Occurred() || t == Py_None) return nullptr;
        PyObject * r = data_ptr_of(t);
        if (!r) return nullptr;
        void * p = address(r);
        Py_DECREF(r);
        return p;
    }
    template <typename T> T * ptr(PyObject * t) { return (T *) data_ptr(t); }
    // the page table from its entry `off` on
    const int32_t * table(PyObject * t, PyObject * off) {
        if (PyErr_Occurred() || t == Py_None) return nullptr;
        PyObject * r = data_ptr_of(t);
        if (!r) return nullptr;
        const char * p = nullptr;
        if (PyLong_Check(r) && PyLong_Check(off)) p = (const char *) (uintptr_t) PyLong_AsUnsignedLongMask(r) + 4 * (ptrdiff_t) PyLong_AsUnsignedLongMask(off);
        else PyErr_SetString(PyExc_TypeError, "the page table's address and offset are whole numbers");
        Py_DECREF(r);
        return (const int32_t *) p;
    }

    // the cache's descriptor as it is now: a KVCache's fields, or what its struct() gives
    bool describe(PyObject * c, p1a_kv & kv) {
        if (PyErr_Occurred()) return false;
        if ((PyObject *) Py_TYPE(c) != kv_class) {
            PyObject * st = PyObject_CallMethodNoArgs(c, s_struct);
            if (!st) return false;
            Py_buffer b;
            const int is = PyObject_IsInstance(st, classes[DESC]);
            if (is == 0) PyErr_SetString(PyExc_TypeError, "struct() gave no p1a_kv");
            if (is == 1 && PyObject_GetBuffer(st, &b, PyBUF_SIMPLE) == 0) {
                memcpy(&kv, b.buf, sizeof kv);
                PyBuffer_Release(&b);
            }
            Py_DECREF(st);
            return !PyErr_Occurred();
        }
        PyObject * f[11] = {};
        for (int i = 0; i < 11 && !PyErr_Occurred(); ++i) f[i] = PyObject_GetAttr(c, s_field[i]);
        if (!PyErr_Occurred()) {
            kv.type = (uint32_t) whole(f[0], UINT, false);
            kv.n_ctx = (int) whole(f[1], INT, false); kv.Hkv = (int) whole(f[2], INT, false); kv.D = (int) whole(f[3], INT, false);
            kv.k = address(f[4]); kv.v = address(f[5]);
            kv.pt = table(f[6], f[10]);
            kv.rtab = ptr<int32_t>(f[7]);
            kv.psh = (int) whole(f[8], INT, false);
            kv.pstride = (size_t) whole(f[9], SIZE, false);
        }
        for (PyObject * x : f) Py_XDECREF(x);
        return !PyErr_Occurred();
    }
    void * stream() {
        if (PyErr_Occurred()) return nullptr;
        PyObject * r = PyObject_CallNoArgs(stream_of);
        if (!r) return nullptr;
        void * p = address(r);
        Py_DECREF(r);
        return p;
    }
};

bool takes(Py_ssize_t n, Py_ssize_t want) {
    if (n != want) PyErr_Format(PyExc_TypeError, "%zd arguments expected, %zd given", want, n);
    return n == want;
}
bool bound(const calls & C) {
    if (!C.f_append) PyErr_SetString(PyExc_RuntimeError, "bind() comes first");
    return C.f_append;
}
#define P1A_CALL(expr) do { if (PyErr_Occurred()) return nullptr; int rc_; Py_BEGIN_ALLOW_THREADS rc_ = (expr); Py_END_ALLOW_THREADS return PyLong_FromLong(rc_); } while (0)

// (qg, k, v, q_norm, k_norm, pos, q, gate, cache, p0, T, Hq, n_rot, freq_base, eps, ldq, ldk, ldv)
PyObject * prep(PyObject * self, PyObject * const * a, Py_ssize_t n) {
    calls & C = *(calls *) PyModule_GetState(self);
    if (!takes(n, 18) || !bound(C)) return nullptr;
    p1a_kv kv;
    float * p[8];
    for (int i = 0; i < 8; ++i) p[i] = C.ptr<float>(a[i]);
    C.describe(a[8], kv);
    const int p0 = C.as_int(a[9]), T = C.as_int(a[10]), Hq = C.as_int(a[11]), nr = C.as_int(a[12]);
    const float base = C.as_float(a[13]), eps = C.as_float(a[14]);
    const int lq = C.as_int(a[15]), lk = C.as_int(a[16]), lv = C.as_int(a[17]);
    void * s = C.stream();
    P1A_CALL(C.f_prep(p[0], p[1], p[2], p[3], p[4], (const int32_t *) p[5], p[6], p[7], &kv, p0, T, Hq, nr, base, eps, lq, lk, lv, s));
}
// (q, cache, out, gate, qbuf, T, p0, p0_dev, pos, rows_per_seq, Hq, scale)
PyObject * decode(PyObject * self, PyObject * const * a, Py_ssize_t n) {
    calls & C = *(calls *) PyModule_GetState(self);
    if (!takes(n, 12) || !bound(C)) return nullptr;
    p1a_kv kv;
    const float * q = C.ptr<float>(a[0]);
    C.describe(a[1], kv);
    float * out = C.ptr<float>(a[2]);
    const float * gate = C.ptr<float>(a[3]);
    void * qbuf = C.data_ptr(a[4]);
    const int T = C.as_int(a[5]), p0 = C.as_int(a[6]);
    const int32_t * p0_dev = C.ptr<int32_t>(a[7]), * pos = C.ptr<int32_t>(a[8]);
    const int rps = C.as_int(a[9]), Hq = C.as_int(a[10]);
    const float scale = C.as_float(a[11]);
    void * s = C.stream();
    P1A_CALL(C.f_decode(q, &kv, out, gate, qbuf, T, p0, p0_dev, pos, rps, Hq, scale, s));
}
// (q, cache, out, gate, T, p0, Hq, scale, scratch, scratch_bytes)
PyObject * prefill(PyObject * self, PyObject * const * a, Py_ssize_t n) {
    calls & C = *(calls *) PyModule_GetState(self);
    if (!takes(n, 10) || !bound(C)) return nullptr;
    p1a_kv kv;
    const float * q = C.ptr<float>(a[0]);
    C.describe(a[1], kv);
    float * out = C.ptr<float>(a[2]);
    const float * gate = C.ptr<float>(a[3]);
    const int T = C.as_int(a[4]), p0 = C.as_int(a[5]), Hq = C.as_int(a[6]);
    const float scale = C.as_float(a[7]);
    void * scratch = C.data_ptr(a[8]);
    const size_t bytes = C.as_size(a[9]);
    void * s = C.stream();
    P1A_CALL(C.f_prefill(q, &kv, out, gate, T, p0, Hq, scale, scratch, bytes, s));
}
// (cache, k, v, p0, p0_dev, pos, T)
PyObject * append(PyObject * self, PyObject * const * a, Py_ssize_t n) {
    calls & C = *(calls *) PyModule_GetState(self);
    if (!takes(n, 7) || !bound(C)) return nullptr;
    p1a_kv kv;
    C.describe(a[0], kv);
    const float * k = C.ptr<float>(a[1]), * v = C.ptr<float>(a[2]);
    const int p0 = C.as_int(a[3]);
    const int32_t * p0_dev = C.ptr<int32_t>(a[4]), * pos = C.ptr<int32_t>(a[5]);
    const int T = C.as_int(a[6]);
    void * s = C.stream();
    P1A_CALL(C.f_append(&kv, k, v, p0, p0_dev, pos, T, s));
}
// (addresses of p1a_attn_prep, p1a_attn_decode_a16, p1a_attn_prefill, p1a_kv_append; the cache class; the current stream's handle; the
// ctypes classes)
PyObject * bind(PyObject * self, PyObject * const * a, Py_ssize_t n) {
    calls & C = *(calls *) PyModule_GetState(self);
    if (!takes(n, 6 + NCLASS)) return nullptr;
    C.f_prep = (decltype(C.f_prep)) C.address(a[0]);
    C.f_decode = (decltype(C.f_decode)) C.address(a[1]);
    C.f_prefill = (decltype(C.f_prefill)) C.address(a[2]);
    C.f_append = (decltype(C.f_append)) C.address(a[3]);
    if (PyErr_Occurred()) return nullptr;
    Py_INCREF(a[4]); Py_XSETREF(C.kv_class, a[4]);
    Py_INCREF(a[5]); Py_XSETREF(C.stream_of, a[5]);
    for (int i = 0; i < NCLASS; ++i) { Py_INCREF(a[6 + i]); Py_XSETREF(C.classes[i], a[6 + i]); }
    Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"bind", (PyCFunction) (void (*)(void)) bind, METH_FASTCALL, nullptr}, {"prep", (PyCFunction) (void (*)(void)) prep, METH_FASTCALL, nullptr},
    {"decode", (PyCFunction) (void (*)(void)) decode, METH_FASTCALL, nullptr}, {"prefill", (PyCFunction) (void (*)(void)) prefill, METH_FASTCALL, nullptr},
    {"append", (PyCFunction) (void (*)(void)) append, METH_FASTCALL, nullptr}, {nullptr, nullptr, 0, nullptr}};
int setup(PyObject *) {
    if (s_data_ptr) return 0;
    s_struct = PyUnicode_InternFromString("struct");
    s_value = PyUnicode_InternFromString("value");
    s_as_parameter = PyUnicode_InternFromString("_as_parameter_");
    for (int i = 0; i < 11; ++i) s_field[i] = PyUnicode_InternFromString(FIELDS[i]);
    s_data_ptr = PyUnicode_InternFromString("data_ptr");
    return PyErr_Occurred() ? -1 : 0;
}
int traverse(PyObject * self, visitproc visit, void * arg) {
    if (calls * C = (calls *) PyModule_GetState(self)) {
        Py_VISIT(C->kv_class); Py_VISIT(C->stream_of);
        for (PyObject * x : C->classes) Py_VISIT(x);
    }
    return 0;
}
int clear(PyObject * self) {
    if (calls * C = (calls *) PyModule_GetState(self)) {
        Py_CLEAR(C->kv_class); Py_CLEAR(C->stream_of);
        for (PyObject * & x : C->classes) Py_CLEAR(x);
    }
    return 0;
}
void drop(void * self) { clear((PyObject *) self); }
PyModuleDef_Slot slots[] = {{Py_mod_exec, (void *) setup}, {0, nullptr}};
PyModuleDef module_ = {PyModuleDef_HEAD_INIT, "_p1a_call", nullptr, sizeof(calls), methods, slots, traverse, clear, drop};

}   // namespace

PyMODINIT_FUNC PyInit__p1a_call(void) { return PyModuleDef_Init(&module_); }
