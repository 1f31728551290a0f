// The object layer of the Python classes in native code: the buffer of a result, the view of it (shape, strides,
// offset) and the call of one host-layer function on views, as the reference's generated C methods do it above
// ndloop. narray.py derives its classes from View and hands the calls that make up nearly every program to the
// functions here; whatever they do not take (a numpy number, an odd axis, a call inside a recording) goes to the
// Python method of the same name, which takes every form.
//
// Why native: a 10000-element x + b cost 7.9 us of the caller's time, of which the library and the launch are 2.9;
// the rest was ctypes structures filled element by element, three more ctypes calls (storage size, error latch,
// release) and the objects around them. Now 3.5 us; sum 7.2 -> 3.9, mulsum 7.6 -> 3.9. A chain of six such calls on
// 10000 elements 52 -> 26 us, on 2^20 54 -> 25; ten reductions of a 500 x 500 matrix 113 -> 54 (all with three to ten
// results looked at as tensors, 1.6 us each).
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <structmember.h>

#include <cstdint>
#include <cstring>
#include <memory>
#include <new>

#include "cumo_hip.h"
#include "cumo_hip_ndloop.h"

namespace {

using Desc = cumo_hip_narray_t;

// what narray.py registers once: the class of each type code, the function that turns a latched error into its
// exception, the object whose _call1 takes the general form of a function of one argument
PyObject* g_class[8];
PyObject* g_raise;
PyObject* g_nmath;
PyObject* g_recording;  // the list of a running recording, or null

// 0 when nothing is latched, else an exception is set
int raise_latched() {
    const char* msg = nullptr;
    const int kind = cumo_hip_last_error(&msg);
    if (kind == 0) return 0;
    PyObject* r = PyObject_CallFunction(g_raise, "iy", kind, msg ? msg : "");
    if (r) {
        Py_DECREF(r);
        PyErr_SetString(PyExc_RuntimeError, "a latched error was not raised");
    }
    return -1;
}

// ---------------------------------------------------------------------------------------------------------------
// Buffer: one pool allocation, returned to the pool when the last view dies (reference: gen/tmpl/alloc_func.c:33-56)
// ---------------------------------------------------------------------------------------------------------------
struct Buffer {
    PyObject_HEAD
    void* ptr;
    Py_ssize_t nbytes;
};

extern PyTypeObject BufferType;

PyObject* buffer_adopt(void* ptr, Py_ssize_t nbytes) {
    Buffer* b = PyObject_New(Buffer, &BufferType);
    if (!b) return nullptr;
    b->ptr = ptr;
    b->nbytes = nbytes;
    return reinterpret_cast<PyObject*>(b);
}

PyObject* buffer_new(PyTypeObject*, PyObject* args, PyObject* kw) {
    static const char* names[] = {"nbytes", "ptr", nullptr};
    Py_ssize_t nbytes = 0;
    PyObject* given = Py_None;
    if (!PyArg_ParseTupleAndKeywords(args, kw, "n|O", const_cast<char**>(names), &nbytes, &given)) return nullptr;
    if (given != Py_None) {
        void* p = PyLong_AsVoidPtr(given);
        if (!p && PyErr_Occurred()) return nullptr;
        return buffer_adopt(p, nbytes);
    }
    void* p = nullptr;
    if (nbytes) {
        Py_BEGIN_ALLOW_THREADS
        p = cumo_cuda_runtime_malloc(static_cast<size_t>(nbytes));
        Py_END_ALLOW_THREADS
        if (raise_latched() < 0) return nullptr;
        if (!p) return PyErr_Format(PyExc_MemoryError, "allocation of %zd bytes failed", nbytes);
    }
    PyObject* b = buffer_adopt(p, nbytes);
    if (!b && p) cumo_cuda_runtime_free_no_raise(static_cast<char*>(p));
    return b;
}

void buffer_dealloc(PyObject* self) {
    Buffer* b = reinterpret_cast<Buffer*>(self);
    if (b->ptr) {
        void* p = b->ptr;
        b->ptr = nullptr;
        if (g_recording) {
            // released inside a recording: the recorded calls still name this memory
            PyObject *t, *v, *tb;
            PyErr_Fetch(&t, &v, &tb);
            PyObject* keep = PyObject_GetAttrString(g_recording, "keep");
            PyObject* again = keep ? buffer_adopt(p, b->nbytes) : nullptr;
            if (!again || PyList_Append(keep, again) < 0) PyErr_WriteUnraisable(self);
            Py_XDECREF(again);
            Py_XDECREF(keep);
            PyErr_Restore(t, v, tb);
        } else {
            Py_BEGIN_ALLOW_THREADS
            cumo_cuda_runtime_free_no_raise(static_cast<char*>(p));
            Py_END_ALLOW_THREADS
        }
    }
    Py_TYPE(self)->tp_free(self);
}

PyObject* buffer_ptr(PyObject* self, void*) {
    void* p = reinterpret_cast<Buffer*>(self)->ptr;
    if (!p) Py_RETURN_NONE;
    return PyLong_FromVoidPtr(p);
}

PyGetSetDef buffer_getset[] = {{"ptr", buffer_ptr, nullptr, "device address, None of an empty one", nullptr}, {}};
PyMemberDef buffer_members[] = {{"nbytes", T_PYSSIZET, offsetof(Buffer, nbytes), READONLY, nullptr}, {}};

PyTypeObject make_buffer_type() {
    PyTypeObject t = {PyVarObject_HEAD_INIT(nullptr, 0)};
    t.tp_name = "cumo_amd._native.Buffer";
    t.tp_basicsize = sizeof(Buffer);
    t.tp_flags = Py_TPFLAGS_DEFAULT;
    t.tp_doc = "One pool allocation; returned to the pool when the last view dies.";
    t.tp_new = buffer_new;
    t.tp_dealloc = buffer_dealloc;
    t.tp_getset = buffer_getset;
    t.tp_members = buffer_members;
    return t;
}
PyTypeObject BufferType = make_buffer_type();

// ---------------------------------------------------------------------------------------------------------------
// View: what narray.py's NArray derives from. Holds tuples of numbers and a Buffer, so no cycle can go through it.
// ---------------------------------------------------------------------------------------------------------------
struct View {
    PyObject_HEAD
    PyObject* shape;
    PyObject* strides;
    PyObject* buf;
    Py_ssize_t offset;
    int code;
};

extern PyTypeObject ViewType;

inline View* as_view(PyObject* o) { return PyObject_TypeCheck(o, &ViewType) ? reinterpret_cast<View*>(o) : nullptr; }

PyObject* view_new(PyTypeObject* type, PyObject*, PyObject*) {
    PyObject* code = PyObject_GetAttrString(reinterpret_cast<PyObject*>(type), "type_code");
    if (!code) return nullptr;
    const long c = PyLong_AsLong(code);
    Py_DECREF(code);
    if (c == -1 && PyErr_Occurred()) return nullptr;
    PyObject* self = type->tp_alloc(type, 0);
    if (self) reinterpret_cast<View*>(self)->code = static_cast<int>(c);
    return self;
}

void view_dealloc(PyObject* self) {
    View* v = reinterpret_cast<View*>(self);
    Py_CLEAR(v->buf);
    Py_CLEAR(v->shape);
    Py_CLEAR(v->strides);
    Py_TYPE(self)->tp_free(self);
}

PyObject* view_get(PyObject* self, void* at) {
    PyObject* o = *reinterpret_cast<PyObject**>(reinterpret_cast<char*>(self) + reinterpret_cast<Py_ssize_t>(at));
    if (!o) {
        PyErr_SetString(PyExc_AttributeError, "the array has not been set up");
        return nullptr;
    }
    Py_INCREF(o);
    return o;
}

int view_set(PyObject* self, PyObject* value, void* at) {
    PyTypeObject* want = reinterpret_cast<Py_ssize_t>(at) == offsetof(View, buf) ? &BufferType : &PyTuple_Type;
    if (!value || !PyObject_TypeCheck(value, want)) {
        PyErr_Format(PyExc_TypeError, "expected %s", want->tp_name);
        return -1;
    }
    PyObject** slot = reinterpret_cast<PyObject**>(reinterpret_cast<char*>(self) + reinterpret_cast<Py_ssize_t>(at));
    PyObject* old = *slot;
    Py_INCREF(value);
    *slot = value;
    Py_XDECREF(old);
    return 0;
}

PyObject* view_ptr(PyObject* self, PyObject*) {
    View* v = reinterpret_cast<View*>(self);
    if (!v->buf) return view_get(self, reinterpret_cast<void*>(offsetof(View, buf)));
    return PyLong_FromSsize_t(reinterpret_cast<Py_ssize_t>(reinterpret_cast<Buffer*>(v->buf)->ptr) + v->offset);
}

PyGetSetDef view_getset[] = {
    {"shape", view_get, view_set, nullptr, reinterpret_cast<void*>(offsetof(View, shape))},
    {"_strides", view_get, view_set, nullptr, reinterpret_cast<void*>(offsetof(View, strides))},
    {"_buf", view_get, view_set, nullptr, reinterpret_cast<void*>(offsetof(View, buf))},
    {}};
PyMemberDef view_members[] = {{"_offset", T_PYSSIZET, offsetof(View, offset), 0, nullptr}, {}};
PyMethodDef view_methods[] = {{"_ptr", view_ptr, METH_NOARGS, "address of the first element"}, {}};

PyTypeObject make_view_type() {
    PyTypeObject t = {PyVarObject_HEAD_INIT(nullptr, 0)};
    t.tp_name = "cumo_amd._native.View";
    t.tp_basicsize = sizeof(View);
    t.tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_BASETYPE;
    t.tp_doc = "shape, strides and offset into a Buffer; strides and offset are bytes (bits for Bit).";
    t.tp_new = view_new;
    t.tp_dealloc = view_dealloc;
    t.tp_getset = view_getset;
    t.tp_members = view_members;
    t.tp_methods = view_methods;
    return t;
}
PyTypeObject ViewType = make_view_type();

// the view as the library's descriptor; -1 with an exception set
int describe(const View* v, Desc* d) {
    if (!v->shape || !v->strides || !v->buf) {
        PyErr_SetString(PyExc_AttributeError, "the array has not been set up");
        return -1;
    }
    const Py_ssize_t n = PyTuple_GET_SIZE(v->shape);
    if (n > CUMO_NA_MAX_DIMENSION || PyTuple_GET_SIZE(v->strides) < n) {
        PyErr_SetString(PyExc_ValueError, "too many dimensions");
        return -1;
    }
    std::memset(d, 0, sizeof(*d));
    d->type = v->code;
    d->ndim = static_cast<int>(n);
    d->ptr = static_cast<char*>(reinterpret_cast<Buffer*>(v->buf)->ptr);
    d->offset = v->offset;
    for (Py_ssize_t k = 0; k < n; k++) {
        d->shape[k] = PyLong_AsSize_t(PyTuple_GET_ITEM(v->shape, k));
        d->stride[k] = PyLong_AsSsize_t(PyTuple_GET_ITEM(v->strides, k));
    }
    return PyErr_Occurred() ? -1 : 0;
}

void release(Desc* d) {
    if (d->ptr) cumo_cuda_runtime_free_no_raise(static_cast<char*>(d->ptr));
    d->ptr = nullptr;
}

// the array of a result that the library allocated; takes its memory in every case
PyObject* wrap(Desc* d) {
    PyObject* cls = d->type >= 0 && d->type < 8 ? g_class[d->type] : nullptr;
    if (!cls) {
        release(d);
        PyErr_SetString(PyExc_TypeError, "a result of an unknown type");
        return nullptr;
    }
    size_t n = 1;
    for (int k = 0; k < d->ndim; k++) n *= d->shape[k];
    PyObject* buf = buffer_adopt(d->ptr, static_cast<Py_ssize_t>(cumo_hip_na_storage_bytes(d->type, n)));
    if (!buf) {
        release(d);
        return nullptr;
    }
    PyTypeObject* type = reinterpret_cast<PyTypeObject*>(cls);
    PyObject* self = type->tp_alloc(type, 0);
    PyObject* shape = PyTuple_New(d->ndim);
    PyObject* strides = PyTuple_New(d->ndim);
    if (!self || !shape || !strides) {
        Py_XDECREF(self);
        Py_XDECREF(shape);
        Py_XDECREF(strides);
        Py_DECREF(buf);
        return nullptr;
    }
    View* v = reinterpret_cast<View*>(self);
    v->code = d->type;
    v->buf = buf;
    v->shape = shape;
    v->strides = strides;
    // a contiguous array: the unit is an element's bytes, a bit for Bit
    static const Py_ssize_t unit[8] = {4, 8, 4, 8, 8, 1, 0, 0};
    Py_ssize_t st = unit[d->type];
    for (int k = d->ndim - 1; k >= 0; k--) {
        PyObject* len = PyLong_FromSize_t(d->shape[k]);
        PyObject* step = PyLong_FromSsize_t(st);
        PyTuple_SET_ITEM(shape, k, len);
        PyTuple_SET_ITEM(strides, k, step);
        if (!len || !step) {
            Py_DECREF(self);
            return nullptr;
        }
        st *= static_cast<Py_ssize_t>(d->shape[k]);
    }
    return self;
}

// Calls f (which queues the work and may wait for it) without the interpreter's lock, then answers with the array of
// the result, or the tuple of two.
template <typename F>
PyObject* run(Desc* z, int nz, F f) {
    for (int k = 0; k < nz; k++) std::memset(&z[k], 0, sizeof(Desc));
    Py_BEGIN_ALLOW_THREADS
    f();
    Py_END_ALLOW_THREADS
    if (raise_latched() < 0) {
        for (int k = 0; k < nz; k++) release(&z[k]);
        return nullptr;
    }
    PyObject* first = wrap(&z[0]);
    if (nz == 1) return first;
    PyObject* second = wrap(&z[1]);
    PyObject* both = first && second ? PyTuple_Pack(2, first, second) : nullptr;
    Py_XDECREF(first);
    Py_XDECREF(second);
    return both;
}

inline bool numeric(const View* v) { return v->code >= 0 && v->code <= 2; }
inline bool is_bit(const View* v) { return v->code == 5; }

// a number as it rides in a launch: exact float and int; false for everything else
bool plain_number(PyObject* o, double* value) {
    if (PyFloat_CheckExact(o)) {
        *value = PyFloat_AS_DOUBLE(o);
        return true;
    }
    if (PyLong_CheckExact(o)) {
        *value = PyLong_AsDouble(o);
        if (*value == -1.0 && PyErr_Occurred()) {
            PyErr_Clear();  // the general form raises it
            return false;
        }
        return true;
    }
    return false;
}

// axis: None, an int or a tuple of ints in range; false for everything else (the general form takes or refuses it)
bool plain_axis(PyObject* axis, Py_ssize_t ndim, unsigned* mask) {
    *mask = 0;
    if (axis == Py_None) return true;
    const bool many = PyTuple_CheckExact(axis);
    const Py_ssize_t n = many ? PyTuple_GET_SIZE(axis) : 1;
    for (Py_ssize_t k = 0; k < n; k++) {
        PyObject* o = many ? PyTuple_GET_ITEM(axis, k) : axis;
        if (!PyLong_CheckExact(o)) return false;
        int over = 0;
        const long a = PyLong_AsLongAndOverflow(o, &over);
        if (over || a < -ndim || a >= ndim) return false;
        *mask |= 1u << (a < 0 ? a + ndim : a);
    }
    return true;
}

inline Py_ssize_t ndim_of(const View* v) { return v->shape ? PyTuple_GET_SIZE(v->shape) : 0; }

PyObject* general(PyObject* self, const char* method, PyObject* const* args, Py_ssize_t nargs) {
    PyObject* f = PyObject_GetAttrString(self, method);
    if (!f) return nullptr;
    PyObject* r = PyObject_Vectorcall(f, args, static_cast<size_t>(nargs), nullptr);
    Py_DECREF(f);
    return r;
}

bool arity(Py_ssize_t have, Py_ssize_t want) {
    if (have == want) return true;
    PyErr_Format(PyExc_TypeError, "expected %zd arguments, got %zd", want, have);
    return false;
}

// ---------------------------------------------------------------------------------------------------------------
// the calls; the first argument is the array whose Python method takes the general form
// ---------------------------------------------------------------------------------------------------------------

// (self, other, op, scalar_is_left): + - * / and the rest that answer in the wider of the two types
PyObject* na_binary(PyObject*, PyObject* const* a, Py_ssize_t n) {
    if (!arity(n, 4)) return nullptr;
    const View* x = as_view(a[0]);
    const char* op = PyUnicode_AsUTF8(a[2]);
    if (!op) return nullptr;
    const bool left = a[3] == Py_True;
    Desc dx, dy, z;
    double sv;
    if (x && numeric(x) && !g_recording) {
        if (const View* y = as_view(a[1])) {
            if (numeric(y)) {
                if (describe(left ? y : x, &dx) < 0 || describe(left ? x : y, &dy) < 0) return nullptr;
                return run(&z, 1, [&] { cumo_hip_na_binary(op, &dx, &dy, &z); });
            }
        } else if (plain_number(a[1], &sv)) {
            // a Float meeting Int32 moves the array to DFloat: the library does it for these four, the general
            // form for the others
            const bool widens = x->code == 2 && PyFloat_CheckExact(a[1]);
            const bool four = !std::strcmp(op, "add") || !std::strcmp(op, "sub") || !std::strcmp(op, "mul") || !std::strcmp(op, "div");
            if (!widens || four) {
                if (describe(x, &dx) < 0) return nullptr;
                return run(&z, 1, [&] {
                    if (widens) cumo_hip_na_binary_fs(op, &dx, sv, left, &z);
                    else cumo_hip_na_binary_s(op, &dx, sv, left, &z);
                });
            }
        }
    }
    return general(a[0], "_binary", a + 1, 3);
}

// (self, other, op): comparisons into Bit
PyObject* na_compare(PyObject*, PyObject* const* a, Py_ssize_t n) {
    if (!arity(n, 3)) return nullptr;
    const View* x = as_view(a[0]);
    const char* op = PyUnicode_AsUTF8(a[2]);
    if (!op) return nullptr;
    Desc dx, dy, z;
    double sv;
    if (x && numeric(x) && !g_recording) {
        if (const View* y = as_view(a[1])) {
            if (numeric(y)) {
                if (describe(x, &dx) < 0 || describe(y, &dy) < 0) return nullptr;
                return run(&z, 1, [&] { cumo_hip_na_compare(op, &dx, &dy, &z); });
            }
        } else if (plain_number(a[1], &sv) && !(x->code == 2 && PyFloat_CheckExact(a[1]))) {
            if (describe(x, &dx) < 0) return nullptr;
            return run(&z, 1, [&] { cumo_hip_na_compare_s(op, &dx, sv, 0, &z); });
        }
    }
    return general(a[0], "_compare", a + 1, 2);
}

// (self, op)
PyObject* na_unary(PyObject*, PyObject* const* a, Py_ssize_t n) {
    if (!arity(n, 2)) return nullptr;
    const View* x = as_view(a[0]);
    const char* op = PyUnicode_AsUTF8(a[1]);
    if (!op) return nullptr;
    if (!x || !numeric(x) || g_recording) return general(a[0], "_unary", a + 1, 1);
    Desc dx, z;
    if (describe(x, &dx) < 0) return nullptr;
    return run(&z, 1, [&] { cumo_hip_na_unary(op, &dx, &z); });
}

// (name, x): NMath's functions of one argument
PyObject* na_math(PyObject*, PyObject* const* a, Py_ssize_t n) {
    if (!arity(n, 2)) return nullptr;
    const char* op = PyUnicode_AsUTF8(a[0]);
    if (!op) return nullptr;
    const View* x = as_view(a[1]);
    if (!x || !numeric(x) || g_recording) return general(g_nmath, "_call1", a, 2);
    Desc dx, z;
    if (describe(x, &dx) < 0) return nullptr;
    return run(&z, 1, [&] { cumo_hip_na_math(op, &dx, &z); });
}

// (self, op, axis, keepdims, nan); minmax answers a tuple of two
PyObject* na_reduce(PyObject*, PyObject* const* a, Py_ssize_t n) {
    if (!arity(n, 5)) return nullptr;
    const View* x = as_view(a[0]);
    const char* op = PyUnicode_AsUTF8(a[1]);
    if (!op) return nullptr;
    unsigned mask = 0;
    if (!x || !numeric(x) || g_recording || !plain_axis(a[2], ndim_of(x), &mask)) return general(a[0], "_reduce", a + 1, 4);
    const int keep = PyObject_IsTrue(a[3]), nan = PyObject_IsTrue(a[4]);
    if (keep < 0 || nan < 0) return nullptr;
    const bool two = !std::strcmp(op, "minmax");
    Desc dx, z[2];
    if (describe(x, &dx) < 0) return nullptr;
    return run(z, two ? 2 : 1, [&] { cumo_hip_na_reduce(op, &dx, mask, keep, nan, &z[0], two ? &z[1] : nullptr); });
}

// (self, other, axis, keepdims, nan)
PyObject* na_mulsum(PyObject*, PyObject* const* a, Py_ssize_t n) {
    if (!arity(n, 5)) return nullptr;
    const View *x = as_view(a[0]), *y = as_view(a[1]);
    unsigned mask = 0;
    if (!x || !y || !numeric(x) || !numeric(y) || g_recording ||
        !plain_axis(a[2], ndim_of(x) > ndim_of(y) ? ndim_of(x) : ndim_of(y), &mask))
        return general(a[0], "_mulsum", a + 1, 4);
    const int keep = PyObject_IsTrue(a[3]), nan = PyObject_IsTrue(a[4]);
    if (keep < 0 || nan < 0) return nullptr;
    Desc dx, dy, z;
    if (describe(x, &dx) < 0 || describe(y, &dy) < 0) return nullptr;
    return run(&z, 1, [&] { cumo_hip_na_mulsum(&dx, &dy, mask, keep, nan, &z); });
}

// (self, op, axis, nan)
PyObject* na_cum(PyObject*, PyObject* const* a, Py_ssize_t n) {
    if (!arity(n, 4)) return nullptr;
    const View* x = as_view(a[0]);
    const char* op = PyUnicode_AsUTF8(a[1]);
    if (!op) return nullptr;
    unsigned mask = 0;
    if (!x || !numeric(x) || g_recording || !plain_axis(a[2], ndim_of(x), &mask)) return general(a[0], "_cum", a + 1, 3);
    const int nan = PyObject_IsTrue(a[3]);
    if (nan < 0) return nullptr;
    Desc dx, z;
    if (describe(x, &dx) < 0) return nullptr;
    return run(&z, 1, [&] { cumo_hip_na_cum(op, &dx, mask, nan, &z); });
}

// (self, other, op): logic on two Bit arrays
PyObject* na_bit_binary(PyObject*, PyObject* const* a, Py_ssize_t n) {
    if (!arity(n, 3)) return nullptr;
    const View *x = as_view(a[0]), *y = as_view(a[1]);
    const char* op = PyUnicode_AsUTF8(a[2]);
    if (!op) return nullptr;
    if (!x || !y || !is_bit(x) || !is_bit(y) || g_recording) return general(a[0], "_bit_op2", a + 1, 2);
    Desc dx, dy, z;
    if (describe(x, &dx) < 0 || describe(y, &dy) < 0) return nullptr;
    return run(&z, 1, [&] { cumo_hip_na_bit_binary(op, &dx, &dy, &z); });
}

// (self, count_false, axis, keepdims)
PyObject* na_bit_count(PyObject*, PyObject* const* a, Py_ssize_t n) {
    if (!arity(n, 4)) return nullptr;
    const View* x = as_view(a[0]);
    unsigned mask = 0;
    if (!x || !is_bit(x) || g_recording || !plain_axis(a[2], ndim_of(x), &mask)) return general(a[0], "_count", a + 1, 3);
    Desc dx, z;
    if (describe(x, &dx) < 0) return nullptr;
    for (int k = 0; k < dx.ndim; k++)
        if (dx.shape[k] == 0) return general(a[0], "_count", a + 1, 3);  // an empty array answers a number
    const int keep = PyObject_IsTrue(a[3]);
    if (keep < 0) return nullptr;
    const int count_false = a[1] == Py_True;
    return run(&z, 1, [&] { cumo_hip_na_bit_count(&dx, mask, keep, count_false, &z); });
}

// (self, positions): self[positions] for a one-dimensional array of 64-bit positions in the first dimension; None where the general
// form answers (other kinds of positions, positions out of range, empty results; arrays of a class derived from the registered
// ones, whose selections are of that class). x[2048 rows] 27.4 -> 8.5 us of the caller's time.
PyObject* na_take(PyObject*, PyObject* const* a, Py_ssize_t n) {
    if (!arity(n, 2)) return nullptr;
    const View* x = as_view(a[0]);
    if (!x || x->code < 0 || x->code > 4 || g_recording || ndim_of(x) < 1) Py_RETURN_NONE;
    if (reinterpret_cast<PyObject*>(Py_TYPE(a[0])) != g_class[x->code]) Py_RETURN_NONE;
    static const size_t element[5] = {4, 8, 4, 8, 8};
    const size_t elmsz = element[x->code];
    Desc dx, z;
    if (describe(x, &dx) < 0) return nullptr;
    size_t row = elmsz, bytes;
    for (int k = 1; k < dx.ndim; k++) row *= dx.shape[k];
    Py_buffer b;
    if (PyObject_GetBuffer(a[1], &b, PyBUF_FORMAT | PyBUF_ND) < 0) {
        PyErr_Clear();   // (not contiguous, say)
        Py_RETURN_NONE;
    }
    const size_t count = static_cast<size_t>(b.len) / sizeof(int64_t);
    bool taken = b.ndim == 1 && b.itemsize == sizeof(int64_t) && b.format && (!std::strcmp(b.format, "l") || !std::strcmp(b.format, "q")) &&
                 reinterpret_cast<uintptr_t>(b.buf) % alignof(int64_t) == 0 && count > 0 && row > 0 && dx.shape[0] > 0 &&
                 !__builtin_mul_overflow(row, count, &bytes);
    std::unique_ptr<size_t[]> pos(taken ? new (std::nothrow) size_t[count] : nullptr);
    taken = taken && pos;
    if (taken) {
        // a negative position counts from the end
        const int64_t* from = static_cast<const int64_t*>(b.buf);
        const int64_t len = static_cast<int64_t>(dx.shape[0]);
        for (size_t i = 0; i < count; i++) {
            const int64_t k = from[i] < 0 ? from[i] + len : from[i];
            taken = taken && k >= 0 && k < len;
            pos[i] = static_cast<size_t>(k);
        }
    }
    PyBuffer_Release(&b);
    if (!taken) Py_RETURN_NONE;
    return run(&z, 1, [&] {
        const ssize_t st = dx.stride[0];
        const size_t last = dx.shape[0] - 1;
        size_t* off = reinterpret_cast<size_t*>(cumo_cuda_runtime_malloc(count * sizeof(size_t)));
        char* out = off ? reinterpret_cast<char*>(cumo_cuda_runtime_malloc(bytes)) : nullptr;
        if (out) {
            z.type = dx.type;
            z.ndim = dx.ndim;
            z.ptr = out;
            cumo_na_iarray_stridx_t view;
            cumo_na_indexer_t ix;
            std::memset(&view, 0, sizeof(view));
            std::memset(&ix, 0, sizeof(ix));
            ix.ndim = dx.ndim;
            ix.total_size = bytes / elmsz;
            for (int k = 0; k < dx.ndim; k++) {
                z.shape[k] = ix.shape[k] = k == 0 ? count : dx.shape[k];
                CUMO_SDX_SET_STRIDE(view.stridx[k], dx.stride[k]);
            }
            // (a reversed dimension counts from its far end)
            CUMO_SDX_SET_INDEX(view.stridx[0], off);
            view.ptr = static_cast<char*>(dx.ptr) + dx.offset + (st < 0 ? st * static_cast<ssize_t>(last) : 0);
            if (cumo_hip_index_from_host(off, pos.get(), count, st < 0 ? -st : st, st < 0 ? 1 : 0, last) == CUMO_HIP_OK)
                cumo_ndloop_copy_to_buffer_kernel_launch(&view, &ix, out, elmsz);
        }
        // (stream-ordered: whoever gets it next can only touch it from later work)
        if (off) cumo_cuda_runtime_free_no_raise(reinterpret_cast<char*>(off));
    });
}

// ---------------------------------------------------------------------------------------------------------------
// views
// ---------------------------------------------------------------------------------------------------------------

// (x, key): x[key] for a key of whole numbers, slices and True (the whole dimension), one or a tuple of them. None: a key that
// the Python form answers (index arrays, an ellipsis, numpy numbers, positions out of range, too many of them) and arrays of a
// derived class. x[::3] 2.3 us of the caller's time -> 0.13, x.T[:, ::2] 2.3 -> 0.16.
PyObject* na_window(PyObject*, PyObject* const* a, Py_ssize_t n) {
    if (!arity(n, 2)) return nullptr;
    const View* x = as_view(a[0]);
    if (!x || x->code < 0 || x->code > 7 || !x->shape || !x->strides || !x->buf) Py_RETURN_NONE;
    PyTypeObject* type = Py_TYPE(a[0]);
    if (reinterpret_cast<PyObject*>(type) != g_class[x->code]) Py_RETURN_NONE;
    const Py_ssize_t nd = PyTuple_GET_SIZE(x->shape);
    const bool many = PyTuple_CheckExact(a[1]);
    const Py_ssize_t given = many ? PyTuple_GET_SIZE(a[1]) : 1;
    if (given > nd || nd > CUMO_NA_MAX_DIMENSION || PyTuple_GET_SIZE(x->strides) != nd) Py_RETURN_NONE;
    // All that is asked of x and all that may send the key elsewhere comes first: a slice's numbers may be objects whose __index__
    // runs, once, and may set x anew.
    Py_ssize_t shape[CUMO_NA_MAX_DIMENSION], strides[CUMO_NA_MAX_DIMENSION], offset = x->offset;
    PyObject* part[CUMO_NA_MAX_DIMENSION];
    for (Py_ssize_t d = 0; d < nd; d++) {
        shape[d] = PyLong_AsSsize_t(PyTuple_GET_ITEM(x->shape, d));
        strides[d] = PyLong_AsSsize_t(PyTuple_GET_ITEM(x->strides, d));
        if ((shape[d] == -1 || strides[d] == -1) && PyErr_Occurred()) return nullptr;
        PyObject* k = part[d] = d >= given ? Py_True : many ? PyTuple_GET_ITEM(a[1], d) : a[1];
        if (PyLong_CheckExact(k)) {
            const Py_ssize_t at = PyLong_AsSsize_t(k);
            if (at == -1 && PyErr_Occurred()) {
                PyErr_Clear();
                Py_RETURN_NONE;
            }
            if (at < -shape[d] || at >= shape[d]) Py_RETURN_NONE;
        } else if (k != Py_True && !PySlice_Check(k)) {
            Py_RETURN_NONE;
        }
    }
    Py_ssize_t left = 0;   // (never past d: what stands there has been read)
    for (Py_ssize_t d = 0; d < nd; d++) {
        const Py_ssize_t len = shape[d], step = strides[d];
        if (part[d] == Py_True) {
            shape[left] = len;
            strides[left++] = step;
        } else if (PyLong_CheckExact(part[d])) {
            const Py_ssize_t at = PyLong_AsSsize_t(part[d]);
            offset += (at < 0 ? at + len : at) * step;
        } else {
            Py_ssize_t from, to, by;
            if (PySlice_Unpack(part[d], &from, &to, &by) < 0) return nullptr;
            shape[left] = PySlice_AdjustIndices(len, &from, &to, by);
            offset += from * step;
            if (by == PY_SSIZE_T_MAX || by == -PY_SSIZE_T_MAX || __builtin_mul_overflow(step, by, &strides[left++])) Py_RETURN_NONE;
        }
    }
    PyObject* self = type->tp_alloc(type, 0);
    PyObject* new_shape = PyTuple_New(left);
    PyObject* new_strides = PyTuple_New(left);
    bool ok = self && new_shape && new_strides;
    for (Py_ssize_t d = 0; ok && d < left; d++) {
        PyObject* len = PyLong_FromSsize_t(shape[d]);
        PyObject* step = PyLong_FromSsize_t(strides[d]);
        PyTuple_SET_ITEM(new_shape, d, len);
        PyTuple_SET_ITEM(new_strides, d, step);
        ok = len && step;
    }
    if (!ok) {
        Py_XDECREF(self);
        Py_XDECREF(new_shape);
        Py_XDECREF(new_strides);
        return nullptr;
    }
    View* v = reinterpret_cast<View*>(self);
    v->code = x->code;
    v->buf = x->buf;
    Py_INCREF(v->buf);
    v->shape = new_shape;
    v->strides = new_strides;
    v->offset = offset;
    return self;
}

// ---------------------------------------------------------------------------------------------------------------
// set-up
// ---------------------------------------------------------------------------------------------------------------

// (classes by type code, the function that raises a latched error, NMath)
PyObject* setup(PyObject*, PyObject* args) {
    PyObject *classes, *raise, *nmath;
    if (!PyArg_ParseTuple(args, "O!OO", &PyDict_Type, &classes, &raise, &nmath)) return nullptr;
    Py_ssize_t at = 0;
    PyObject *key, *cls;
    while (PyDict_Next(classes, &at, &key, &cls)) {
        const long code = PyLong_AsLong(key);
        if (code < 0 || code >= 8 || !PyType_Check(cls) || !PyType_IsSubtype(reinterpret_cast<PyTypeObject*>(cls), &ViewType)) {
            PyErr_SetString(PyExc_TypeError, "classes by type code");
            return nullptr;
        }
        Py_INCREF(cls);
        g_class[code] = cls;
    }
    Py_INCREF(raise);
    g_raise = raise;
    Py_INCREF(nmath);
    g_nmath = nmath;
    Py_RETURN_NONE;
}

PyObject* set_recording(PyObject*, PyObject* rec) {
    PyObject* old = g_recording;
    if (rec == Py_None) {
        g_recording = nullptr;
    } else {
        Py_INCREF(rec);
        g_recording = rec;
    }
    Py_XDECREF(old);
    Py_RETURN_NONE;
}

#define CALL(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(na_##name)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {CALL(binary), CALL(compare), CALL(unary), CALL(math), CALL(reduce), CALL(mulsum), CALL(cum), CALL(bit_binary),
                         CALL(bit_count), CALL(take), CALL(window), {"setup", setup, METH_VARARGS, nullptr}, {"set_recording", set_recording, METH_O, nullptr}, {}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "cumo_amd._native", "Buffers, views and calls of the array classes.", -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit__native(void) {
    if (PyType_Ready(&BufferType) < 0 || PyType_Ready(&ViewType) < 0) return nullptr;
    PyObject* m = PyModule_Create(&module);
    if (!m) return nullptr;
    Py_INCREF(&BufferType);
    Py_INCREF(&ViewType);
    if (PyModule_AddObject(m, "Buffer", reinterpret_cast<PyObject*>(&BufferType)) < 0 ||
        PyModule_AddObject(m, "View", reinterpret_cast<PyObject*>(&ViewType)) < 0) {
        Py_DECREF(m);
        return nullptr;
    }
    return m;
}
