// The short way from Python into the C ABI, for arguments that are what they usually are: `Slice` and `GroupedShape` objects
// (not subclasses) of plain non-negative ints, plain int counts, float scales, ctypes tables. A function here either makes the
// call that loadngo_amd/compute.py would have made through ctypes and gives its result, or gives None without having called
// anything, and compute.py goes its own way, which converts, refuses and reports as ever. Nothing is kept between calls but the
// addresses of the library's functions and where the two classes keep their fields.
//
// Recording is most of what a small batch costs the host: a token through 24 attention blocks (97 dispatches, 578 slices) is
// recorded in 54 us through here, 300 through ctypes.
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <structmember.h>

#include <climits>
#include <initializer_list>

#include "../../include/lng_hip.h"

namespace {

struct {
    decltype(&lng_hip_batch) batch;
    decltype(&lng_hip_batch_commit) batch_commit;
    decltype(&lng_hip_batch_wait) batch_wait;
    decltype(&lng_hip_batch_drop) batch_drop;
    decltype(&lng_hip_attention_grouped) attention_grouped;
    decltype(&lng_hip_attention_grouped_tiled) attention_grouped_tiled;
    decltype(&lng_hip_attention_grouped_static) attention_grouped_static;
    decltype(&lng_hip_attention_decode_batched) attention_decode_batched;
    decltype(&lng_hip_copy_rows) copy_rows;
    decltype(&lng_hip_rmsnorm_rows) rmsnorm_rows;
    decltype(&lng_hip_add_rows) add_rows;
    decltype(&lng_hip_prepare_attention) prepare_attention;
    decltype(&lng_hip_gemm_q8_0) gemm_q8_0;
    decltype(&lng_hip_gemm_q8_0_tiled) gemm_q8_0_tiled;
    decltype(&lng_hip_gemm_q8_0_bf16) gemm_q8_0_bf16;
    decltype(&lng_hip_gemm_q8_0_many) gemm_q8_0_many;
    decltype(&lng_hip_gemm_q8_0_many_normed) gemm_q8_0_many_normed;
    decltype(&lng_hip_gemm_q8_0_residual) gemm_q8_0_residual;
} g_lib;
PyTypeObject *g_slice, *g_shape, *g_item, *g_prepare_item;
Py_ssize_t g_slice_at[3], g_shape_at[8];
PyObject *g_names[7], *g_element; // q, k, v, table, q_out, k_cache, v_cache; _type_

// A plain int in 0 .. 2^64 - 1.
bool u64_of(PyObject *o, uint64_t *out) {
    if (!o || !PyLong_CheckExact(o)) return false;
    const unsigned long long v = PyLong_AsUnsignedLongLong(o);
    if (v == ~0ull && PyErr_Occurred()) {
        PyErr_Clear();
        return false;
    }
    *out = v;
    return true;
}

bool int_of(PyObject *o, int *out) {
    uint64_t v;
    if (!u64_of(o, &v) || v > INT_MAX) return false;
    *out = (int)v;
    return true;
}

bool float_of(PyObject *o, float *out) {
    if (!PyFloat_CheckExact(o)) return false;
    *out = (float)PyFloat_AS_DOUBLE(o);
    return true;
}

bool pointer_of(PyObject *o, void **out) { // a handle or an address
    uint64_t v;
    if (!u64_of(o, &v)) return false;
    *out = (void *)(uintptr_t)v;
    return true;
}

bool handle_of(PyObject *o, void **out) { return pointer_of(o, out) && *out; }

PyObject *field(PyObject *o, Py_ssize_t at) { return *(PyObject **)((char *)o + at); } // NULL where it was never set

bool slice_of(PyObject *o, lng_slice *s) {
    return Py_TYPE(o) == g_slice && u64_of(field(o, g_slice_at[0]), &s->buffer) && u64_of(field(o, g_slice_at[1]), &s->offset) &&
           u64_of(field(o, g_slice_at[2]), &s->len);
}

bool shape_of(PyObject *o, lng_grouped_shape *s) {
    if (Py_TYPE(o) != g_shape) return false;
    uint64_t *const into[7] = {&s->t, &s->start, &s->heads, &s->kv_heads, &s->dim, &s->window, &s->slots};
    for (int i = 0; i < 7; ++i) {
        if (!u64_of(field(o, g_shape_at[i]), into[i])) return false;
    }
    PyObject *scale = field(o, g_shape_at[7]);
    return scale && float_of(scale, &s->scale);
}

// (a, b) as a tuple or a list
bool two_of(PyObject *o, PyObject **a, PyObject **b) {
    if (!(PyTuple_CheckExact(o) || PyList_CheckExact(o)) || PySequence_Fast_GET_SIZE(o) != 2) return false;
    *a = PySequence_Fast_GET_ITEM(o, 0);
    *b = PySequence_Fast_GET_ITEM(o, 1);
    return true;
}

bool matrix_of(PyObject *o, lng_slice *codes, lng_slice *scales) {
    PyObject *a, *b;
    return two_of(o, &a, &b) && slice_of(a, codes) && slice_of(b, scales);
}

// A ctypes array of `element`s, for the time of a call.
struct Table {
    Py_buffer view{};
    bool held = false;
    bool of(PyObject *o, PyTypeObject *element) {
        PyObject *type = PyObject_GetAttr((PyObject *)Py_TYPE(o), g_element);
        if (!type) PyErr_Clear();
        const bool ours = type == (PyObject *)element;
        Py_XDECREF(type);
        if (!ours) return false;
        held = PyObject_GetBuffer(o, &view, PyBUF_SIMPLE) == 0;
        if (!held) PyErr_Clear();
        return held;
    }
    ~Table() {
        if (held) PyBuffer_Release(&view);
    }
};

template <typename F> PyObject *call(F f) { // the library may wait for other threads
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = f();
    Py_END_ALLOW_THREADS
    return PyLong_FromLong(rc);
}

#define ARGUMENTS(count) \
    if (n_args != (count)) Py_RETURN_NONE; \
    (void)0
typedef PyObject *const *Args;

PyObject *batch(PyObject *, Args a, Py_ssize_t n_args) { // gpu, [handles] -> a handle, or a negative status
    ARGUMENTS(2);
    void *gpu;
    if (!handle_of(a[0], &gpu) || !PyList_CheckExact(a[1])) Py_RETURN_NONE;
    const Py_ssize_t n = PyList_GET_SIZE(a[1]);
    lng_buffer *buffers[64];
    if (n > 64) Py_RETURN_NONE;
    for (Py_ssize_t i = 0; i < n; ++i) {
        if (!handle_of(PyList_GET_ITEM(a[1], i), (void **)&buffers[i])) Py_RETURN_NONE;
    }
    lng_batch *b = nullptr;
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = g_lib.batch((lng_gpu *)gpu, buffers, (size_t)n, &b);
    Py_END_ALLOW_THREADS
    return rc ? PyLong_FromLong(rc) : PyLong_FromVoidPtr(b);
}

PyObject *commit(PyObject *, Args a, Py_ssize_t n_args) { // without a callback
    ARGUMENTS(1);
    void *b;
    if (!handle_of(a[0], &b)) Py_RETURN_NONE;
    return call([&] { return g_lib.batch_commit((lng_batch *)b, nullptr, nullptr); });
}

PyObject *wait(PyObject *, Args a, Py_ssize_t n_args) { // seconds, or a negative status
    ARGUMENTS(1);
    void *b;
    if (!handle_of(a[0], &b)) Py_RETURN_NONE;
    double seconds = 0.0;
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = g_lib.batch_wait((lng_batch *)b, &seconds);
    Py_END_ALLOW_THREADS
    return rc ? PyLong_FromLong(rc) : PyFloat_FromDouble(seconds);
}

PyObject *drop(PyObject *, Args a, Py_ssize_t n_args) {
    ARGUMENTS(1);
    void *b;
    if (!handle_of(a[0], &b)) Py_RETURN_NONE;
    return call([&] { return g_lib.batch_drop((lng_batch *)b), 0; });
}

PyObject *attention(Args a, Py_ssize_t n_args, decltype(&lng_hip_attention_grouped) f) { // batch, q, k, v, out, sinks or None, shape, dtype
    ARGUMENTS(8);
    void *b;
    lng_slice q, k, v, out, sinks;
    lng_grouped_shape shape;
    int dtype;
    if (!handle_of(a[0], &b) || !slice_of(a[1], &q) || !slice_of(a[2], &k) || !slice_of(a[3], &v) || !slice_of(a[4], &out) ||
        (a[5] != Py_None && !slice_of(a[5], &sinks)) || !shape_of(a[6], &shape) || !int_of(a[7], &dtype)) Py_RETURN_NONE;
    const lng_slice *s = a[5] == Py_None ? nullptr : &sinks;
    return call([&] { return f((lng_batch *)b, q, k, v, out, s, &shape, dtype); });
}
PyObject *attention_grouped(PyObject *, Args a, Py_ssize_t n) { return attention(a, n, g_lib.attention_grouped); }
PyObject *attention_grouped_tiled(PyObject *, Args a, Py_ssize_t n) { return attention(a, n, g_lib.attention_grouped_tiled); }

PyObject *attention_grouped_static(PyObject *, Args a, Py_ssize_t n_args) { // gpu, stream or None, q, k, v, out, sinks or None, shape, dtype
    ARGUMENTS(9);
    void *gpu, *stream = nullptr, *q, *k, *v, *out, *sinks = nullptr;
    lng_grouped_shape shape;
    int dtype;
    if (!handle_of(a[0], &gpu) || (a[1] != Py_None && !pointer_of(a[1], &stream)) || !pointer_of(a[2], &q) || !pointer_of(a[3], &k) ||
        !pointer_of(a[4], &v) || !pointer_of(a[5], &out) || (a[6] != Py_None && !pointer_of(a[6], &sinks)) || !shape_of(a[7], &shape) ||
        !int_of(a[8], &dtype)) Py_RETURN_NONE;
    return call([&] { return g_lib.attention_grouped_static((lng_gpu *)gpu, stream, q, k, v, out, (const float *)sinks, &shape, dtype); });
}

PyObject *attention_decode_batched(PyObject *, Args a, Py_ssize_t n_args) { // batch, five buffers, items, heads, kv_heads, dim, scale, dtype
    ARGUMENTS(12);
    void *b;
    uint64_t u[8];
    float scale;
    int dtype;
    for (int i = 0; i < 8; ++i) {
        if (!u64_of(a[i < 5 ? 1 + i : 2 + i], &u[i])) Py_RETURN_NONE;
    }
    Table items;
    if (!handle_of(a[0], &b) || !float_of(a[10], &scale) || !int_of(a[11], &dtype) || !items.of(a[6], g_item)) Py_RETURN_NONE;
    return call([&] {
        return g_lib.attention_decode_batched((lng_batch *)b, u[0], u[1], u[2], u[3], u[4], (const lng_decode_item *)items.view.buf,
                                              (size_t)items.view.len / sizeof(lng_decode_item), u[5], u[6], u[7], scale, dtype);
    });
}

PyObject *copy_rows(PyObject *, Args a, Py_ssize_t n_args) { // batch, (src, stride), (dst, stride), rows, width, src_dtype, dst_dtype
    ARGUMENTS(7);
    void *b;
    PyObject *s, *ss, *d, *ds;
    lng_slice src, dst;
    uint64_t src_stride, dst_stride, rows, width;
    int src_dtype, dst_dtype;
    if (!handle_of(a[0], &b) || !two_of(a[1], &s, &ss) || !two_of(a[2], &d, &ds) || !slice_of(s, &src) || !u64_of(ss, &src_stride) ||
        !slice_of(d, &dst) || !u64_of(ds, &dst_stride) || !u64_of(a[3], &rows) || !u64_of(a[4], &width) || !int_of(a[5], &src_dtype) ||
        !int_of(a[6], &dst_dtype)) Py_RETURN_NONE;
    return call([&] { return g_lib.copy_rows((lng_batch *)b, src, src_stride, src_dtype, dst, dst_stride, dst_dtype, rows, width); });
}

PyObject *rmsnorm_rows(PyObject *, Args a, Py_ssize_t n_args) { // batch, (v, w), rows, (d, stride), eps
    ARGUMENTS(5);
    void *b;
    PyObject *v, *w, *d, *stride;
    lng_slice vs, ws;
    uint64_t rows, width, by;
    float eps;
    if (!handle_of(a[0], &b) || !two_of(a[1], &v, &w) || !slice_of(v, &vs) || !slice_of(w, &ws) || !u64_of(a[2], &rows) ||
        !two_of(a[3], &d, &stride) || !u64_of(d, &width) || !u64_of(stride, &by) || !float_of(a[4], &eps)) Py_RETURN_NONE;
    return call([&] { return g_lib.rmsnorm_rows((lng_batch *)b, vs, ws, rows, width, by, eps); });
}

PyObject *add_rows(PyObject *, Args a, Py_ssize_t n_args) { // batch, dst, (src, stride), rows, width
    ARGUMENTS(5);
    void *b;
    PyObject *s, *stride;
    lng_slice dst, src;
    uint64_t by, rows, width;
    if (!handle_of(a[0], &b) || !slice_of(a[1], &dst) || !two_of(a[2], &s, &stride) || !slice_of(s, &src) || !u64_of(stride, &by) ||
        !u64_of(a[3], &rows) || !u64_of(a[4], &width)) Py_RETURN_NONE;
    return call([&] { return g_lib.add_rows((lng_batch *)b, dst, src, by, rows, width); });
}

PyObject *prepare_attention(PyObject *, Args a, Py_ssize_t n_args) { // batch, {buffers}, items, heads, kv_heads, dim, rotary, dtype, three biases or None
    ARGUMENTS(11);
    void *b;
    uint64_t heads, kv_heads, dim, rotary;
    int dtype;
    lng_prepare_buffers pb{};
    uint64_t *const into[7] = {&pb.q, &pb.k, &pb.v, &pb.table, &pb.q_out, &pb.k_cache, &pb.v_cache};
    const lng_slice **const biases[3] = {&pb.q_bias, &pb.k_bias, &pb.v_bias};
    lng_slice held[3];
    if (!handle_of(a[0], &b) || !PyDict_CheckExact(a[1])) Py_RETURN_NONE;
    for (int i = 0; i < 7; ++i) {
        PyObject *at = PyDict_GetItemWithError(a[1], g_names[i]);
        if (!at || !u64_of(at, into[i])) {
            PyErr_Clear();
            Py_RETURN_NONE;
        }
    }
    for (int i = 0; i < 3; ++i) {
        if (a[8 + i] == Py_None) continue;
        if (!slice_of(a[8 + i], &held[i])) Py_RETURN_NONE;
        *biases[i] = &held[i];
    }
    Table items;
    if (!u64_of(a[3], &heads) || !u64_of(a[4], &kv_heads) || !u64_of(a[5], &dim) || !u64_of(a[6], &rotary) || !int_of(a[7], &dtype) ||
        !items.of(a[2], g_prepare_item)) Py_RETURN_NONE;
    return call([&] {
        return g_lib.prepare_attention((lng_batch *)b, &pb, (const lng_prepare_item *)items.view.buf,
                                       (size_t)items.view.len / sizeof(lng_prepare_item), heads, kv_heads, dim, rotary, dtype);
    });
}

PyObject *gemm(Args a, Py_ssize_t n_args, decltype(&lng_hip_gemm_q8_0) f) { // batch, matrix, x, y, rows, cols, n, strides
    ARGUMENTS(8);
    void *b;
    PyObject *xs, *ys;
    lng_slice codes, scales, x, y;
    uint64_t rows, cols, n, x_stride, y_stride;
    if (!handle_of(a[0], &b) || !matrix_of(a[1], &codes, &scales) || !slice_of(a[2], &x) || !slice_of(a[3], &y) || !u64_of(a[4], &rows) ||
        !u64_of(a[5], &cols) || !u64_of(a[6], &n) || !two_of(a[7], &xs, &ys) || !u64_of(xs, &x_stride) || !u64_of(ys, &y_stride)) Py_RETURN_NONE;
    return call([&] { return f((lng_batch *)b, codes, scales, x, y, rows, cols, n, x_stride, y_stride); });
}
PyObject *gemm_q8_0(PyObject *, Args a, Py_ssize_t n) { return gemm(a, n, g_lib.gemm_q8_0); }
PyObject *gemm_q8_0_tiled(PyObject *, Args a, Py_ssize_t n) { return gemm(a, n, g_lib.gemm_q8_0_tiled); }
PyObject *gemm_q8_0_bf16(PyObject *, Args a, Py_ssize_t n) { return gemm(a, n, g_lib.gemm_q8_0_bf16); }

bool matrices_of(PyObject *o, lng_q8_matrix *m, size_t *count) { // a list of ((codes, scales), y, rows)
    if (!PyList_CheckExact(o) || PyList_GET_SIZE(o) > 4) return false;
    *count = (size_t)PyList_GET_SIZE(o);
    for (size_t i = 0; i < *count; ++i) {
        PyObject *one = PyList_GET_ITEM(o, (Py_ssize_t)i);
        if (!PyTuple_CheckExact(one) || PyTuple_GET_SIZE(one) != 3 || !matrix_of(PyTuple_GET_ITEM(one, 0), &m[i].codes, &m[i].scales) ||
            !slice_of(PyTuple_GET_ITEM(one, 1), &m[i].y) || !u64_of(PyTuple_GET_ITEM(one, 2), &m[i].rows)) return false;
    }
    return true;
}

PyObject *gemm_q8_0_many(PyObject *, Args a, Py_ssize_t n_args) { // batch, matrices, x, cols, n, x_stride
    ARGUMENTS(6);
    void *b;
    lng_q8_matrix m[4];
    size_t count;
    lng_slice x;
    uint64_t cols, n, x_stride;
    if (!handle_of(a[0], &b) || !matrices_of(a[1], m, &count) || !slice_of(a[2], &x) || !u64_of(a[3], &cols) || !u64_of(a[4], &n) ||
        !u64_of(a[5], &x_stride)) Py_RETURN_NONE;
    return call([&] { return g_lib.gemm_q8_0_many((lng_batch *)b, m, count, x, cols, n, x_stride); });
}

PyObject *gemm_q8_0_many_normed(PyObject *, Args a, Py_ssize_t n_args) { // batch, matrices, x, (weights, eps), cols, n, x_stride
    ARGUMENTS(7);
    void *b;
    PyObject *w, *e;
    lng_q8_matrix m[4];
    size_t count;
    lng_slice x, weights;
    float eps;
    uint64_t cols, n, x_stride;
    if (!handle_of(a[0], &b) || !matrices_of(a[1], m, &count) || !slice_of(a[2], &x) || !two_of(a[3], &w, &e) || !slice_of(w, &weights) ||
        !float_of(e, &eps) || !u64_of(a[4], &cols) || !u64_of(a[5], &n) || !u64_of(a[6], &x_stride)) Py_RETURN_NONE;
    return call([&] { return g_lib.gemm_q8_0_many_normed((lng_batch *)b, m, count, x, weights, eps, cols, n, x_stride); });
}

PyObject *gemm_q8_0_residual(PyObject *, Args a, Py_ssize_t n_args) { // batch, matrix, x, bias or None, h, rows, cols, n, strides, x_dtype
    ARGUMENTS(10);
    void *b;
    PyObject *xs, *hs;
    lng_slice codes, scales, x, bias, h;
    uint64_t rows, cols, n, x_stride, h_stride;
    int dtype;
    if (!handle_of(a[0], &b) || !matrix_of(a[1], &codes, &scales) || !slice_of(a[2], &x) || (a[3] != Py_None && !slice_of(a[3], &bias)) ||
        !slice_of(a[4], &h) || !u64_of(a[5], &rows) || !u64_of(a[6], &cols) || !u64_of(a[7], &n) || !two_of(a[8], &xs, &hs) ||
        !u64_of(xs, &x_stride) || !u64_of(hs, &h_stride) || !int_of(a[9], &dtype)) Py_RETURN_NONE;
    const lng_slice *with = a[3] == Py_None ? nullptr : &bias;
    return call([&] { return g_lib.gemm_q8_0_residual((lng_batch *)b, codes, scales, x, dtype, with, h, rows, cols, n, x_stride, h_stride); });
}

bool fields_of(PyTypeObject *type, const char *const *names, int n, Py_ssize_t *at) { // where a class with __slots__ keeps them
    for (int i = 0; i < n; ++i) {
        PyObject *d = PyObject_GetAttrString((PyObject *)type, names[i]);
        if (!d || Py_TYPE(d) != &PyMemberDescr_Type || ((PyMemberDescrObject *)d)->d_member->type != T_OBJECT_EX) {
            Py_XDECREF(d);
            if (!PyErr_Occurred()) PyErr_Format(PyExc_TypeError, "%s has no slot %s", type->tp_name, names[i]);
            return false;
        }
        at[i] = ((PyMemberDescrObject *)d)->d_member->offset;
        Py_DECREF(d);
    }
    return true;
}

PyObject *bind(PyObject *, PyObject *args) { // {function: address}, Slice, GroupedShape, the decode item's and the prepare item's ctypes
    PyObject *addresses, *slice, *shape, *item, *prepare_item;
    if (!PyArg_ParseTuple(args, "O!O!O!O!O!", &PyDict_Type, &addresses, &PyType_Type, &slice, &PyType_Type, &shape, &PyType_Type, &item,
                          &PyType_Type, &prepare_item)) return nullptr;
    static const char *const slice_fields[] = {"buffer", "offset", "len"};
    static const char *const shape_fields[] = {"t", "start", "heads", "kv_heads", "dim", "window", "slots", "scale"};
    if (!fields_of((PyTypeObject *)slice, slice_fields, 3, g_slice_at) || !fields_of((PyTypeObject *)shape, shape_fields, 8, g_shape_at)) return nullptr;
    const struct { const char *name; void *into; } functions[] = {
        {"lng_hip_batch", &g_lib.batch}, {"lng_hip_batch_commit", &g_lib.batch_commit}, {"lng_hip_batch_wait", &g_lib.batch_wait},
        {"lng_hip_batch_drop", &g_lib.batch_drop}, {"lng_hip_attention_grouped", &g_lib.attention_grouped},
        {"lng_hip_attention_grouped_tiled", &g_lib.attention_grouped_tiled}, {"lng_hip_attention_grouped_static", &g_lib.attention_grouped_static},
        {"lng_hip_attention_decode_batched", &g_lib.attention_decode_batched}, {"lng_hip_copy_rows", &g_lib.copy_rows},
        {"lng_hip_rmsnorm_rows", &g_lib.rmsnorm_rows}, {"lng_hip_add_rows", &g_lib.add_rows}, {"lng_hip_prepare_attention", &g_lib.prepare_attention},
        {"lng_hip_gemm_q8_0", &g_lib.gemm_q8_0}, {"lng_hip_gemm_q8_0_tiled", &g_lib.gemm_q8_0_tiled}, {"lng_hip_gemm_q8_0_bf16", &g_lib.gemm_q8_0_bf16},
        {"lng_hip_gemm_q8_0_many", &g_lib.gemm_q8_0_many}, {"lng_hip_gemm_q8_0_many_normed", &g_lib.gemm_q8_0_many_normed},
        {"lng_hip_gemm_q8_0_residual", &g_lib.gemm_q8_0_residual}};
    for (const auto &f : functions) {
        PyObject *address = PyDict_GetItemString(addresses, f.name);
        uint64_t v;
        if (!address || !u64_of(address, &v) || !v) return PyErr_Format(PyExc_TypeError, "no address of %s", f.name);
        *(uint64_t *)f.into = v;
    }
    for (PyObject *type : {slice, shape, item, prepare_item}) Py_INCREF(type); // for good: bound once, as the library is
    g_slice = (PyTypeObject *)slice;
    g_shape = (PyTypeObject *)shape;
    g_item = (PyTypeObject *)item;
    g_prepare_item = (PyTypeObject *)prepare_item;
    Py_RETURN_NONE;
}

#define SHORT(name) {#name, (PyCFunction)(void (*)(void))name, METH_FASTCALL, nullptr}
PyMethodDef g_methods[] = {
    {"bind", bind, METH_VARARGS, nullptr}, SHORT(batch), SHORT(commit), SHORT(wait), SHORT(drop), SHORT(attention_grouped), SHORT(attention_grouped_tiled),
    SHORT(attention_grouped_static), SHORT(attention_decode_batched), SHORT(copy_rows), SHORT(rmsnorm_rows), SHORT(add_rows), SHORT(prepare_attention),
    SHORT(gemm_q8_0), SHORT(gemm_q8_0_tiled), SHORT(gemm_q8_0_bf16), SHORT(gemm_q8_0_many), SHORT(gemm_q8_0_many_normed), SHORT(gemm_q8_0_residual),
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "_record", "The short way from compute.py into the C ABI.", -1, g_methods, nullptr, nullptr, nullptr, nullptr};

} // namespace

PyMODINIT_FUNC PyInit__record(void) {
    static const char *const names[7] = {"q", "k", "v", "table", "q_out", "k_cache", "v_cache"};
    for (int i = 0; i < 7; ++i) {
        if (!(g_names[i] = PyUnicode_InternFromString(names[i]))) return nullptr;
    }
    if (!(g_element = PyUnicode_InternFromString("_type_"))) return nullptr;
    return PyModule_Create(&g_module);
}
