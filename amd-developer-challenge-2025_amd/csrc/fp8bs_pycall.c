/* CPython binding of the compute entry points of libfp8bs.so (include/fp8bs.h), for callers that issue many
 * small calls from Python: ctypes spends ~1.2 us marshalling the 13 arguments of fp8bs_gemm_ex, this module
 * ~0.15 us.  Pointers and the stream arrive as Python ints (tensor.data_ptr(), the raw hipStream_t) or None;
 * the status code is returned as an int.  Nothing else lives here: checks, planning and launches are the
 * library's.  Built by build.py with the host compiler; when the module is missing the package binds the same
 * functions through ctypes (the library itself has no substitute).
 * Stands where the reference has its pybind11 module built by load_inline
 * (1-amd-fp8-mm/amd-fp8-mm-submission.py:582-592). */
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <stdint.h>

#include "fp8bs.h"

/* a Python int (address) or None -> pointer; -1 with an exception set on anything else */
static int as_pointer(PyObject* o, void** out) {
    if (o == Py_None) { *out = NULL; return 0; }
    void* p = PyLong_AsVoidPtr(o);
    if (p == NULL && PyErr_Occurred()) return -1;
    *out = p;
    return 0;
}

static int as_int(PyObject* o, int* out) {
    long v = PyLong_AsLong(o);
    if (v == -1 && PyErr_Occurred()) return -1;
    if (v < INT32_MIN || v > INT32_MAX) { PyErr_SetString(PyExc_OverflowError, "argument does not fit a C int"); return -1; }
    *out = (int)v;
    return 0;
}

/* gemm_ex(a, b, a_scale, b_scale, c, ws, ws_bytes, m, n, k, variant, split_k, stream) -> status */
static PyObject* py_gemm_ex(PyObject* self, PyObject* const* args, Py_ssize_t nargs) {
    (void)self;
    if (nargs != 13) { PyErr_SetString(PyExc_TypeError, "gemm_ex takes 13 arguments"); return NULL; }
    void* p[6]; void* stream; int v[5];
    for (int i = 0; i < 6; i++) if (as_pointer(args[i], &p[i]) < 0) return NULL;
    size_t ws_bytes = PyLong_AsSize_t(args[6]);
    if (ws_bytes == (size_t)-1 && PyErr_Occurred()) return NULL;
    for (int i = 0; i < 5; i++) if (as_int(args[7 + i], &v[i]) < 0) return NULL;
    if (as_pointer(args[12], &stream) < 0) return NULL;
    int st = fp8bs_gemm_ex(p[0], p[1], (const float*)p[2], (const float*)p[3], p[4], p[5], ws_bytes, v[0], v[1], v[2], v[3], v[4], stream);
    return PyLong_FromLong(st);
}

/* gemm_grouped_ex(a, b, a_scale, b_scale, c, row_offsets, num_experts, total_rows, n, k, variant, stream) -> status */
static PyObject* py_gemm_grouped_ex(PyObject* self, PyObject* const* args, Py_ssize_t nargs) {
    (void)self;
    if (nargs != 12) { PyErr_SetString(PyExc_TypeError, "gemm_grouped_ex takes 12 arguments"); return NULL; }
    void* p[6]; void* stream; int v[5];
    for (int i = 0; i < 6; i++) if (as_pointer(args[i], &p[i]) < 0) return NULL;
    for (int i = 0; i < 5; i++) if (as_int(args[6 + i], &v[i]) < 0) return NULL;
    if (as_pointer(args[11], &stream) < 0) return NULL;
    int st = fp8bs_gemm_grouped_ex(p[0], p[1], (const float*)p[2], (const float*)p[3], p[4], (const int32_t*)p[5], v[0], v[1], v[2], v[3], v[4], stream);
    return PyLong_FromLong(st);
}

/* gemm_grouped_ws / gemm_silu_mul_ws(a, b, a_scale, b_scale, c, row_offsets, num_experts, rows, n, k, variant, split_k, ws, ws_bytes, stream) -> status */
typedef int (*grouped_fn)(const void*, const void*, const float*, const float*, void*, const int32_t*, int, int, int, int, int, int, void*, size_t, void*);
static PyObject* call_grouped(grouped_fn fn, PyObject* const* args, Py_ssize_t nargs) {
    if (nargs != 15) { PyErr_SetString(PyExc_TypeError, "15 arguments expected"); return NULL; }
    void* p[6]; void* stream; void* ws; int v[6];
    for (int i = 0; i < 6; i++) if (as_pointer(args[i], &p[i]) < 0) return NULL;
    for (int i = 0; i < 6; i++) if (as_int(args[6 + i], &v[i]) < 0) return NULL;
    if (as_pointer(args[12], &ws) < 0) return NULL;
    size_t ws_bytes = PyLong_AsSize_t(args[13]);
    if (ws_bytes == (size_t)-1 && PyErr_Occurred()) return NULL;
    if (as_pointer(args[14], &stream) < 0) return NULL;
    return PyLong_FromLong(fn(p[0], p[1], (const float*)p[2], (const float*)p[3], p[4], (const int32_t*)p[5], v[0], v[1], v[2], v[3], v[4], v[5], ws, ws_bytes, stream));
}
static PyObject* py_gemm_grouped_ws(PyObject* self, PyObject* const* args, Py_ssize_t nargs) { (void)self; return call_grouped(fp8bs_gemm_grouped_ws, args, nargs); }
static PyObject* py_gemm_silu_mul_ws(PyObject* self, PyObject* const* args, Py_ssize_t nargs) { (void)self; return call_grouped(fp8bs_gemm_silu_mul_ws, args, nargs); }

/* The quantisers and the routing kernels: arguments as `format` says, 'p' an address or None, 'i' an int, 'l' an int64, 'z' a size_t */
typedef union { void* p; int i; int64_t l; size_t z; } arg;
static int unpack(PyObject* const* args, Py_ssize_t nargs, const char* format, arg* out) {
    Py_ssize_t n = 0;
    for (; format[n]; n++) {
        if (n >= nargs) break;
        if (format[n] == 'p') { if (as_pointer(args[n], &out[n].p) < 0) return -1; }
        else if (format[n] == 'i') { if (as_int(args[n], &out[n].i) < 0) return -1; }
        else if (format[n] == 'l') { out[n].l = PyLong_AsLongLong(args[n]); if (out[n].l == -1 && PyErr_Occurred()) return -1; }
        else { out[n].z = PyLong_AsSize_t(args[n]); if (out[n].z == (size_t)-1 && PyErr_Occurred()) return -1; }
    }
    if (format[n] || n != nargs) { PyErr_SetString(PyExc_TypeError, "wrong number of arguments"); return -1; }
    return 0;
}
static PyObject* py_quantize_a(PyObject* self, PyObject* const* args, Py_ssize_t nargs) {
    (void)self;
    arg v[10];
    if (unpack(args, nargs, "pilpippiip", v) < 0) return NULL;
    return PyLong_FromLong(fp8bs_quantize_a(v[0].p, v[1].i, v[2].l, (const int32_t*)v[3].p, v[4].i, v[5].p, (float*)v[6].p, v[7].i, v[8].i, v[9].p));
}
static PyObject* py_quantize_b(PyObject* self, PyObject* const* args, Py_ssize_t nargs) {
    (void)self;
    arg v[8];
    if (unpack(args, nargs, "pilppiip", v) < 0) return NULL;
    return PyLong_FromLong(fp8bs_quantize_b(v[0].p, v[1].i, v[2].l, v[3].p, (float*)v[4].p, v[5].i, v[6].i, v[7].p));
}
static PyObject* py_gather_a(PyObject* self, PyObject* const* args, Py_ssize_t nargs) {
    (void)self;
    arg v[9];
    if (unpack(args, nargs, "ppipppiip", v) < 0) return NULL;
    return PyLong_FromLong(fp8bs_gather_a(v[0].p, (const float*)v[1].p, v[2].i, (const int32_t*)v[3].p, v[4].p, (float*)v[5].p, v[6].i, v[7].i, v[8].p));
}
static PyObject* py_moe_topk(PyObject* self, PyObject* const* args, Py_ssize_t nargs) {
    (void)self;
    arg v[6];
    if (unpack(args, nargs, "piiipp", v) < 0) return NULL;
    return PyLong_FromLong(fp8bs_moe_topk((const float*)v[0].p, v[1].i, v[2].i, v[3].i, (int32_t*)v[4].p, v[5].p));
}
static PyObject* py_moe_route(PyObject* self, PyObject* const* args, Py_ssize_t nargs) {
    (void)self;
    arg v[10];
    if (unpack(args, nargs, "piiippppzp", v) < 0) return NULL;
    return PyLong_FromLong(fp8bs_moe_route((const int32_t*)v[0].p, v[1].i, v[2].i, v[3].i, (int32_t*)v[4].p, (int32_t*)v[5].p, (int32_t*)v[6].p, v[7].p, v[8].z, v[9].p));
}
static PyObject* py_moe_combine(PyObject* self, PyObject* const* args, Py_ssize_t nargs) {
    (void)self;
    arg v[9];
    if (unpack(args, nargs, "pipppiiip", v) < 0) return NULL;
    return PyLong_FromLong(fp8bs_moe_combine(v[0].p, v[1].i, (const int32_t*)v[2].p, (const float*)v[3].p, v[4].p, v[5].i, v[6].i, v[7].i, v[8].p));
}

static PyMethodDef methods[] = {
    {"gemm_ex", (PyCFunction)(void (*)(void))py_gemm_ex, METH_FASTCALL, "fp8bs_gemm_ex with addresses as ints; returns the status code"},
    {"gemm_grouped_ex", (PyCFunction)(void (*)(void))py_gemm_grouped_ex, METH_FASTCALL, "fp8bs_gemm_grouped_ex with addresses as ints; returns the status code"},
    {"gemm_grouped_ws", (PyCFunction)(void (*)(void))py_gemm_grouped_ws, METH_FASTCALL, "fp8bs_gemm_grouped_ws with addresses as ints; returns the status code"},
    {"gemm_silu_mul_ws", (PyCFunction)(void (*)(void))py_gemm_silu_mul_ws, METH_FASTCALL, "fp8bs_gemm_silu_mul_ws with addresses as ints; returns the status code"},
    {"quantize_a", (PyCFunction)(void (*)(void))py_quantize_a, METH_FASTCALL, "fp8bs_quantize_a with addresses as ints; returns the status code"},
    {"quantize_b", (PyCFunction)(void (*)(void))py_quantize_b, METH_FASTCALL, "fp8bs_quantize_b with addresses as ints; returns the status code"},
    {"gather_a", (PyCFunction)(void (*)(void))py_gather_a, METH_FASTCALL, "fp8bs_gather_a with addresses as ints; returns the status code"},
    {"moe_topk", (PyCFunction)(void (*)(void))py_moe_topk, METH_FASTCALL, "fp8bs_moe_topk with addresses as ints; returns the status code"},
    {"moe_route", (PyCFunction)(void (*)(void))py_moe_route, METH_FASTCALL, "fp8bs_moe_route with addresses as ints; returns the status code"},
    {"moe_combine", (PyCFunction)(void (*)(void))py_moe_combine, METH_FASTCALL, "fp8bs_moe_combine with addresses as ints; returns the status code"},
    {NULL, NULL, 0, NULL},
};

static struct PyModuleDef module = {PyModuleDef_HEAD_INIT, "_fp8bs_pycall", "fast calls into libfp8bs.so", -1, methods, NULL, NULL, NULL, NULL};

PyMODINIT_FUNC PyInit__fp8bs_pycall(void) { return PyModule_Create(&module); }
