// The compute entry points on torch tensors, for callers that issue many small calls from Python: checks, allocation of the results and
// the call in one native function each.  custom_kernel's checks in Python were some forty attribute reads and comparisons; here they are read from the tensors themselves, at
// every call.  Calls issued one after another: 256 x 512 x 1024 5.2 us before, 4.1 now (the kernel takes 3.8), 3 x 2092 x 384 5.2
// and 3.6, 1 x 3968 x 384 5.3 and 3.9; with tensors that were not seen before 24 and 16, waiting for each.  The others, host time a call, before and now:
// quantize_b 7.1 and 4.9; quantise, gate/up with SiLU*mul, quantise and down of 8 x 1792 x 2176, bound by the host, 23.1 and 16.6; a layer
// (seven calls) of 6 tokens to 2 of 8 experts 46.7 and 32.8; of each 3 us are the launch.
// Whatever is not the usual case (another layout, type or device, an empty product, a tensor subclass, a size that has not been
// planned yet) is handed back: the Python path takes it, or says what is wrong with it.
// Built by build.py with the host compiler against torch's headers; without this module the Python path takes every call.
#define PY_SSIZE_T_CLEAN
#include <torch/csrc/autograd/python_variable.h>
#include <ATen/ATen.h>
#include <c10/hip/HIPStream.h>
#include <hip/hip_runtime_api.h>

#include <exception>
#include <initializer_list>

#include "fp8bs.h"

namespace {

constexpr long NOT_HERE = -1;

// (the stride of a dimension of one element is immaterial)
bool kmajor(const at::Tensor& t) { return (t.size(0) == 1 || t.stride(0) == 1) && (t.size(1) == 1 || t.stride(1) == t.size(0)); }

// The call's status code, NOT_HERE, or -(bytes) where a larger workspace is wanted than the one given.
// Throws what torch throws.
long dense_call(const at::Tensor* const* t, PyObject* planned, void* ws, size_t ws_bytes) {
    const at::Tensor &a = *t[0], &b = *t[1], &as = *t[2], &bs = *t[3], &c = *t[4];
    const at::ScalarType types[5] = {at::kFloat8_e4m3fn, at::kFloat8_e4m3fn, at::kFloat, at::kFloat, at::kBFloat16};
    for (int i = 0; i < 5; i++)
        if (t[i]->scalar_type() != types[i] || !t[i]->is_cuda() || t[i]->layout() != at::kStrided || t[i]->dim() != 2 || t[i]->device() != a.device()) return NOT_HERE;
    const int64_t m = a.size(0), k = a.size(1), n = b.size(0), nb = (n + 127) / 128, kb = k / 128;
    if (m < 1 || n < 1 || k < 128 || k % 128 != 0 || m > INT32_MAX || n > INT32_MAX || k > INT32_MAX) return NOT_HERE;
    if (b.size(1) != k || as.size(0) != m || as.size(1) != kb || bs.size(0) != nb || bs.size(1) != kb || c.size(0) != m || c.size(1) != n) return NOT_HERE;
    if (!kmajor(a) || !kmajor(b) || !kmajor(as) || !kmajor(bs) || !c.is_contiguous()) return NOT_HERE;
    int device = -1;
    if (hipGetDevice(&device) != hipSuccess || device != a.get_device()) return NOT_HERE;
    PyObject* const key = Py_BuildValue("(LLL)", (long long)m, (long long)n, (long long)k);
    PyObject* const bytes = key ? PyDict_GetItem(planned, key) : nullptr;      // (borrowed)
    Py_XDECREF(key);
    const size_t want = bytes ? PyLong_AsSize_t(bytes) : 0;
    if (!bytes || PyErr_Occurred()) { PyErr_Clear(); return NOT_HERE; }
    if (want > ws_bytes) return -(long)want;
    return fp8bs_gemm_ex(a.const_data_ptr(), b.const_data_ptr(), (const float*)as.const_data_ptr(), (const float*)bs.const_data_ptr(), c.mutable_data_ptr(), ws, ws_bytes,
                         (int)m, (int)n, (int)k, FP8BS_VARIANT_AUTO, 0, c10::hip::getCurrentHIPStream((c10::DeviceIndex)device).stream());
}

// dense(data, planned, workspace, workspace_bytes): data the five tensors, planned a dict (m, n, k) -> bytes of workspace
PyObject* dense(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    if (nargs != 4 || !PyDict_CheckExact(args[1])) { PyErr_SetString(PyExc_TypeError, "dense(data, planned, workspace, workspace_bytes)"); return nullptr; }
    void* const ws = PyLong_AsVoidPtr(args[2]);
    if (PyErr_Occurred()) return nullptr;
    const size_t ws_bytes = PyLong_AsSize_t(args[3]);
    if (PyErr_Occurred()) return nullptr;
    if (!(PyTuple_CheckExact(args[0]) || PyList_CheckExact(args[0])) || PySequence_Fast_GET_SIZE(args[0]) != 5) return PyLong_FromLong(NOT_HERE);
    const at::Tensor* t[5];
    for (int i = 0; i < 5; i++) {
        PyObject* const o = PySequence_Fast_GET_ITEM(args[0], i);
        if (!THPVariable_CheckExact(o)) return PyLong_FromLong(NOT_HERE);      // a subclass has rules of its own
        t[i] = &THPVariable_Unpack(o);
    }
    // (a tensor without storage or with symbolic sizes, as tracing and vmap make them, throws: the Python path raises its error)
    long result = NOT_HERE;
    try { result = dense_call(t, args[1], ws, ws_bytes); } catch (const std::exception&) { result = NOT_HERE; }
    return PyLong_FromLong(result);
}

// ---- the other entry points: nullptr with no exception set stands for "not taken" until done() ----

// A tensor of the plain class, type and number of dimensions on the device that is current; nullptr: not one.
const at::Tensor* plain(PyObject* o, at::ScalarType type, int64_t dim, int device) {
    if (!THPVariable_CheckExact(o)) return nullptr;                              // a subclass has rules of its own
    const at::Tensor& t = THPVariable_Unpack(o);
    return t.scalar_type() == type && t.is_cuda() && t.layout() == at::kStrided && t.dim() == dim && t.get_device() == device ? &t : nullptr;
}
int current_device() { int d = -1; return hipGetDevice(&d) == hipSuccess ? d : -1; }
bool fits(int64_t v, int64_t least) { return v >= least && v <= INT32_MAX; }
void* current_stream(int device) { return c10::hip::getCurrentHIPStream((c10::DeviceIndex)device).stream(); }
at::Tensor empty(at::IntArrayRef size, at::IntArrayRef stride, at::ScalarType type, int device) {
    return at::empty_strided(size, stride, at::TensorOptions().dtype(type).device(at::Device(at::kCUDA, (c10::DeviceIndex)device)));
}
// Runs f, which returns a new reference, or nullptr for "not taken"; what torch throws is left to the Python path to raise.
template <typename F> PyObject* taken(F&& f) {
    PyObject* r = nullptr;
    try { r = f(); } catch (const std::exception&) { r = nullptr; }
    if (!r) { if (PyErr_Occurred()) PyErr_Clear(); Py_RETURN_NONE; }
    return r;
}
PyObject* results(int status, std::initializer_list<at::Tensor> out) {             // the tensor, a tuple of them, or the status code
    if (status != 0) return PyLong_FromLong(status);
    if (out.size() == 1) return THPVariable_Wrap(*out.begin());
    PyObject* const tuple = PyTuple_New((Py_ssize_t)out.size());
    if (!tuple) return nullptr;
    Py_ssize_t i = 0;
    for (const at::Tensor& t : out) {
        PyObject* const o = THPVariable_Wrap(t);
        if (!o) { Py_DECREF(tuple); return nullptr; }
        PyTuple_SET_ITEM(tuple, i++, o);
    }
    return tuple;
}
bool number(PyObject* o, long long* v) { *v = PyLong_CheckExact(o) ? PyLong_AsLongLong(o) : -1; return PyLong_CheckExact(o) && !PyErr_Occurred(); }

// quantize(x, row_map or None, of_b): (codes, scales), both K-major
PyObject* quantize(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    if (nargs != 3) { PyErr_SetString(PyExc_TypeError, "quantize(x, row_map, of_b)"); return nullptr; }
    return taken([&]() -> PyObject* {
        const int device = current_device();
        const at::Tensor* x = plain(args[0], at::kBFloat16, 2, device);
        const int type = x ? 1 : 0;
        if (!x) x = plain(args[0], at::kFloat, 2, device);
        if (!x) return nullptr;
        const bool of_b = args[2] == Py_True;
        const int64_t t = x->size(0), k = x->size(1);
        int64_t m = t;
        const int32_t* row_map = nullptr;
        if (args[1] != Py_None) {
            const at::Tensor* const map = plain(args[1], at::kInt, 1, device);
            if (!map || of_b || !map->is_contiguous()) return nullptr;
            m = map->numel();
            row_map = (const int32_t*)map->const_data_ptr();
        }
        if (!fits(t, 1) || !fits(m, 1) || !fits(k, 128) || k % 128 != 0 || x->stride(1) != 1) return nullptr;
        const void* const from = x->const_data_ptr();
        const int64_t ldx = t > 1 ? x->stride(0) : k, groups = of_b ? (m + 127) / 128 : m;
        at::Tensor q = empty({m, k}, {1, m}, at::kFloat8_e4m3fn, device), scale = empty({groups, k / 128}, {1, groups}, at::kFloat, device);
        void* const stream = current_stream(device);
        const int st = of_b ? fp8bs_quantize_b(from, type, ldx, q.mutable_data_ptr(), (float*)scale.mutable_data_ptr(), (int)m, (int)k, stream)
                            : fp8bs_quantize_a(from, type, ldx, row_map, (int)t, q.mutable_data_ptr(), (float*)scale.mutable_data_ptr(), (int)m, (int)k, stream);
        return results(st, {q, scale});
    });
}

// experts(data, planned, workspace, workspace_bytes, silu): grouped_kernel's and gate_up_silu's checks and call, c at the end of data; the
// status code, -1, or -(bytes) as dense has them.  planned: a dict (silu, experts or 0, rows, n, k) -> bytes of workspace
PyObject* experts(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    if (nargs != 5 || !PyDict_CheckExact(args[1])) { PyErr_SetString(PyExc_TypeError, "experts(data, planned, workspace, workspace_bytes, silu)"); return nullptr; }
    void* const ws = PyLong_AsVoidPtr(args[2]);
    if (PyErr_Occurred()) return nullptr;
    const size_t ws_bytes = PyLong_AsSize_t(args[3]);
    if (PyErr_Occurred()) return nullptr;
    long result = NOT_HERE;
    try {
        result = [&]() -> long {
            if (!(PyTuple_CheckExact(args[0]) || PyList_CheckExact(args[0])) || PySequence_Fast_GET_SIZE(args[0]) != 6) return NOT_HERE;
            PyObject* const* const o = PySequence_Fast_ITEMS(args[0]);
            const bool silu = args[4] == Py_True, grouped = o[4] != Py_None;
            const int device = current_device(), dim = grouped ? 3 : 2;
            const at::Tensor *a = plain(o[0], at::kFloat8_e4m3fn, 2, device), *b = plain(o[1], at::kFloat8_e4m3fn, dim, device);
            const at::Tensor *as = plain(o[2], at::kFloat, 2, device), *bs = plain(o[3], at::kFloat, dim, device), *c = plain(o[5], at::kBFloat16, 2, device);
            const at::Tensor* const ro = grouped ? plain(o[4], at::kInt, 1, device) : nullptr;
            if (!a || !b || !as || !bs || !c || (grouped && !ro)) return NOT_HERE;
            const int64_t m = a->size(0), k = a->size(1), e = grouped ? b->size(0) : 0, n = b->size(dim - 2), nb = (n + 127) / 128, kb = k / 128;
            if (!fits(m, 1) || !fits(n, 1) || !fits(k, 128) || k % 128 != 0 || (grouped && !fits(e, 1)) || (silu && n % 2 != 0)) return NOT_HERE;
            if (b->size(dim - 1) != k || as->size(0) != m || as->size(1) != kb || bs->size(dim - 2) != nb || bs->size(dim - 1) != kb) return NOT_HERE;
            if (c->size(0) != m || c->size(1) != (silu ? n / 2 : n) || !kmajor(*a) || !kmajor(*as) || !c->is_contiguous()) return NOT_HERE;
            if (grouped) {
                if (bs->size(0) != e || ro->size(0) != e + 1 || !ro->is_contiguous()) return NOT_HERE;
                if (b->stride(0) != n * k || b->stride(1) != 1 || b->stride(2) != n || bs->stride(0) != nb * kb || bs->stride(1) != 1 || bs->stride(2) != nb) return NOT_HERE;
            } else if (!kmajor(*b) || !kmajor(*bs)) {
                return NOT_HERE;
            }
            PyObject* const key = Py_BuildValue("(iLLLL)", silu ? 1 : 0, (long long)e, (long long)m, (long long)n, (long long)k);
            PyObject* const bytes = key ? PyDict_GetItem(args[1], key) : nullptr;                    // (borrowed)
            Py_XDECREF(key);
            const size_t want = bytes ? PyLong_AsSize_t(bytes) : 0;
            if (!bytes || PyErr_Occurred()) { PyErr_Clear(); return NOT_HERE; }
            if (want > ws_bytes) return -(long)want;
            const auto call = silu ? fp8bs_gemm_silu_mul_ws : fp8bs_gemm_grouped_ws;
            return call(a->const_data_ptr(), b->const_data_ptr(), (const float*)as->const_data_ptr(), (const float*)bs->const_data_ptr(), c->mutable_data_ptr(),
                        ro ? (const int32_t*)ro->const_data_ptr() : nullptr, (int)e, (int)m, (int)n, (int)k, FP8BS_VARIANT_AUTO, 0, want ? ws : nullptr, want ? ws_bytes : 0, current_stream(device));
        }();
    } catch (const std::exception&) { result = NOT_HERE; }
    return PyLong_FromLong(result);
}

// topk(scores, k): top_idx
PyObject* topk(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    if (nargs != 2) { PyErr_SetString(PyExc_TypeError, "topk(scores, k)"); return nullptr; }
    return taken([&]() -> PyObject* {
        const int device = current_device();
        long long k;
        const at::Tensor* const x = plain(args[0], at::kFloat, 2, device);
        if (!x || !x->is_contiguous() || !fits(x->size(0), 1) || !fits(x->size(1), 1) || !number(args[1], &k) || k < 1 || k > x->size(1)) return nullptr;
        const void* const from = x->const_data_ptr();
        at::Tensor out = empty({x->size(0), k}, {k, 1}, at::kInt, device);
        return results(fp8bs_moe_topk((const float*)from, (int)x->size(0), (int)x->size(1), (int)k, (int32_t*)out.mutable_data_ptr(), current_stream(device)), {out});
    });
}

// route(top_idx, experts, workspace, workspace_bytes): (row_offsets, row_map, slot_of)
PyObject* route(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    if (nargs != 4) { PyErr_SetString(PyExc_TypeError, "route(top_idx, experts, workspace, workspace_bytes)"); return nullptr; }
    void* const ws = PyLong_AsVoidPtr(args[2]);
    if (PyErr_Occurred()) return nullptr;
    const size_t ws_bytes = PyLong_AsSize_t(args[3]);
    if (PyErr_Occurred()) return nullptr;
    return taken([&]() -> PyObject* {
        const int device = current_device();
        long long e;
        const at::Tensor* const x = plain(args[0], at::kInt, 2, device);
        if (!x || !x->is_contiguous() || !fits(x->size(0), 1) || !fits(x->size(1), 1) || !fits(x->numel(), 1) || !number(args[1], &e) || !fits(e, 1)) return nullptr;
        const int64_t t = x->size(0), k = x->size(1);
        const void* const from = x->const_data_ptr();
        at::Tensor offsets = empty({e + 1}, {1}, at::kInt, device), map = empty({t * k}, {1}, at::kInt, device), slots = empty({t, k}, {k, 1}, at::kInt, device);
        return results(fp8bs_moe_route((const int32_t*)from, (int)t, (int)e, (int)k, (int32_t*)offsets.mutable_data_ptr(), (int32_t*)map.mutable_data_ptr(),
                                       (int32_t*)slots.mutable_data_ptr(), ws, ws_bytes, current_stream(device)), {offsets, map, slots});
    });
}

// combine(y, slot_of, weights): out
PyObject* combine(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    if (nargs != 3) { PyErr_SetString(PyExc_TypeError, "combine(y, slot_of, weights)"); return nullptr; }
    return taken([&]() -> PyObject* {
        const int device = current_device();
        const at::Tensor *y = plain(args[0], at::kBFloat16, 2, device), *slots = plain(args[1], at::kInt, 2, device), *w = plain(args[2], at::kFloat, 2, device);
        if (!y || !slots || !w || !y->is_contiguous() || !slots->is_contiguous() || !w->is_contiguous()) return nullptr;
        const int64_t t = slots->size(0), k = slots->size(1), rows = y->size(0), d = y->size(1);
        if (w->size(0) != t || w->size(1) != k || !fits(t, 1) || !fits(k, 1) || !fits(rows, 1) || !fits(d, 1)) return nullptr;
        const void *py = y->const_data_ptr(), *ps = slots->const_data_ptr(), *pw = w->const_data_ptr();
        at::Tensor out = empty({t, d}, {d, 1}, at::kBFloat16, device);
        return results(fp8bs_moe_combine(py, (int)rows, (const int32_t*)ps, (const float*)pw, out.mutable_data_ptr(), (int)t, (int)k, (int)d, current_stream(device)), {out});
    });
}

PyMethodDef methods[] = {
    {"dense", (PyCFunction)(void (*)(void))dense, METH_FASTCALL, "custom_kernel's checks and call: the status code, -1 (not taken), or -(bytes of workspace that it wants)"},
    {"quantize", (PyCFunction)(void (*)(void))quantize, METH_FASTCALL, "the quantisers: (codes, scales), the status code, or None (not taken)"},
    {"experts", (PyCFunction)(void (*)(void))experts, METH_FASTCALL, "grouped_kernel and gate_up_silu: the status code, -1 (not taken), or -(bytes of workspace that it wants)"},
    {"topk", (PyCFunction)(void (*)(void))topk, METH_FASTCALL, "moe.topk: the result, the status code, or None (not taken)"},
    {"route", (PyCFunction)(void (*)(void))route, METH_FASTCALL, "moe.route: the results, the status code, or None (not taken)"},
    {"combine", (PyCFunction)(void (*)(void))combine, METH_FASTCALL, "moe.combine: the result, the status code, or None (not taken)"},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_fp8bs_torch", "the compute entry points on torch tensors", -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__fp8bs_torch(void) {
    PyObject* const mod = PyModule_Create(&module);
    if (mod && PyModule_AddStringConstant(mod, "torch_version", FP8BS_TORCH_VERSION) < 0) { Py_DECREF(mod); return nullptr; }
    return mod;
}
