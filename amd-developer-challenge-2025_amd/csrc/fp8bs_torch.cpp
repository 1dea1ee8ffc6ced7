// custom_kernel on torch tensors, for callers that issue many small products from Python: its checks and its call in one native
// function.  In Python they were some forty attribute reads and comparisons; here they are read from the tensors themselves, at
// every call.  Calls issued one after another: 256 x 512 x 1024 5.2 us before, 4.1 now (the kernel takes 3.8), 3 x 2092 x 384 5.2
// and 3.6, 1 x 3968 x 384 5.3 and 3.9; with tensors that were not seen before 24 and 16, waiting for each.
// Whatever is not the usual case (another layout, type or device, an empty product, a tensor subclass, a size that has not been
// planned yet) is handed back: the Python path takes it, or says what is wrong with it.
// Built by build.py with the host compiler against torch's headers; without this module the Python path takes every call.
#define PY_SSIZE_T_CLEAN
#include <torch/csrc/autograd/python_variable.h>
#include <ATen/ATen.h>
#include <c10/hip/HIPStream.h>
#include <hip/hip_runtime_api.h>

#include <exception>

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

PyMethodDef methods[] = {
    {"dense", (PyCFunction)(void (*)(void))dense, METH_FASTCALL, "custom_kernel's checks and call: the status code, -1 (not taken), or -(bytes of workspace that it wants)"},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_fp8bs_torch", "custom_kernel's checks and call on torch tensors", -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__fp8bs_torch(void) {
    PyObject* const mod = PyModule_Create(&module);
    if (mod && PyModule_AddStringConstant(mod, "torch_version", FP8BS_TORCH_VERSION) < 0) { Py_DECREF(mod); return nullptr; }
    return mod;
}
