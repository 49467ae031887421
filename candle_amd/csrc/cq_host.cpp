// The host path of a plain call, in native code: a Python module with QTensor.fwd's checks, allocation, workspace and library call in one function.
//
// A one-row product takes the GPU 4.6 us (Q8_0 4096 x 4096) and the Python path 12.9, 5.1 through this function: attribute reads, two lookups of the current stream, the
// workspace's context manager and a ctypes call of 14 arguments.  This function takes what they all come to from the objects themselves, on every call, and keeps nothing between calls.  Whatever is not
// an ordinary call (another tensor type, a tracing or transforming mode, a shape, type or device that the call refuses, a workspace that is missing, too small or in another thread's
// hands) it leaves to the Python path, by returning None: errors are raised and buffers are grown there alone.
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/object_ptr.h>

#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/ops/empty.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/hip/HIPStream.h>

namespace {

using WorkspaceBytes = int64_t (*)(int, int64_t, int64_t, int64_t);
using Forward = int (*)(int, const void *, const void *, int, void *, int, int64_t, int64_t, int64_t, void *, int64_t, void *);
WorkspaceBytes workspace_bytes = nullptr;
Forward forward = nullptr;
PyObject *s_lock, *s_buf, *s_acquire, *s_release;

PyObject *bind(PyObject *, PyObject *args) {
    unsigned long long a, b;
    if (!PyArg_ParseTuple(args, "KK", &a, &b)) return nullptr;
    workspace_bytes = reinterpret_cast<WorkspaceBytes>(a);
    forward = reinterpret_cast<Forward>(b);
    Py_RETURN_NONE;
}

// weights that QMatMul takes: Q4_0, Q4_1, Q5_0, Q5_1, Q8_0, Q2_K .. Q6_K
bool matmul_dtype(long t) { return t == 2 || t == 3 || (t >= 6 && t <= 8) || (t >= 10 && t <= 14); }

// a dense tensor on the GPU with nothing between it and its memory
bool plain(const at::Tensor &t) {
    using K = c10::DispatchKey;
    static constexpr c10::DispatchKeySet usual{K::CUDA, K::ADInplaceOrView, K::AutogradCUDA, K::AutocastCUDA};
    return t.is_cuda() && (t.key_set() | usual) == usual && t.has_storage();
}

// no mode or transform that wants to see the operations of this call
bool eager() {
    using K = c10::DispatchKey;
    static constexpr c10::DispatchKeySet modes{K::Python, K::PythonTLSSnapshot, K::PreDispatch, K::FuncTorchDynamicLayerFrontMode, K::FuncTorchDynamicLayerBackMode, K::Tracer,
                                               K::Functionalize, K::Fake};
    return !c10::impl::tls_local_dispatch_key_set().included_.has_any(modes) && !at::impl::torch_function_mode_enabled();
}

// Gives a lock back, whatever ends the block that holds it.
struct Unlock {
    PyObject *lock;
    ~Unlock() {
        PyObject *type, *value, *trace;
        PyErr_Fetch(&type, &value, &trace);
        PyObject *const r = PyObject_CallMethodNoArgs(lock, s_release);
        if (!r) PyErr_WriteUnraisable(lock);
        Py_XDECREF(r);
        PyErr_Restore(type, value, trace);
    }
};

// qmatmul(xs, blocks, dtype, shape, workspaces) -> the product, a status other than 0 of the library, or None for the Python path
PyObject *qmatmul(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    if (nargs != 5 || !forward || !THPVariable_CheckExact(args[0]) || !THPVariable_CheckExact(args[1]) || !PyTuple_CheckExact(args[3]) || PyTuple_GET_SIZE(args[3]) != 2 ||
        !PyDict_CheckExact(args[4]) || !eager())
        Py_RETURN_NONE;
    const at::Tensor &xs = THPVariable_Unpack(args[0]), &blocks = THPVariable_Unpack(args[1]);
    if (!plain(xs) || !plain(blocks)) Py_RETURN_NONE;
    const long dtype = PyLong_AsLong(args[2]);
    const int64_t n = PyLong_AsLongLong(PyTuple_GET_ITEM(args[3], 0)), k = PyLong_AsLongLong(PyTuple_GET_ITEM(args[3], 1));
    if (PyErr_Occurred()) {
        PyErr_Clear();
        Py_RETURN_NONE;
    }
    const auto type = xs.scalar_type();
    const int cq = type == at::kFloat ? 0 : type == at::kHalf ? 1 : type == at::kBFloat16 ? 30 : -1;
    const int64_t count = xs.numel();
    if (cq < 0 || !matmul_dtype(dtype) || xs.dim() < 2 || k <= 0 || xs.size(-1) != k || count == 0 || !xs.is_contiguous()) Py_RETURN_NONE;
    const auto stream = c10::hip::getCurrentHIPStream();                // of the current device, like the library's launches
    if (stream.device_index() != xs.get_device()) Py_RETURN_NONE;
    const int64_t m = count / k, need = workspace_bytes((int)dtype, m, k, n);
    hipStream_t const s = stream.stream();
    // the stream's scratch buffer, if it is there, large enough and free
    THPObjectPtr key(Py_BuildValue("(iK)", (int)stream.device_index(), (unsigned long long)reinterpret_cast<uintptr_t>(s)));
    if (!key) return nullptr;
    PyObject *const found = PyDict_GetItemWithError(args[4], key.get());
    if (!found) {
        if (PyErr_Occurred()) return nullptr;
        Py_RETURN_NONE;
    }
    Py_INCREF(found);
    THPObjectPtr slot(found), lock(PyObject_GetAttr(found, s_lock));
    if (!lock) return nullptr;
    auto sizes = xs.sizes().vec();
    sizes.back() = n;
    at::Tensor dst = at::empty(sizes, xs.options());
    const void *const w = blocks.const_data_ptr(), *const x = xs.const_data_ptr();
    void *const d = dst.data_ptr();
    THPObjectPtr got(PyObject_CallMethodOneArg(lock.get(), s_acquire, Py_False));
    if (!got) return nullptr;
    if (got.get() != Py_True) Py_RETURN_NONE;
    const Unlock held{lock.get()};
    THPObjectPtr buf(PyObject_GetAttr(slot.get(), s_buf));
    if (!buf) return nullptr;
    if (!THPVariable_Check(buf.get())) Py_RETURN_NONE;
    const at::Tensor &ws = THPVariable_Unpack(buf.get());
    const int64_t bytes = (int64_t)ws.nbytes();
    if (bytes < need) Py_RETURN_NONE;
    void *const scratch = ws.data_ptr();
    int rc;
    Py_BEGIN_ALLOW_THREADS                                              // (the launch may wait for room in the stream's queue)
    rc = forward((int)dtype, w, x, cq, d, cq, m, k, n, scratch, bytes, s);
    Py_END_ALLOW_THREADS
    return rc == 0 ? THPVariable_Wrap(std::move(dst)) : PyLong_FromLong(rc);
    END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {{"bind", bind, METH_VARARGS, "addresses of cq_qmatmul_workspace_bytes and cq_qmatmul_forward"},
                         {"qmatmul", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(qmatmul)), METH_FASTCALL, "QTensor.fwd of an ordinary call, or None"},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host() {
    s_lock = PyUnicode_InternFromString("lock");
    s_buf = PyUnicode_InternFromString("buf");
    s_acquire = PyUnicode_InternFromString("acquire");
    s_release = PyUnicode_InternFromString("release");
    return PyModule_Create(&module);
}
