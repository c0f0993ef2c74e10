// Python calls of the dequant-matmul without an interpreter's worth of
// argument handling: reads the tensors' pointers and strides, allocates the
// outputs and the workspace from torch's caching allocator and calls the C
// ABI of include/epure_hip.h, in one native call per linear.
//
// What a 4096 x 4096 token costs is this path, not the kernel: the launch
// parameters gathered in Python and passed through ctypes took 16.7 us a
// call around a 5.3 us kernel.  Nothing is kept between calls: every pointer,
// stride and flag is read from the tensors again.
//
// Host code only (no HIP header): the current stream's handle comes from
// torch, the entry points' addresses from the loaded library.
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/core/GradMode.h>
#include <c10/core/impl/LocalDispatchKeySet.h>

#include <stdint.h>

#include "epure_hip.h"

namespace {

decltype(&ep_dequant_matmul_workspace) fn_ws;
decltype(&ep_dequant_matmul) fn_matmul;
decltype(&ep_dequant_matmul_bwd_workspace) fn_bwd_ws;
decltype(&ep_dequant_matmul_bwd) fn_backward;
decltype(&ep_last_error) fn_error;
PyObject *fn_stream;  // torch._C._cuda_getCurrentRawStream

// EP_F32 / EP_F16 / EP_BF16, or -1.
int dtype_code(const at::Tensor &t)
{
    switch (t.scalar_type()) {
    case at::kFloat:
        return EP_F32;
    case at::kHalf:
        return EP_F16;
    case at::kBFloat16:
        return EP_BF16;
    default:
        return -1;
    }
}

// A call that a torch mode, a functorch transform or a tensor wrapper wants
// to see: those take the path through torch's operators.
bool plain_call()
{
    static const c10::DispatchKeySet seen(
        {c10::DispatchKey::Python, c10::DispatchKey::PythonTLSSnapshot, c10::DispatchKey::FuncTorchDynamicLayerFrontMode,
         c10::DispatchKey::FuncTorchDynamicLayerBackMode, c10::DispatchKey::FuncTorchVmapMode,
         c10::DispatchKey::VmapMode, c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper,
         c10::DispatchKey::Functionalize, c10::DispatchKey::Tracer});
    return !c10::impl::tls_local_dispatch_key_set().included_.has_any(seen) && !at::impl::torch_function_mode_enabled();
}

bool plain_tensor(PyObject *o)
{
    if (!THPVariable_CheckExact(o))
        return false;
    static const c10::DispatchKeySet wrapped(
        {c10::DispatchKey::Python, c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper,
         c10::DispatchKey::Functionalize, c10::DispatchKey::Negative, c10::DispatchKey::ZeroTensor});
    const at::Tensor &t = THPVariable_Unpack(o);
    return t.defined() && t.layout() == at::kStrided && t.unsafeGetTensorImpl()->has_storage() &&
           !t.key_set().has_any(wrapped);
}

struct Weight {
    const uint8_t *packed;
    const void *scale, *cb;
    int scale_dt, cb_dt, levels, group;
    int64_t ld_scale, n, k;
};

// The launch parameters of a packed store's tensors; false where the kernels
// do not read them as they are (a Python caller declines those).
bool weight(const at::Tensor &packed, const at::Tensor &scale, const at::Tensor &cb, int64_t n, int64_t k, int levels,
            int group, Weight &w)
{
    w = Weight{};
    w.scale_dt = dtype_code(scale);
    w.cb_dt = dtype_code(cb);
    if (w.scale_dt < 0 || w.cb_dt < 0 || !packed.is_contiguous() || !cb.is_contiguous() || scale.dim() == 0 ||
        (scale.dim() == 2 && scale.stride(1) != 1))
        return false;
    w.packed = (const uint8_t *)packed.const_data_ptr();
    w.scale = scale.const_data_ptr();
    w.cb = cb.const_data_ptr();
    w.ld_scale = scale.dim() == 2 ? scale.stride(0) : scale.size(-1);
    w.n = n;
    w.k = k;
    w.levels = levels;
    w.group = group;
    return true;
}

// The current stream of the tensor's device (nullptr and *ok false: a Python
// error is set).  A host tensor is refused here: its device index, -1, names
// the current device's stream to torch, and the kernels would read host memory.
void *stream_of(const at::Tensor &t, bool *ok)
{
    TORCH_CHECK_VALUE(t.is_cuda(), "expected a GPU tensor, but got one on ", t.device());
    PyObject *idx = PyLong_FromLong(t.get_device());
    PyObject *r = idx ? PyObject_CallOneArg(fn_stream, idx) : nullptr;
    Py_XDECREF(idx);
    void *s = r ? PyLong_AsVoidPtr(r) : nullptr;
    Py_XDECREF(r);
    *ok = !PyErr_Occurred();
    return s;
}

at::Tensor bytes_like(const at::Tensor &t, size_t n)
{
    return n ? at::empty({(int64_t)n}, t.options().dtype(at::kByte).requires_grad(false)) : at::Tensor();
}

PyObject *failed(const char *what, int rc)
{
    return PyErr_Format(PyExc_RuntimeError, "%s failed (%d): %s", what, rc, fn_error());
}

// y = x2 . W^T, `out` given or of x2's type.  A new reference to y, None
// where the library declines, nullptr with an error set.
PyObject *run_matmul(const at::Tensor &x2, const Weight &w, at::Tensor out, const at::Tensor &shown, bool accumulate)
{
    const int64_t m = x2.size(0), k = x2.size(1);
    bool ok;
    void *stream = stream_of(x2, &ok);
    if (!ok)
        return nullptr;
    const size_t need = fn_ws(m, w.n, k, w.levels, w.group);
    at::Tensor ws = bytes_like(x2, need);
    const int xdt = dtype_code(x2), ydt = dtype_code(out);
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = fn_matmul(x2.const_data_ptr(), xdt, x2.stride(0), w.packed, w.scale, w.scale_dt, w.ld_scale, w.cb, w.cb_dt,
                   w.levels, w.group, m, w.n, k, out.data_ptr(), ydt, out.stride(0), accumulate ? EP_FLAG_ACCUMULATE : 0,
                   need ? ws.data_ptr() : nullptr, need, stream);
    Py_END_ALLOW_THREADS
    if (rc < 0)
        return failed("ep_dequant_matmul", rc);
    if (rc > 0)
        Py_RETURN_NONE;
    return THPVariable_Wrap(shown);
}

bool args_are(Py_ssize_t n, Py_ssize_t want)
{
    if (n == want)
        return true;
    PyErr_Format(PyExc_TypeError, "%zd arguments wanted, %zd given", want, n);
    return false;
}

bool tensors(PyObject *const *args, int n)
{
    for (int i = 0; i < n; ++i)
        if (!THPVariable_Check(args[i])) {
            PyErr_Format(PyExc_TypeError, "argument %d is not a tensor", i);
            return false;
        }
    return true;
}

// linear(x, packed, scale, cb, N, K, levels, group, serve_f32): the whole of
// an inference call.  None: declined.  NotImplemented: the caller's path
// through torch's operators takes it (autograd, a torch mode, a tensor
// subclass, an empty or mismatched x).
PyObject *linear(PyObject *, PyObject *const *args, Py_ssize_t nargs)
{
    HANDLE_TH_ERRORS
    if (!args_are(nargs, 9))
        return nullptr;
    if (!plain_call())
        Py_RETURN_NOTIMPLEMENTED;
    for (int i = 0; i < 4; ++i)
        if (!plain_tensor(args[i]))
            Py_RETURN_NOTIMPLEMENTED;
    const at::Tensor &x = THPVariable_Unpack(args[0]), &packed = THPVariable_Unpack(args[1]);
    const at::Tensor &scale = THPVariable_Unpack(args[2]), &cb = THPVariable_Unpack(args[3]);
    const int64_t n = PyLong_AsLongLong(args[4]), k = PyLong_AsLongLong(args[5]);
    const int levels = (int)PyLong_AsLong(args[6]), group = (int)PyLong_AsLong(args[7]);
    const bool f32 = PyObject_IsTrue(args[8]) == 1;
    if (PyErr_Occurred())
        return nullptr;
    if (!x.is_cuda() || !packed.is_cuda() || !scale.is_cuda() || !cb.is_cuda() || x.dim() < 1 || x.numel() == 0 ||
        x.size(-1) != k)
        Py_RETURN_NOTIMPLEMENTED;
    if (c10::GradMode::is_enabled() && (x.requires_grad() || cb.requires_grad() || scale.requires_grad()))
        Py_RETURN_NOTIMPLEMENTED;
    const int xdt = dtype_code(x);
    if (xdt < 0 || (xdt == EP_F32 && !f32))
        Py_RETURN_NONE;
    Weight w;
    if (!weight(packed, scale, cb, n, k, levels, group, w))
        Py_RETURN_NONE;
    at::Tensor x2 = x.dim() == 2 ? x : x.reshape({-1, k});
    if (x2.stride(1) != 1)
        x2 = x2.contiguous();
    at::DimVector shape(x.sizes().begin(), x.sizes().end());
    shape.back() = n;
    const at::Tensor y = at::empty(shape, x.options().requires_grad(false));
    return run_matmul(x2, w, x.dim() == 2 ? y : y.view({x2.size(0), n}), y, false);
    END_HANDLE_TH_ERRORS
}

// matmul(x2, packed, scale, cb, N, levels, group, out or None, accumulate)
PyObject *matmul(PyObject *, PyObject *const *args, Py_ssize_t nargs)
{
    HANDLE_TH_ERRORS
    if (!args_are(nargs, 9) || !tensors(args, 4))
        return nullptr;
    const at::Tensor &x2 = THPVariable_Unpack(args[0]);
    const int64_t n = PyLong_AsLongLong(args[4]);
    const int levels = (int)PyLong_AsLong(args[5]), group = (int)PyLong_AsLong(args[6]);
    const bool acc = PyObject_IsTrue(args[8]) == 1;
    if (PyErr_Occurred())
        return nullptr;
    TORCH_CHECK_VALUE(x2.dim() == 2, "x must be 2-D");
    if (args[7] != Py_None && !tensors(args + 7, 1))
        return nullptr;
    Weight w;
    if (!weight(THPVariable_Unpack(args[1]), THPVariable_Unpack(args[2]), THPVariable_Unpack(args[3]), n, x2.size(1),
                levels, group, w))
        Py_RETURN_NONE;
    const at::Tensor out = args[7] == Py_None ? at::empty({x2.size(0), n}, x2.options().requires_grad(false))
                                              : THPVariable_Unpack(args[7]);
    return run_matmul(x2, w, out, out, acc);
    END_HANDLE_TH_ERRORS
}

// backward(gy2, x2, packed, scale, cb, N, levels, group, need_x, need_cb,
// need_scale, grad_x's dtype as a tensor of it or None): (grad_x, grad_cb,
// grad_scale), None for each that is not needed; None where declined.
PyObject *backward(PyObject *, PyObject *const *args, Py_ssize_t nargs)
{
    HANDLE_TH_ERRORS
    if (!args_are(nargs, 12) || !tensors(args, 5))
        return nullptr;
    const at::Tensor &gy = THPVariable_Unpack(args[0]), &x2 = THPVariable_Unpack(args[1]);
    const int64_t n = PyLong_AsLongLong(args[5]);
    const int levels = (int)PyLong_AsLong(args[6]), group = (int)PyLong_AsLong(args[7]);
    bool need[3];
    for (int i = 0; i < 3; ++i)
        need[i] = PyObject_IsTrue(args[8 + i]) == 1;
    const long gxdt = args[11] == Py_None ? -1 : PyLong_AsLong(args[11]);
    if (PyErr_Occurred())
        return nullptr;
    TORCH_CHECK_VALUE(gy.dim() == 2 && x2.dim() == 2 && gy.size(1) == n && group > 0 && levels > 0,
                      "gy must be [M, N] and x [M, K]");
    const int64_t m = gy.size(0), k = x2.size(1), g = (k + group - 1) / group;
    Weight w;
    if (!weight(THPVariable_Unpack(args[2]), THPVariable_Unpack(args[3]), THPVariable_Unpack(args[4]), n, k, levels,
                group, w))
        Py_RETURN_NONE;
    const auto opt = x2.options().requires_grad(false);
    const auto gxt = gxdt == EP_F32    ? at::kFloat
                     : gxdt == EP_F16  ? at::kHalf
                     : gxdt == EP_BF16 ? at::kBFloat16
                                       : x2.scalar_type();
    at::Tensor out[3];
    if (need[0])
        out[0] = at::empty({m, k}, opt.dtype(gxt));
    if (need[1])
        out[1] = at::empty({levels}, opt.dtype(at::kFloat));
    if (need[2])
        out[2] = at::empty({n, g}, opt.dtype(at::kFloat));
    bool ok;
    void *stream = stream_of(x2, &ok);
    if (!ok)
        return nullptr;
    const size_t nb = fn_bwd_ws(m, n, k, levels, group);
    at::Tensor ws = bytes_like(x2, nb);
    const int gydt = dtype_code(gy), xdt = dtype_code(x2);
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = fn_backward(gy.const_data_ptr(), gydt, gy.stride(0), x2.const_data_ptr(), xdt, x2.stride(0), w.packed, w.scale,
                     w.scale_dt, w.ld_scale, w.cb, w.cb_dt, w.levels, w.group, m, n, k,
                     need[0] ? out[0].data_ptr() : nullptr, need[0] ? dtype_code(out[0]) : xdt, k,
                     need[1] ? (float *)out[1].data_ptr() : nullptr, need[2] ? (float *)out[2].data_ptr() : nullptr, g,
                     nb ? ws.data_ptr() : nullptr, nb, stream);
    Py_END_ALLOW_THREADS
    if (rc < 0)
        return failed("ep_dequant_matmul_bwd", rc);
    if (rc > 0)
        Py_RETURN_NONE;
    PyObject *r = PyTuple_New(3);
    for (int i = 0; r && i < 3; ++i) {
        PyObject *v = need[i] ? THPVariable_Wrap(out[i]) : Py_NewRef(Py_None);
        if (!v) {
            Py_DECREF(r);
            return nullptr;
        }
        PyTuple_SET_ITEM(r, i, v);
    }
    return r;
    END_HANDLE_TH_ERRORS
}

// bind(matmul_workspace, matmul, bwd_workspace, bwd, last_error, stream_fn):
// addresses of the C ABI's entry points and torch's raw-stream lookup.
PyObject *bind(PyObject *, PyObject *const *args, Py_ssize_t nargs)
{
    if (!args_are(nargs, 6))
        return nullptr;
    fn_ws = (decltype(fn_ws))PyLong_AsVoidPtr(args[0]);
    fn_matmul = (decltype(fn_matmul))PyLong_AsVoidPtr(args[1]);
    fn_bwd_ws = (decltype(fn_bwd_ws))PyLong_AsVoidPtr(args[2]);
    fn_backward = (decltype(fn_backward))PyLong_AsVoidPtr(args[3]);
    fn_error = (decltype(fn_error))PyLong_AsVoidPtr(args[4]);
    if (PyErr_Occurred())
        return nullptr;
    fn_stream = Py_NewRef(args[5]);
    Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"bind", (PyCFunction)(void (*)(void))bind, METH_FASTCALL, nullptr},
    {"linear", (PyCFunction)(void (*)(void))linear, METH_FASTCALL, nullptr},
    {"matmul", (PyCFunction)(void (*)(void))matmul, METH_FASTCALL, nullptr},
    {"backward", (PyCFunction)(void (*)(void))backward, METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "epure_torch", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_epure_torch(void) { return PyModule_Create(&module); }
