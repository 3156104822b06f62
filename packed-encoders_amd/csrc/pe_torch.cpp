// CPython extension _pe_torch: the launches of the encoder layer's small kernels with their argument
// checks and output allocation in native code. A short batch's forward is bound by host time (some
// hundred launches of a few microseconds each); the same checks in Python cost more than the torch
// operations they replace.
//
// Each function returns None for a call its kernel does not serve, which the caller runs in torch:
// another dtype or device, rows that are not contiguous 16-byte pieces, a gradient, or anything that
// has to see the torch operations themselves (autocast, tracing, function transforms, forward-mode
// derivatives, dispatch and function modes, tensor subclasses).
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/autocast_mode.h>
#include <c10/core/GradMode.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/pe_attn.h"

namespace {

using at::Tensor;
using c10::DispatchKey;

// Whether nothing on this thread has to see torch operations instead of a kernel launch.
bool plain_thread() {
    static const c10::DispatchKeySet watched(
        {DispatchKey::FuncTorchDynamicLayerFrontMode, DispatchKey::FuncTorchVmapMode, DispatchKey::FuncTorchGradWrapper,
         DispatchKey::FuncTorchBatched, DispatchKey::Functionalize, DispatchKey::Tracer, DispatchKey::Python,
         DispatchKey::PythonDispatcher, DispatchKey::PreDispatch});
    return !c10::impl::tls_local_dispatch_key_set().included_.has_any(watched) &&
           !at::autocast::is_autocast_enabled(at::kCUDA) && !at::impl::torch_function_mode_enabled() &&
           !c10::impl::TorchDispatchModeTLS::any_modes_set();
}

// A dense bf16 tensor on the current HIP device, contiguous from a 16-byte boundary, that records
// nothing and is what it says (no subclass, wrapper, lazy conjugation or forward derivative).
bool plain_tensor(PyObject *obj, const Tensor *&out) {
    if (!THPVariable_CheckExact(obj)) return false;
    const Tensor &t = THPVariable_Unpack(obj);
    static const c10::DispatchKeySet wrapped({DispatchKey::FuncTorchGradWrapper, DispatchKey::FuncTorchBatched,
                                              DispatchKey::Functionalize, DispatchKey::Python, DispatchKey::Conjugate,
                                              DispatchKey::Negative, DispatchKey::ZeroTensor});
    if (!t.defined() || !t.is_cuda() || t.scalar_type() != at::kBFloat16 || t.layout() != at::kStrided ||
        t.key_set().has_any(wrapped))
        return false;
    if (!t.is_contiguous() || (reinterpret_cast<uintptr_t>(t.const_data_ptr()) & 15) ||
        t.get_device() != c10::hip::current_device())
        return false;
    if (t.requires_grad() && c10::GradMode::is_enabled()) return false;
    if (t._fw_grad(0).defined()) return false;
    out = &t;
    return true;
}

hipStream_t stream_of(const Tensor &t) { return c10::hip::getCurrentHIPStream(t.get_device()).stream(); }

// The exception _lib.check raises for a status, or false for none.
bool failed(int status, const char *what) {
    if (status == PE_ATTN_OK) return false;
    PyErr_Format(status == PE_ATTN_ELAUNCH ? PyExc_RuntimeError : PyExc_ValueError, "%s: %s (%d)", what,
                 pe_attn_strerror(status), status);
    return true;
}

// layer_norm(x, residual or None, weight, eps) -> out, (sum, out) with a residual, or None
PyObject *layer_norm(PyObject *, PyObject *const *args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 4) {
        PyErr_SetString(PyExc_TypeError, "layer_norm takes x, residual, weight and eps");
        return nullptr;
    }
    const bool add = args[1] != Py_None;
    const Tensor *x = nullptr, *r = nullptr, *w = nullptr;
    if (!plain_thread() || !plain_tensor(args[0], x) || !plain_tensor(args[2], w) || (add && !plain_tensor(args[1], r)))
        Py_RETURN_NONE;
    const int64_t cols = x->dim() ? x->size(-1) : 0;
    if (cols < 8 || cols % 8 || cols > PE_LAYER_NORM_MAX_COLS || w->dim() != 1 || w->size(0) != cols ||
        (add && r->sizes() != x->sizes()))
        Py_RETURN_NONE;
    const double eps = PyFloat_AsDouble(args[3]);
    if (eps == -1.0 && PyErr_Occurred()) return nullptr;
    Tensor out = at::empty(x->sizes(), x->options());
    Tensor sum = add ? at::empty(x->sizes(), x->options()) : Tensor();
    if (failed(pe_layer_norm_fwd(x->const_data_ptr(), add ? r->const_data_ptr() : nullptr, w->const_data_ptr(),
                                 add ? sum.mutable_data_ptr() : nullptr, out.mutable_data_ptr(), x->numel() / cols,
                                 (int32_t)cols, (float)eps, stream_of(*x)),
               "pe_layer_norm_fwd"))
        return nullptr;
    if (!add) return THPVariable_Wrap(std::move(out));
    PyObject *pair = PyTuple_New(2);
    if (!pair) return nullptr;
    PyTuple_SET_ITEM(pair, 0, THPVariable_Wrap(std::move(sum)));
    PyTuple_SET_ITEM(pair, 1, THPVariable_Wrap(std::move(out)));
    return pair;
    END_HANDLE_TH_ERRORS
}

// geglu(proj) -> out, or None
PyObject *geglu(PyObject *, PyObject *arg) {
    HANDLE_TH_ERRORS
    const Tensor *x = nullptr;
    if (!plain_thread() || !plain_tensor(arg, x)) Py_RETURN_NONE;
    const int64_t both = x->dim() ? x->size(-1) : 0;
    if (both < 16 || both % 16 || both / 2 > INT32_MAX) Py_RETURN_NONE;
    auto sizes = x->sizes().vec();
    sizes.back() = both / 2;
    Tensor out = at::empty(sizes, x->options());
    if (failed(pe_geglu_fwd(x->const_data_ptr(), out.mutable_data_ptr(), x->numel() / both, (int32_t)(both / 2),
                            stream_of(*x)),
               "pe_geglu_fwd"))
        return nullptr;
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {
    {"layer_norm", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(layer_norm)), METH_FASTCALL,
     "layer_norm(x, residual, weight, eps) -> out, (sum, out) or None"},
    {"geglu", geglu, METH_O, "geglu(proj) -> out or None"},
    {nullptr, nullptr, 0, nullptr},
};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_pe_torch", "Native launches of the encoder layer's small kernels", -1,
                      methods};

}  // namespace

PyMODINIT_FUNC PyInit__pe_torch() { return PyModule_Create(&module); }
