// CPython extension _pe_torch: the launches of the package's kernels on torch tensors with their
// argument checks and output allocation in native code. A short batch's forward is bound by host
// time (some hundred launches of a few microseconds each); the same checks in Python cost more than
// the torch operations they replace. An attention call on 32 queries (5.7 us of kernel) takes 20.1 us
// through the torch operator and its Python body and 7.2 us from here, calls back to back; the
// 22-layer forward of 8 queries 3.84 ms with the norms and gates alone launched here, 2.99 ms with
// attention and RoPE.
//
// Each function returns None for a call it does not serve: another dtype or device, rows that are
// not 16-byte pieces, a gradient, or anything that has to see the torch operations themselves
// (autocast, tracing, function transforms, forward-mode derivatives, dispatch and function modes,
// tensor subclasses). The caller then takes the general path: torch's operations for the layer's
// norm and gate, the registered torch operators for attention and RoPE, which also raise the errors.
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

#include <cstring>

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

// A dense tensor on the current HIP device that records nothing and is what it says (no subclass,
// wrapper, batched stand-in without storage, lazy conjugation or forward derivative).
bool plain_any(PyObject *obj, const Tensor *&out, at::ScalarType type) {
    if (!THPVariable_CheckExact(obj)) return false;
    const Tensor &t = THPVariable_Unpack(obj);
    static const c10::DispatchKeySet wrapped({DispatchKey::FuncTorchGradWrapper, DispatchKey::FuncTorchBatched,
                                              DispatchKey::Functionalize, DispatchKey::Python, DispatchKey::Conjugate,
                                              DispatchKey::Negative, DispatchKey::ZeroTensor});
    if (!t.defined() || !t.has_storage() || !t.is_cuda() || t.scalar_type() != type || t.layout() != at::kStrided ||
        t.key_set().has_any(wrapped) || t.get_device() != c10::hip::current_device())
        return false;
    if (t.requires_grad() && c10::GradMode::is_enabled()) return false;
    if (t._fw_grad(0).defined()) return false;
    out = &t;
    return true;
}

bool aligned16(const Tensor &t) { return (reinterpret_cast<uintptr_t>(t.const_data_ptr()) & 15) == 0; }

// A plain bf16 tensor, contiguous from a 16-byte boundary.
bool plain_tensor(PyObject *obj, const Tensor *&out) {
    return plain_any(obj, out, at::kBFloat16) && out->is_contiguous() && aligned16(*out);
}

// A plain bf16 [tokens, heads, head_dim] whose rows are 16-byte pieces.
bool plain_rows(PyObject *obj, const Tensor *&out) {
    return plain_any(obj, out, at::kBFloat16) && out->dim() == 3 && out->stride(2) == 1 && aligned16(*out) &&
           out->stride(0) % 8 == 0 && out->stride(1) % 8 == 0;
}

bool plain_bounds(PyObject *obj, const Tensor *&out) {
    return plain_any(obj, out, at::kInt) && out->dim() == 1 && out->is_contiguous();
}

// RoPE tables [rows, d] or [.., rows, d], both alike.
bool plain_tables(PyObject *cos_obj, PyObject *sin_obj, int64_t d, const Tensor *&cos, const Tensor *&sin) {
    return plain_tensor(cos_obj, cos) && plain_tensor(sin_obj, sin) && (cos->dim() == 2 || cos->dim() == 3) &&
           cos->size(-1) == d && cos->sizes() == sin->sizes() && cos->numel() > 0 && cos->numel() / d <= INT32_MAX;
}

hipStream_t stream_of(const Tensor &t) { return c10::hip::getCurrentHIPStream(t.get_device()).stream(); }

// Allocations and launches run without the interpreter lock: either can wait (a full queue, an
// allocator that synchronises to free memory), and the process's other Python threads, host
// callbacks among them, go on meanwhile. Everything they need is read from the tensors before; no
// Python call is made inside.
class Unlocked {
  public:
    Unlocked() : state_(PyEval_SaveThread()) {}
    ~Unlocked() { PyEval_RestoreThread(state_); }
    Unlocked(const Unlocked &) = delete;
    Unlocked &operator=(const Unlocked &) = delete;

  private:
    PyThreadState *state_;
};

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
    const auto sizes = x->sizes().vec();
    const auto options = x->options();
    const void *src = x->const_data_ptr(), *res = add ? r->const_data_ptr() : nullptr, *weight = w->const_data_ptr();
    const int64_t rows = x->numel() / cols;
    const hipStream_t stream = stream_of(*x);
    Tensor out, sum;
    int status;
    {
        Unlocked unlocked;
        out = at::empty(sizes, options);
        if (add) sum = at::empty(sizes, options);
        status = pe_layer_norm_fwd(src, res, weight, add ? sum.mutable_data_ptr() : nullptr, out.mutable_data_ptr(), rows,
                                   (int32_t)cols, (float)eps, stream);
    }
    if (failed(status, "pe_layer_norm_fwd")) return nullptr;
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
    const auto options = x->options();
    const void *src = x->const_data_ptr();
    const int64_t rows = x->numel() / both;
    const hipStream_t stream = stream_of(*x);
    Tensor out;
    int status;
    {
        Unlocked unlocked;
        out = at::empty(sizes, options);
        status = pe_geglu_fwd(src, out.mutable_data_ptr(), rows, (int32_t)(both / 2), stream);
    }
    if (failed(status, "pe_geglu_fwd")) return nullptr;
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// rope_rows(positions [T] int64, max_positions, d, theta) -> (cos, sin) [1, T, d] bf16, or None
PyObject *rope_rows(PyObject *, PyObject *const *args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 4) {
        PyErr_SetString(PyExc_TypeError, "rope_rows takes positions, max_positions, d and theta");
        return nullptr;
    }
    const int64_t max_positions = PyLong_AsLongLong(args[1]), d = PyLong_AsLongLong(args[2]);
    if (PyErr_Occurred()) return nullptr;
    const double theta = PyFloat_AsDouble(args[3]);
    if (theta == -1.0 && PyErr_Occurred()) return nullptr;
    const Tensor *pos = nullptr;
    if (max_positions < 0 || (d != 64 && d != 128 && d != 256) || !(theta > 0.0) || !plain_thread() ||
        !plain_any(args[0], pos, at::kLong) || pos->dim() != 1 || !pos->is_contiguous() || pos->numel() == 0)
        Py_RETURN_NONE;
    const int64_t sizes[3] = {1, pos->numel(), d};
    const auto options = pos->options().dtype(at::kBFloat16);
    const int64_t *positions = static_cast<const int64_t *>(pos->const_data_ptr());
    const hipStream_t stream = stream_of(*pos);
    Tensor cos, sin;
    int status;
    {
        Unlocked unlocked;
        cos = at::empty(sizes, options);
        sin = at::empty(sizes, options);
        status = pe_rope_gather_fwd(positions, max_positions, (float)theta, sizes[1], (int32_t)d, cos.mutable_data_ptr(),
                                    sin.mutable_data_ptr(), stream);
    }
    if (failed(status, "pe_rope_gather_fwd")) return nullptr;
    PyObject *pair = PyTuple_New(2);
    if (!pair) return nullptr;
    PyTuple_SET_ITEM(pair, 0, THPVariable_Wrap(std::move(cos)));
    PyTuple_SET_ITEM(pair, 1, THPVariable_Wrap(std::move(sin)));
    return pair;
    END_HANDLE_TH_ERRORS
}

// rope(qkv [.., 3 h d], h, d, cos, sin) -> (q, k) [.., h, d], or None
PyObject *rope(PyObject *, PyObject *const *args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 5) {
        PyErr_SetString(PyExc_TypeError, "rope takes qkv, h, d, cos and sin");
        return nullptr;
    }
    const int64_t h = PyLong_AsLongLong(args[1]), d = PyLong_AsLongLong(args[2]);
    if (PyErr_Occurred()) return nullptr;
    const Tensor *qkv = nullptr, *cos = nullptr, *sin = nullptr;
    if (h < 1 || h > (1 << 20) || (d != 64 && d != 128 && d != 256) || !plain_thread() || !plain_tensor(args[0], qkv) ||
        !plain_tables(args[3], args[4], d, cos, sin))
        Py_RETURN_NONE;
    const int64_t width = 3 * h * d;
    if (!qkv->dim() || qkv->size(-1) != width || qkv->numel() == 0 || qkv->numel() / width > INT32_MAX) Py_RETURN_NONE;
    auto sizes = qkv->sizes().vec();
    sizes.back() = h;
    sizes.push_back(d);
    const auto options = qkv->options();
    const hipStream_t stream = stream_of(*qkv);
    pe_rope_args a;
    std::memset(&a, 0, sizeof(a));
    a.struct_size = sizeof(a);
    a.dtype = PE_ATTN_DTYPE_BF16;
    a.qkv = qkv->const_data_ptr();
    a.cos = cos->const_data_ptr();
    a.sin = sin->const_data_ptr();
    a.qkv_stride_row = width;
    a.table_stride_row = d;
    a.table_rows = (int32_t)(cos->numel() / d);
    a.n_rows = (int32_t)(qkv->numel() / width);
    a.n_heads = (int32_t)h;
    a.head_dim = (int32_t)d;
    Tensor q, k;
    int status;
    {
        Unlocked unlocked;
        q = at::empty(sizes, options);
        k = at::empty(sizes, options);
        a.q_out = q.mutable_data_ptr();
        a.k_out = k.mutable_data_ptr();
        status = pe_rope_qkv_fwd(&a, stream);
    }
    if (failed(status, "pe_rope_qkv_fwd")) return nullptr;
    PyObject *pair = PyTuple_New(2);
    if (!pair) return nullptr;
    PyTuple_SET_ITEM(pair, 0, THPVariable_Wrap(std::move(q)));
    PyTuple_SET_ITEM(pair, 1, THPVariable_Wrap(std::move(k)));
    return pair;
    END_HANDLE_TH_ERRORS
}

// The attention calls' arguments past their tensors, in the order Python passes them.
struct Options {
    int64_t max_seqlen, window_left, window_right, causal, short_max, max_seqlen_k, band_kernel, min_seqlen;
    double scale;
    void *args;  // a pe_attn_args to fill instead of launching, or NULL

    // false with a Python exception set, or (ok = false) for a value no kernel argument holds
    bool parse(PyObject *const *a, bool &ok) {
        int64_t *ints[8] = {&max_seqlen, &window_left, &window_right, &causal, &short_max, &max_seqlen_k, &band_kernel,
                            &min_seqlen};
        ok = true;
        for (int i = 0; i < 8; ++i) {
            *ints[i] = PyLong_AsLongLong(a[i]);
            if (*ints[i] == -1 && PyErr_Occurred()) return false;
            ok = ok && *ints[i] >= INT32_MIN && *ints[i] <= INT32_MAX;
        }
        scale = PyFloat_AsDouble(a[8]);
        if (scale == -1.0 && PyErr_Occurred()) return false;
        args = PyLong_AsVoidPtr(a[9]);
        return args || !PyErr_Occurred();
    }
    static constexpr int kCount = 10;
};

// Completes `a` (q, k, v and the tables filled in), allocates the output shaped `sizes` and either
// launches the whole call, returning the output, or hands the arguments over: (output, stream).
PyObject *finish(pe_attn_args &a, const Options &o, const Tensor &like, at::IntArrayRef sizes, const Tensor &cu) {
    a.struct_size = sizeof(a);
    a.dtype = PE_ATTN_DTYPE_BF16;
    a.cu_seqlens = static_cast<const int32_t *>(cu.const_data_ptr());
    a.n_seq = (int32_t)(cu.numel() - 1);
    a.max_seqlen = (int32_t)o.max_seqlen;
    a.softmax_scale = (float)o.scale;
    a.window_left = (int32_t)o.window_left;
    a.window_right = (int32_t)o.window_right;
    a.causal = o.causal ? 1 : 0;
    a.short_max = (int32_t)o.short_max;
    a.band_kernel = (int32_t)o.band_kernel;
    a.min_seqlen = (int32_t)o.min_seqlen;
    a.o_stride_head = a.head_dim;
    a.o_stride_token = (int64_t)a.n_heads_q * a.head_dim;
    const auto shape = sizes.vec();
    const auto options = like.options();
    const hipStream_t stream = stream_of(like);
    Tensor out, workspace;
    const char *what = "pe_attn_workspace_size";
    int status = PE_ATTN_OK;
    {
        Unlocked unlocked;
        out = at::empty(shape, options);
        a.o = out.mutable_data_ptr();
        size_t bytes = 0;
        if (!o.args) status = pe_attn_workspace_size(&a, &bytes);
        if (!o.args && status == PE_ATTN_OK) {
            if (bytes) workspace = at::empty({(int64_t)bytes}, options.dtype(at::kByte));
            what = "pe_varlen_attn_fwd";
            status = pe_varlen_attn_fwd(&a, bytes ? workspace.mutable_data_ptr() : nullptr, bytes, stream);
        }
    }
    if (failed(status, what)) return nullptr;
    if (o.args) {
        std::memcpy(o.args, &a, sizeof(a));
        PyObject *pair = PyTuple_New(2);
        if (!pair) return nullptr;
        PyTuple_SET_ITEM(pair, 0, THPVariable_Wrap(std::move(out)));
        PyTuple_SET_ITEM(pair, 1, PyLong_FromVoidPtr(stream));
        return pair;
    }
    return THPVariable_Wrap(std::move(out));
}

// attention(q, k, v, cu, gate or None, cu_k or None, cos or None, sin or None, *Options)
PyObject *attention(PyObject *, PyObject *const *args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 8 + Options::kCount) {
        PyErr_SetString(PyExc_TypeError, "attention takes its eight tensors and ten options");
        return nullptr;
    }
    Options o;
    bool ok;
    if (!o.parse(args + 8, ok)) return nullptr;
    const Tensor *q = nullptr, *k = nullptr, *v = nullptr, *cu = nullptr, *g = nullptr, *cuk = nullptr, *cos = nullptr,
                 *sin = nullptr;
    const bool gated = args[4] != Py_None, own_keys = args[5] != Py_None, rotate = args[6] != Py_None;
    if (!ok || !plain_thread() || !plain_rows(args[0], q) || !plain_rows(args[1], k) || !plain_rows(args[2], v) ||
        !plain_bounds(args[3], cu) || (gated && !plain_rows(args[4], g)) || (own_keys && !plain_bounds(args[5], cuk)) ||
        rotate != (args[7] != Py_None) || (rotate && !plain_tables(args[6], args[7], q->size(2), cos, sin)))
        Py_RETURN_NONE;
    const int64_t hkv = k->size(1);
    if (k->sizes() != v->sizes() || q->size(2) != k->size(2) || (!own_keys && q->size(0) != k->size(0)) || hkv < 1 ||
        q->size(1) % hkv || (gated && g->sizes() != q->sizes()) || (own_keys && cuk->numel() != cu->numel()) ||
        q->size(0) == 0 || q->size(0) > INT32_MAX || k->size(0) > INT32_MAX || q->size(1) > INT32_MAX ||
        q->size(2) > 256 || cu->numel() < 2 || cu->numel() > INT32_MAX)
        Py_RETURN_NONE;
    pe_attn_args a;
    std::memset(&a, 0, sizeof(a));
    a.q = q->const_data_ptr();
    a.k = k->const_data_ptr();
    a.v = v->const_data_ptr();
    a.q_stride_token = q->stride(0);
    a.q_stride_head = q->stride(1);
    a.k_stride_token = k->stride(0);
    a.k_stride_head = k->stride(1);
    a.v_stride_token = v->stride(0);
    a.v_stride_head = v->stride(1);
    if (gated) {
        a.gate = g->const_data_ptr();
        a.gate_stride_token = g->stride(0);
        a.gate_stride_head = g->stride(1);
    }
    a.total_tokens = (int32_t)q->size(0);
    a.n_heads_q = (int32_t)q->size(1);
    a.n_heads_kv = (int32_t)hkv;
    a.head_dim = (int32_t)q->size(2);
    if (own_keys) {
        a.cu_seqlens_k = static_cast<const int32_t *>(cuk->const_data_ptr());
        a.total_tokens_k = (int32_t)k->size(0);
        a.max_seqlen_k = (int32_t)o.max_seqlen_k;
    }
    if (rotate) {
        a.rope_cos = cos->const_data_ptr();
        a.rope_sin = sin->const_data_ptr();
        a.rope_table_stride = a.head_dim;
        a.rope_table_rows = (int32_t)(cos->numel() / a.head_dim);
    }
    return finish(a, o, *q, q->sizes(), *cu);
    END_HANDLE_TH_ERRORS
}

// attention_qkv(qkv [1, tokens, 3 h d], h, d, cu, cos, sin, *Options): RoPE and attention from the
// packed projection, the output [1, tokens, h d]
PyObject *attention_qkv(PyObject *, PyObject *const *args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 6 + Options::kCount) {
        PyErr_SetString(PyExc_TypeError, "attention_qkv takes qkv, h, d, cu, cos, sin and ten options");
        return nullptr;
    }
    Options o;
    bool ok;
    if (!o.parse(args + 6, ok)) return nullptr;
    const int64_t h = PyLong_AsLongLong(args[1]), d = PyLong_AsLongLong(args[2]);
    if (PyErr_Occurred()) return nullptr;
    const Tensor *qkv = nullptr, *cu = nullptr, *cos = nullptr, *sin = nullptr;
    if (!ok || h < 1 || h > (1 << 20) || (d != 64 && d != 128) || !plain_thread() || !plain_tensor(args[0], qkv) ||
        !plain_bounds(args[3], cu) || !plain_tables(args[4], args[5], d, cos, sin))
        Py_RETURN_NONE;
    const int64_t width = 3 * h * d;
    if (qkv->dim() != 3 || qkv->size(0) != 1 || qkv->size(2) != width || qkv->size(1) == 0 || qkv->size(1) > INT32_MAX ||
        cu->numel() < 2 || cu->numel() > INT32_MAX)
        Py_RETURN_NONE;
    pe_attn_args a;
    std::memset(&a, 0, sizeof(a));
    const char *base = static_cast<const char *>(qkv->const_data_ptr());
    a.q = base;
    a.k = base + 2 * h * d;
    a.v = base + 4 * h * d;
    a.q_stride_token = a.k_stride_token = a.v_stride_token = width;
    a.q_stride_head = a.k_stride_head = a.v_stride_head = d;
    a.total_tokens = (int32_t)qkv->size(1);
    a.n_heads_q = a.n_heads_kv = (int32_t)h;
    a.head_dim = (int32_t)d;
    a.rope_cos = cos->const_data_ptr();
    a.rope_sin = sin->const_data_ptr();
    a.rope_table_stride = d;
    a.rope_table_rows = (int32_t)(cos->numel() / d);
    const int64_t sizes[3] = {1, qkv->size(1), h * d};
    return finish(a, o, *qkv, sizes, *cu);
    END_HANDLE_TH_ERRORS
}

#define PE_FASTCALL(f) reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(f)), METH_FASTCALL

PyMethodDef methods[] = {
    {"layer_norm", PE_FASTCALL(layer_norm), "layer_norm(x, residual, weight, eps) -> out, (sum, out) or None"},
    {"geglu", geglu, METH_O, "geglu(proj) -> out or None"},
    {"rope_rows", PE_FASTCALL(rope_rows), "rope_rows(positions, max_positions, d, theta) -> (cos, sin) or None"},
    {"rope", PE_FASTCALL(rope), "rope(qkv, h, d, cos, sin) -> (q, k) or None"},
    {"attention", PE_FASTCALL(attention),
     "attention(q, k, v, cu, gate, cu_k, cos, sin, max_seqlen, window_left, window_right, causal, short_max, "
     "max_seqlen_k, band_kernel, min_seqlen, scale, args) -> out, (out, stream) or None"},
    {"attention_qkv", PE_FASTCALL(attention_qkv),
     "attention_qkv(qkv, h, d, cu, cos, sin, max_seqlen, window_left, window_right, causal, short_max, max_seqlen_k, "
     "band_kernel, min_seqlen, scale, args) -> out, (out, stream) or None"},
    {nullptr, nullptr, 0, nullptr},
};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_pe_torch", "Native launches of the package's kernels on torch tensors", -1,
                      methods};

}  // namespace

PyMODINIT_FUNC PyInit__pe_torch() {
    if (pe_attn_abi_version() != PE_ATTN_ABI_VERSION) {
        PyErr_Format(PyExc_ImportError, "_pe_torch was built for ABI %d of libpe_attn.so, which has %d", PE_ATTN_ABI_VERSION,
                     pe_attn_abi_version());
        return nullptr;
    }
    return PyModule_Create(&module);
}
