// Native host path of the attention calls: the checks, allocations, parameter blocks, launches and
// the autograd node of flash_attn.py for the plain case (GPU tensors whose layout the kernels read
// as it is). Anything else returns NotImplemented and takes the Python path, which copies what has
// to be copied and raises what has to be raised.
//
// Why native: torch runs a GPU node's backward on a thread of its own, and there the Python
// backward of a small call took about 60 us (the interpreter's objects move between the cores at
// every call) around kernels of 60 us: 16 x 1024 x 4 heads of 64, forward and backward, 131 us a
// call; a one-token decode spent 22 us in Python around 15 us of kernels.
#include <Python.h>

#include <ATen/TensorSubclassLikeUtils.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cmath>

#include "../../include/mykfa.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

// libmykfa.so's entry points, resolved by the Python side from the library it loaded.
struct Entries {
    decltype(&mykfa_fwd) fwd;
    decltype(&mykfa_fwd_workspace_size) fwd_workspace_size;
    decltype(&mykfa_fwd_grown) fwd_grown;
    decltype(&mykfa_bwd) bwd;
    decltype(&mykfa_bwd_workspace_per_kv_head) bwd_workspace_per_kv_head;
    decltype(&mykfa_decode) decode;
    decltype(&mykfa_decode_num_splits) decode_num_splits;
    decltype(&mykfa_decode_workspace_size) decode_workspace_size;
    decltype(&mykfa_kv_append) kv_append;
} L{};
PyObject* py_check = nullptr;     // _lib.check: raises for a status
PyObject* py_backward = nullptr;  // flash_attn._backward_launch: the stored-dS backward's planning

constexpr int kDecodeMaxQ = 16;
constexpr int64_t kSplitMaxRows = 128 * 224;

// Raises MykfaError for a failed call (the message is this thread's).
void check(int status) {
    if (status == MYKFA_OK) return;
    PyGILState_STATE g = PyGILState_Ensure();
    PyObject* r = PyObject_CallFunction(py_check, "i", status);
    Py_XDECREF(r);
    python_error e;
    e.persist();
    PyGILState_Release(g);
    throw e;
}

// Other Python threads run while this one allocates and launches, which can wait for the device. (The
// arguments are the caller's, who holds them until the call returns.)
struct WithoutGil {
    PyThreadState* state = PyEval_SaveThread();
    WithoutGil() = default;
    WithoutGil(const WithoutGil&) = delete;
    ~WithoutGil() { PyEval_RestoreThread(state); }
};

bool plain(const Tensor& x) {
    return x.is_cuda() && x.layout() == at::kStrided && !at::isTensorSubclassLike(x) && !x._fw_grad(0).defined();
}
// 16-byte rows along head_dim: what _kernel_ready asks for.
bool ready(const Tensor& x) {
    const auto s = x.strides();
    int64_t odd = 0;
    for (size_t i = 0; i + 1 < s.size(); ++i) odd |= s[i];
    return s.back() == 1 && (odd & 7) == 0 && (reinterpret_cast<uintptr_t>(x.const_data_ptr()) & 15) == 0;
}
bool head_dim_ok(int64_t d) { return d == 16 || d == 32 || d == 64 || d == 128 || d == 256; }

// q, k, v as the kernels take them: the checks of _check and _kernel_ready, none of which copies.
bool usable(const Tensor& q, const Tensor& k, const Tensor& v, int64_t dim) {
    if (q.dim() != dim || k.dim() != dim || v.dim() != dim || !plain(q) || !plain(k) || !plain(v)) return false;
    const auto t = q.scalar_type();
    if ((t != at::kBFloat16 && t != at::kHalf) || k.scalar_type() != t || v.scalar_type() != t) return false;
    const int64_t d = q.size(-1);
    if (!head_dim_ok(d) || k.size(-1) != d || v.size(-1) != d) return false;
    if (k.size(-2) == 0 || q.size(-2) % k.size(-2) != 0 || k.size(-2) != v.size(-2)) return false;
    return k.device() == q.device() && v.device() == q.device() && ready(q) && ready(k) && ready(v);
}
bool lengths_ok(const Tensor& x, const Tensor& q) {
    return plain(x) && x.device() == q.device() && x.scalar_type() == at::kInt && x.is_contiguous();
}

hipStream_t stream_of(const Tensor& x) { return c10::hip::getCurrentHIPStream(x.device().index()).stream(); }
mykfa_stream_t abi(hipStream_t s) { return reinterpret_cast<mykfa_stream_t>(s); }

void strides(const Tensor& x, int64_t& b, int64_t& t, int64_t& h) {
    const auto s = x.strides();
    const bool dense = s.size() == 4;
    b = dense ? s[0] : 0;
    t = dense ? s[1] : s[0];
    h = dense ? s[2] : s[1];
}

struct Seqs {
    Tensor cu_q, cu_k, seqused;  // undefined: none
    int64_t max_q, max_k;
    double scale;
    int64_t wl, wr;
    int32_t grown = 0;  // keys past seqused
};

mykfa_fwd_params params(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& out, const Tensor& lse,
                        const Seqs& s) {
    mykfa_fwd_params p{};
    p.q = q.const_data_ptr();
    p.k = k.const_data_ptr();
    p.v = v.const_data_ptr();
    p.o = out.data_ptr();
    p.lse = static_cast<float*>(lse.data_ptr());
    strides(q, p.q_batch_stride, p.q_token_stride, p.q_head_stride);
    strides(k, p.k_batch_stride, p.k_token_stride, p.k_head_stride);
    strides(v, p.v_batch_stride, p.v_token_stride, p.v_head_stride);
    strides(out, p.o_batch_stride, p.o_token_stride, p.o_head_stride);
    p.lse_head_stride = lse.stride(0);
    const bool varlen = s.cu_q.defined();
    if (varlen) {
        p.cu_seqlens_q = static_cast<const int32_t*>(s.cu_q.const_data_ptr());
        p.cu_seqlens_k = static_cast<const int32_t*>(s.cu_k.const_data_ptr());
    }
    if (s.seqused.defined()) p.seqused_k = static_cast<const int32_t*>(s.seqused.const_data_ptr());
    p.batch = (int32_t)(varlen ? s.cu_q.numel() - 1 : q.size(0));
    p.num_heads = (int32_t)q.size(-2);
    p.num_kv_heads = (int32_t)k.size(-2);
    p.head_dim = (int32_t)q.size(-1);
    p.max_seqlen_q = (int32_t)s.max_q;
    p.max_seqlen_k = (int32_t)s.max_k;
    p.window_left = (int32_t)s.wl;
    p.window_right = (int32_t)s.wr;
    p.softmax_scale = (float)s.scale;
    p.dtype = q.scalar_type() == at::kBFloat16 ? MYKFA_BF16 : MYKFA_FP16;
    return p;
}

Tensor workspace(size_t bytes, const Tensor& like) {
    return at::empty({(int64_t)bytes}, like.options().dtype(at::kByte));
}

// Split-K decode with its merge; with kn / vn it first stores them into the caches.
void launch_decode(const mykfa_fwd_params& p, const Tensor& q, const Tensor* kn, const Tensor* vn) {
    mykfa_decode_params d{};
    d.fwd = p;
    d.num_splits = L.decode_num_splits(p.batch, p.num_heads, p.num_kv_heads, p.max_seqlen_q, p.max_seqlen_k);
    if (kn) {
        d.seqlen_new = (int32_t)kn->size(1);
        d.k_new = kn->const_data_ptr();
        d.v_new = vn->const_data_ptr();
        strides(*kn, d.kn_batch_stride, d.kn_token_stride, d.kn_head_stride);
        strides(*vn, d.vn_batch_stride, d.vn_token_stride, d.vn_head_stride);
    }
    const size_t bytes = L.decode_workspace_size(p.batch, p.num_heads, p.max_seqlen_q, p.head_dim, d.num_splits);
    const Tensor ws = workspace(bytes < 16 ? 16 : bytes, q);
    check(L.decode(&d, ws.data_ptr(), ws.numel(), abi(stream_of(q))));
}

// (O, LSE) of flash_attn._forward.
std::pair<Tensor, Tensor> forward(const Tensor& q, const Tensor& k, const Tensor& v, const Seqs& s) {
    const bool varlen = s.cu_q.defined();
    const Tensor out = at::empty(q.sizes(), q.options());
    const Tensor lse = at::empty({q.size(-2), varlen ? q.size(0) : q.size(0) * q.size(1)}, q.options().dtype(at::kFloat));
    const mykfa_fwd_params p = params(q, k, v, out, lse, s);
    const c10::DeviceGuard guard(q.device());
    size_t bytes = 0;
    if (!varlen && s.max_q > 0 && s.max_q <= kDecodeMaxQ) {
        launch_decode(p, q, nullptr, nullptr);
    } else if (!varlen && q.size(0) * q.size(1) * q.size(2) <= kSplitMaxRows && (bytes = L.fwd_workspace_size(&p)) > 0) {
        Tensor ws;
        try {
            ws = workspace(bytes, q);
        } catch (const c10::OutOfMemoryError&) {
            bytes = 0;  // the keys then stay whole
        }
        check(L.fwd_grown(&p, s.grown, bytes ? ws.data_ptr() : nullptr, bytes, abi(stream_of(q))));
    } else if (s.grown > 0) {
        check(L.fwd_grown(&p, s.grown, nullptr, 0, abi(stream_of(q))));
    } else {
        check(L.fwd(&p, abi(stream_of(q))));
    }
    return {out, lse};
}

// (O, LSE) of flash_attn_with_kvcache: k and v appended to the caches, q over the grown lengths.
std::pair<Tensor, Tensor> cached(const Tensor& q, const Tensor& kc, const Tensor& vc, const Tensor& k, const Tensor& v, Seqs& s) {
    const c10::DeviceGuard guard(q.device());
    const int64_t b = q.size(0), nq = q.size(1);
    if (nq <= kDecodeMaxQ) {
        const Tensor out = at::empty(q.sizes(), q.options());
        const Tensor lse = at::empty({q.size(2), b * nq}, q.options().dtype(at::kFloat));
        launch_decode(params(q, kc, vc, out, lse, s), q, &k, &v);
        return {out, lse};
    }
    mykfa_kv_append_params p{};
    p.k_cache = kc.data_ptr();
    p.v_cache = vc.data_ptr();
    p.k_new = k.const_data_ptr();
    p.v_new = v.const_data_ptr();
    p.cache_seqlens = static_cast<const int32_t*>(s.seqused.const_data_ptr());
    strides(kc, p.kc_batch_stride, p.kc_token_stride, p.kc_head_stride);
    strides(vc, p.vc_batch_stride, p.vc_token_stride, p.vc_head_stride);
    strides(k, p.kn_batch_stride, p.kn_token_stride, p.kn_head_stride);
    strides(v, p.vn_batch_stride, p.vn_token_stride, p.vn_head_stride);
    p.batch = (int32_t)b;
    p.seqlen_new = (int32_t)k.size(1);
    p.capacity = (int32_t)kc.size(1);
    p.num_kv_heads = (int32_t)k.size(2);
    p.head_dim = (int32_t)k.size(3);
    p.dtype = k.scalar_type() == at::kBFloat16 ? MYKFA_BF16 : MYKFA_FP16;
    check(L.kv_append(&p, abi(stream_of(q))));
    s.grown = (int32_t)k.size(1);  // (a launch of their addition less: the forward's merge is one more)
    return forward(q, kc, vc, s);
}

Tensor as_ready(const Tensor& x) { return ready(x) ? x : x.contiguous(); }

variable_list backward(Tensor dout, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& out,
                       const Tensor& lse, const Seqs& s) {
    dout = as_ready(dout);
    Tensor dq = at::empty(q.sizes(), q.options()), dk = at::empty(k.sizes(), k.options()),
           dv = at::empty(v.sizes(), v.options()), delta = at::empty(lse.sizes(), lse.options());
    mykfa_bwd_params b{};
    b.fwd = params(q, k, v, out, lse, s);
    b.dout = dout.const_data_ptr();
    b.dq = dq.data_ptr();
    b.dk = dk.data_ptr();
    b.dv = dv.data_ptr();
    b.delta = static_cast<float*>(delta.data_ptr());
    strides(dout, b.do_batch_stride, b.do_token_stride, b.do_head_stride);
    strides(dq, b.dq_batch_stride, b.dq_token_stride, b.dq_head_stride);
    strides(dk, b.dk_batch_stride, b.dk_token_stride, b.dk_head_stride);
    strides(dv, b.dv_batch_stride, b.dv_token_stride, b.dv_head_stride);
    if (L.bwd_workspace_per_kv_head(&b) > 0) {
        // The stored-dS backward plans its passes against the device's memory in Python, with gradients of
        // its own: these go back first, or they would count against the passes.
        for (Tensor* x : {&dq, &dk, &dv, &delta}) x->reset();
        PyGILState_STATE g = PyGILState_Ensure();
        const auto wrap = [](const Tensor& x) -> PyObject* { return x.defined() ? THPVariable_Wrap(x) : Py_NewRef(Py_None); };
        PyObject* r = PyObject_CallFunction(py_backward, "NNNNNNNNLLdLL", wrap(dout), wrap(q), wrap(k), wrap(v), wrap(out),
                                            wrap(lse), wrap(s.cu_q), wrap(s.cu_k), (long long)s.max_q, (long long)s.max_k,
                                            s.scale, (long long)s.wl, (long long)s.wr);
        if (r == nullptr) {
            python_error e;
            e.persist();
            PyGILState_Release(g);
            throw e;
        }
        variable_list got;
        for (int i = 0; i < 3; ++i) got.push_back(THPVariable_Unpack(PyTuple_GET_ITEM(r, i)));
        Py_DECREF(r);
        PyGILState_Release(g);
        return got;
    }
    const c10::DeviceGuard guard(q.device());
    check(L.bwd(&b, abi(stream_of(q))));
    return {dq, dk, dv};
}

struct FlashAttn : torch::autograd::Function<FlashAttn> {
    static variable_list forward(AutogradContext* ctx, const Tensor& q, const Tensor& k, const Tensor& v, const Seqs* s,
                                 bool with_lse) {
        auto [out, lse] = ::forward(q, k, v, *s);
        ctx->save_for_backward({q, k, v, out, lse, s->cu_q, s->cu_k});
        ctx->saved_data["s"] = c10::IValue(std::vector<int64_t>{s->max_q, s->max_k, s->wl, s->wr});
        ctx->saved_data["c"] = c10::IValue(s->scale);
        ctx->set_materialize_grads(false);  // an unused output gets no zero-filled gradient
        if (!with_lse) return {out};
        ctx->mark_non_differentiable({lse});
        return {out, lse};
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        variable_list got(5);
        if (!grads[0].defined()) return got;
        const auto t = ctx->get_saved_variables();
        const auto n = ctx->saved_data["s"].toIntVector();
        const Seqs s{t[5], t[6], Tensor(), n[0], n[1], ctx->saved_data["c"].toDouble(), n[2], n[3]};
        variable_list g = ::backward(grads[0], as_ready(t[0]), as_ready(t[1]), as_ready(t[2]), as_ready(t[3]), t[4], s);
        for (int i = 0; i < 3; ++i) got[i] = g[i];
        return got;
    }
};

bool tensor_arg(PyObject* o) { return THPVariable_Check(o); }

// The window as offsets (flash_attn.py:435-439), false unless the tuple holds two integers.
bool window_arg(PyObject* window, bool causal, int64_t& wl, int64_t& wr) {
    if (!PyTuple_Check(window) || PyTuple_GET_SIZE(window) != 2) return false;
    PyObject *l = PyTuple_GET_ITEM(window, 0), *r = PyTuple_GET_ITEM(window, 1);
    if (!PyLong_Check(l) || !PyLong_Check(r)) return false;
    int over = 0, over2 = 0;
    wl = PyLong_AsLongLongAndOverflow(l, &over);
    wr = PyLong_AsLongLongAndOverflow(r, &over2);
    if (over || over2 || wl > MYKFA_UNBOUNDED || wr > MYKFA_UNBOUNDED) return false;
    if (wl < 0) wl = MYKFA_UNBOUNDED;
    wr = causal ? 0 : (wr < 0 ? MYKFA_UNBOUNDED : wr);
    return true;
}
bool scale_arg(PyObject* o, int64_t d, double& scale) {
    if (o == Py_None) {
        scale = 1.0 / std::sqrt((double)d);
        return true;
    }
    if (!PyFloat_Check(o)) return false;
    scale = PyFloat_AS_DOUBLE(o);
    return true;
}
bool int_arg(PyObject* o, int64_t& x) {
    if (!PyLong_CheckExact(o)) return false;
    int over = 0;
    x = PyLong_AsLongLongAndOverflow(o, &over);
    return !over && x >= 0 && x <= INT32_MAX;
}

// attention(q, k, v, cu_q, cu_k, max_q, max_k, causal, window, scale, with_lse): cu_q None = dense.
PyObject* attention(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 11 || !tensor_arg(a[0]) || !tensor_arg(a[1]) || !tensor_arg(a[2])) Py_RETURN_NOTIMPLEMENTED;
    const Tensor &q = THPVariable_Unpack(a[0]), &k = THPVariable_Unpack(a[1]), &v = THPVariable_Unpack(a[2]);
    const bool varlen = a[3] != Py_None;
    if (!usable(q, k, v, varlen ? 3 : 4)) Py_RETURN_NOTIMPLEMENTED;
    Seqs s;
    if (varlen) {
        if (!tensor_arg(a[3]) || !tensor_arg(a[4]) || !int_arg(a[5], s.max_q) || !int_arg(a[6], s.max_k)) Py_RETURN_NOTIMPLEMENTED;
        s.cu_q = THPVariable_Unpack(a[3]);
        s.cu_k = THPVariable_Unpack(a[4]);
        if (!lengths_ok(s.cu_q, q) || !lengths_ok(s.cu_k, q)) Py_RETURN_NOTIMPLEMENTED;
    } else {
        s.max_q = q.size(1);
        s.max_k = k.size(1);
    }
    if (!window_arg(a[8], a[7] == Py_True, s.wl, s.wr) || !PyBool_Check(a[7]) ||
        !scale_arg(a[9], q.size(-1), s.scale))
        Py_RETURN_NOTIMPLEMENTED;
    if (!PyBool_Check(a[10])) Py_RETURN_NOTIMPLEMENTED;
    const bool with_lse = a[10] == Py_True;
    variable_list r;
    {
        const WithoutGil threads;
        if (at::GradMode::is_enabled() && (q.requires_grad() || k.requires_grad() || v.requires_grad())) {
            r = FlashAttn::apply(q, k, v, &s, with_lse);
        } else {
            auto [out, lse] = forward(q, k, v, s);
            r = {out, lse};
        }
    }
    if (!with_lse) return THPVariable_Wrap(r[0]);
    return Py_BuildValue("NN", THPVariable_Wrap(r[0]), THPVariable_Wrap(r[1]));
    END_HANDLE_TH_ERRORS
}

// kvcache(q, k_cache, v_cache, k, v, cache_seqlens, causal, window, scale, with_lse).
PyObject* kvcache(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 10) Py_RETURN_NOTIMPLEMENTED;
    for (int i = 0; i < 6; ++i)
        if (!tensor_arg(a[i])) Py_RETURN_NOTIMPLEMENTED;
    const Tensor &q = THPVariable_Unpack(a[0]), &kc = THPVariable_Unpack(a[1]), &vc = THPVariable_Unpack(a[2]),
                 &k = THPVariable_Unpack(a[3]), &v = THPVariable_Unpack(a[4]), &lens = THPVariable_Unpack(a[5]);
    if (!usable(q, kc, vc, 4) || !usable(q, k, v, 4) || !lengths_ok(lens, q) || lens.dim() != 1) Py_RETURN_NOTIMPLEMENTED;
    const int64_t b = q.size(0), nq = q.size(1), cap = kc.size(1);
    const std::array<int64_t, 4> want = {b, k.size(1), kc.size(2), kc.size(3)};
    if (k.sizes() != at::IntArrayRef(want) || v.sizes() != at::IntArrayRef(want) || lens.size(0) != b || kc.size(0) != b ||
        vc.sizes() != kc.sizes() || b == 0 || nq == 0 || k.size(1) == 0)
        Py_RETURN_NOTIMPLEMENTED;
    Seqs s;
    s.seqused = lens;
    s.max_q = nq;
    s.max_k = cap;
    if (!window_arg(a[7], a[6] == Py_True, s.wl, s.wr) || !PyBool_Check(a[6]) || !PyBool_Check(a[9]) ||
        !scale_arg(a[8], q.size(-1), s.scale))
        Py_RETURN_NOTIMPLEMENTED;
    Tensor out, lse;
    {
        const WithoutGil threads;
        const at::NoGradGuard no_grad;
        std::tie(out, lse) = cached(q, kc, vc, k, v, s);
    }
    if (a[9] != Py_True) return THPVariable_Wrap(out);
    return Py_BuildValue("NN", THPVariable_Wrap(out), THPVariable_Wrap(lse));
    END_HANDLE_TH_ERRORS
}

// setup(addresses of the entry points in Entries' order, _lib.check, _backward_launch)
PyObject* setup(PyObject*, PyObject* const* a, Py_ssize_t n) {
    constexpr Py_ssize_t N = sizeof(Entries) / sizeof(void*);
    if (n != N + 2) {
        PyErr_SetString(PyExc_TypeError, "setup takes the entry points, the status check and the backward");
        return nullptr;
    }
    void** to = reinterpret_cast<void**>(&L);
    for (Py_ssize_t i = 0; i < N; ++i) {
        to[i] = PyLong_AsVoidPtr(a[i]);
        if (to[i] == nullptr) {
            if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "an entry point is NULL");
            return nullptr;
        }
    }
    Py_XSETREF(py_check, Py_NewRef(a[N]));
    Py_XSETREF(py_backward, Py_NewRef(a[N + 1]));
    Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"attention", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(attention)), METH_FASTCALL, nullptr},
    {"kvcache", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(kvcache)), METH_FASTCALL, nullptr},
    {"setup", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(setup)), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host(void) { return PyModule_Create(&module); }
