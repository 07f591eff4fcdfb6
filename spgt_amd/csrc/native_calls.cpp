// The operators that training steps and small inputs call most, from Python straight to the C ABI: operand checks, outputs
// and workspaces from torch's allocator, the current stream, the launch.  A function here takes only the plain case (exact
// torch.Tensor or Parameter, float32, on the current device, contiguous, sizes that match, nothing that records or replaces
// operators) and returns None for any other, and for calls that the C ABI refuses: the Python operator of the same name
// then does the call, or raises what it raises.  Per call, Python operator and this: 128 -> 128 linear of 100 tokens 9.8
// and 4.8 us in a loop, of which the launch takes 3.
// The first argument is the library object that the caller would use; another one than the bound one is not served.
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>

#include "../../include/spgt_hip.h"

namespace {

PyObject* g_lib = nullptr;  // borrowed: the Python module that binds it keeps it

#define SPGT_FUNCTIONS(X)                                                                                              \
    X(spgt_linear_forward) X(spgt_linear_input_grad) X(spgt_linear_weight_grad) X(spgt_linear_weight_grad_out_major)   \
    X(spgt_linear_weight_grad_workspace_bytes) X(spgt_galerkin_attention_fused_forward)                                \
    X(spgt_galerkin_attention_fused_workspace_bytes) X(spgt_galerkin_attention_fused_backward)                         \
    X(spgt_galerkin_attention_fused_backward_workspace_bytes) X(spgt_encoder_tail_forward) X(spgt_encoder_layer_pays)  \
    X(spgt_encoder_layer_forward) X(spgt_encoder_layer_workspace_bytes) X(spgt_truncated_dft_rows_forward)             \
    X(spgt_truncated_dft_rows_inverse) X(spgt_spectral_modes_middle) X(spgt_spectral_modes_middle_workspace_bytes)     \
    X(spgt_spectral_inverse_linear) X(spgt_conv3x3_forward) X(spgt_conv3x3_workspace_bytes)                            \
    X(spgt_multihead_projection_with_position_rrc_forward)                                                             \
    X(spgt_multihead_projection_layernorm_with_position_rrc_forward) X(spgt_galerkin_attention_cccr_forward)           \
    X(spgt_galerkin_attention_cccr_workspace_bytes) X(spgt_galerkin_attention_cccr_backward)                           \
    X(spgt_galerkin_attention_cccr_backward_workspace_bytes) X(spgt_heads_feature_to_token_major)                      \
    X(spgt_projection_input_grad) X(spgt_layernorm_heads_backward) X(spgt_layernorm_heads_backward_workspace_bytes)
#define SPGT_POINTER(name) decltype(&::name) p_##name = nullptr;
SPGT_FUNCTIONS(SPGT_POINTER)
#undef SPGT_POINTER

// Nothing records or replaces the operators that this thread runs.
bool eager() {
    return !at::impl::torch_function_mode_enabled() && !c10::impl::dispatch_mode_enabled() && !torch::jit::tracer::isTracing();
}

// Classes of tensors whose data pointer is not the whole story.
const c10::DispatchKeySet kWrapped({c10::DispatchKey::Python, c10::DispatchKey::FuncTorchBatched,
                                    c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::Batched,
                                    c10::DispatchKey::Functionalize, c10::DispatchKey::Conjugate,
                                    c10::DispatchKey::Negative, c10::DispatchKey::ZeroTensor});

struct Call {
    PyObject* const* args;
    bool ok = true;
    c10::DeviceIndex device = -1;
    hipStream_t stream = nullptr;

    explicit Call(PyObject* const* a) : args(a) {}

    // Argument i as a float32 tensor (or `type`) on the current device, of any strides
    const at::Tensor* strided(int i, at::ScalarType type = at::kFloat) {
        if (!ok || !THPVariable_CheckExact(args[i])) return miss();
        const at::Tensor& t = THPVariable_Unpack(args[i]);
        if (!t.defined() || !t.is_cuda() || t.scalar_type() != type || t.layout() != c10::kStrided || t.key_set().has_any(kWrapped))
            return miss();
        if (device < 0) {
            device = t.device().index();
            if (device != c10::hip::current_device()) return miss();
            stream = c10::hip::getCurrentHIPStream(device).stream();
        } else if (t.device().index() != device) {
            return miss();
        }
        return &t;
    }
    const at::Tensor* tensor(int i, at::ScalarType type = at::kFloat) {
        const at::Tensor* t = strided(i, type);
        return t && t->is_contiguous() ? t : miss();
    }
    // A vector of n values; None where `optional`
    const float* vector(int i, int64_t n, bool optional) {
        if (optional && args[i] == Py_None) return nullptr;
        const at::Tensor* t = tensor(i);
        if (t && t->numel() != n) t = miss();
        return t ? t->const_data_ptr<float>() : nullptr;
    }
    // Positions [B, S, d]; None where `optional`
    const float* positions(int i, int64_t B, int64_t S, int64_t d, bool optional) {
        if (optional && args[i] == Py_None) return nullptr;
        const at::Tensor* t = tensor(i);
        if (t && !(t->dim() == 3 && t->size(0) == B && t->size(1) == S && t->size(2) == d)) t = miss();
        return t ? t->const_data_ptr<float>() : nullptr;
    }
    int64_t integer(int i) {
        const int64_t v = PyLong_AsLongLong(args[i]);
        if (v == -1 && PyErr_Occurred()) PyErr_Clear(), ok = false;
        return v;
    }
    double real(int i) {
        const double v = PyFloat_AsDouble(args[i]);
        if (v == -1.0 && PyErr_Occurred()) PyErr_Clear(), ok = false;
        return v;
    }
    void require(bool condition) { ok = ok && condition; }
    const at::Tensor* miss() {
        ok = false;
        return nullptr;
    }
    at::Tensor empty(at::IntArrayRef sizes, at::ScalarType type = at::kFloat) const {
        return at::empty(sizes, at::TensorOptions().dtype(type).device(c10::Device(c10::kCUDA, device)));
    }
    at::Tensor workspace(size_t bytes) const { return empty({(int64_t)std::max<size_t>(bytes, 16)}, at::kByte); }
};

const float* data(const at::Tensor* t) { return t->const_data_ptr<float>(); }
bool aligned16(const at::Tensor& t) { return (reinterpret_cast<uintptr_t>(t.const_data_ptr()) & 15u) == 0; }

template <class F, class... A>
int launch(F fn, A... a) {
    int rc;
    Py_BEGIN_ALLOW_THREADS;  // a launch may wait for room in the queue
    rc = fn(a...);
    Py_END_ALLOW_THREADS;
    return rc;
}

PyObject* wrap(const at::Tensor& t) { return THPVariable_Wrap(t); }
template <class... T>
PyObject* wrap_all(const T&... t) {
    PyObject* tuple = PyTuple_New(sizeof...(t));
    if (!tuple) return nullptr;
    Py_ssize_t i = 0;
    (PyTuple_SET_ITEM(tuple, i++, THPVariable_Wrap(t)), ...);
    return tuple;
}

// Every function: `n` arguments after the library; C++ exceptions (an allocation that fails) become None, and the Python
// operator meets the same condition.
#define SPGT_NATIVE(name, n)                                                           \
    PyObject* name##_body(PyObject* const* args);                                      \
    PyObject* name(PyObject*, PyObject* const* args, Py_ssize_t nargs) {               \
        if (nargs != (n) + 1 || !g_lib || args[0] != g_lib || !eager()) Py_RETURN_NONE; \
        try {                                                                          \
            return name##_body(args + 1);                                              \
        } catch (const std::exception&) {                                              \
            Py_RETURN_NONE;                                                            \
        }                                                                              \
    }                                                                                  \
    PyObject* name##_body(PyObject* const* args)

// x [..., K], weight [K, N], bias or None, residual or None, activation, residual after the activation, planes
SPGT_NATIVE(linear, 7) {
    Call c(args);
    const at::Tensor *x = c.tensor(0), *w = c.tensor(1);
    const int64_t act = c.integer(4), after = c.integer(5), planes = c.integer(6);
    if (!c.ok || x->dim() < 1 || w->dim() != 2 || x->size(-1) != w->size(0) || planes < 1) Py_RETURN_NONE;
    const int64_t K = w->size(0), N = w->size(1), T = x->numel() / std::max<int64_t>(K, 1);
    const float* bias = c.vector(2, N, true);
    const float* res = c.vector(3, T * N, true);
    if (c.ok && res) {  // of two dimensions: rows of the result, of any other: its values
        const at::Tensor& r = THPVariable_Unpack(args[3]);
        c.require(r.dim() != 2 || r.size(1) == N);
    }
    c.require(T > 0 && N % planes == 0 && (N / planes) % 32 == 0 && aligned16(*x));
    if (!c.ok) Py_RETURN_NONE;
    c10::SmallVector<int64_t, 6> sizes;
    if (planes > 1) sizes.push_back(planes);
    for (int64_t d = 0; d + 1 < x->dim(); ++d) sizes.push_back(x->size(d));
    const int64_t pc = N / planes;
    sizes.push_back(pc);
    const at::Tensor out = c.empty(sizes);
    const int mode = !res ? SPGT_RES_NONE : after ? SPGT_RES_AFTER_ACT : SPGT_RES_BEFORE_ACT;
    if (launch(p_spgt_linear_forward, data(x), K, data(w), bias, res, res ? N : 0, mode, (int)act, nullptr, (int64_t)0, nullptr,
               0, out.data_ptr<float>(), pc, (int)pc, T * pc, T, (int)K, (int)N, c.stream))
        Py_RETURN_NONE;
    return wrap(out);
}

// grad [..., N], weight [N, K], add or None, ReLU's output or None
SPGT_NATIVE(input_grad, 4) {
    Call c(args);
    const at::Tensor *g = c.tensor(0), *w = c.tensor(1);
    if (!c.ok || g->dim() < 1 || w->dim() != 2 || g->size(-1) != w->size(0)) Py_RETURN_NONE;
    const int64_t N = w->size(0), K = w->size(1), T = g->numel() / std::max<int64_t>(N, 1);
    const float *add = c.vector(2, T * K, true), *relu = c.vector(3, T * K, true);
    c.require(T > 0 && !(add && relu));
    if (!c.ok) Py_RETURN_NONE;
    c10::SmallVector<int64_t, 6> sizes(g->sizes().begin(), g->sizes().end());
    sizes.back() = K;
    const at::Tensor out = c.empty(sizes);
    if (launch(p_spgt_linear_input_grad, data(g), N, (int64_t)0, data(w), nullptr, nullptr, 1, add, relu, out.data_ptr<float>(), T,
               (int)N, (int)K, c.stream))
        Py_RETURN_NONE;
    return wrap(out);
}

// grad [..., C], weight [C, C] (used as x @ W)
SPGT_NATIVE(projection_input_grad, 2) {
    Call c(args);
    const at::Tensor *g = c.tensor(0), *w = c.tensor(1);
    if (!c.ok || g->dim() < 1 || w->dim() != 2 || g->numel() == 0) Py_RETURN_NONE;
    const int64_t C = g->size(-1);
    if (w->size(0) != C || w->size(1) != C || C > INT32_MAX) Py_RETURN_NONE;
    const at::Tensor out = c.empty(g->sizes());
    if (launch(p_spgt_projection_input_grad, data(g), C, data(w), out.data_ptr<float>(), g->numel() / C, (int)C, c.stream))
        Py_RETURN_NONE;
    return wrap(out);
}

// grads [3, T, C], three weights [C, C], add or None
SPGT_NATIVE(packed_input_grad, 5) {
    Call c(args);
    const at::Tensor* g = c.tensor(0);
    if (!c.ok || g->dim() != 3 || g->size(0) != 3 || g->size(1) < 1) Py_RETURN_NONE;
    const int64_t T = g->size(1), C = g->size(2);
    const float* w[3];
    for (int i = 0; i < 3; ++i) {
        const at::Tensor* t = c.tensor(1 + i);
        if (!t || t->dim() != 2 || t->size(0) != C || t->size(1) != C) Py_RETURN_NONE;
        w[i] = data(t);
    }
    const float* add = c.vector(4, T * C, true);
    if (!c.ok) Py_RETURN_NONE;
    const at::Tensor out = c.empty({T, C});
    if (launch(p_spgt_linear_input_grad, data(g), C, T * C, w[0], w[1], w[2], 3, add, nullptr, out.data_ptr<float>(), T, (int)C,
               (int)C, c.stream))
        Py_RETURN_NONE;
    return wrap(out);
}

// x [..., K], grad [..., N], out-major: (dW, db)
SPGT_NATIVE(weight_grad, 3) {
    Call c(args);
    const at::Tensor *x = c.tensor(0), *g = c.tensor(1);
    const bool out_major = c.integer(2) != 0;
    if (!c.ok || x->dim() < 1 || g->dim() < 1) Py_RETURN_NONE;
    const int64_t K = x->size(-1), N = g->size(-1);
    if (K < 1 || N < 1 || x->numel() / K != g->numel() / N || (out_major && K % 4)) Py_RETURN_NONE;
    const int64_t T = x->numel() / K;
    const size_t bytes = K <= INT32_MAX && N <= INT32_MAX ? p_spgt_linear_weight_grad_workspace_bytes(T, (int)K, (int)N, 1) : 0;
    if (bytes == 0) Py_RETURN_NONE;
    const at::Tensor ws = c.workspace(bytes), out = c.empty({K * N + N});
    if (launch(out_major ? p_spgt_linear_weight_grad_out_major : p_spgt_linear_weight_grad, data(x), K, (int64_t)0, data(g), N,
               (int64_t)0, out.data_ptr<float>(), ws.data_ptr(), (size_t)ws.numel(), T, (int)K, (int)N, 1, c.stream))
        Py_RETURN_NONE;
    const int64_t rows = out_major ? N : K, columns = out_major ? K : N;
    return wrap_all(out.as_strided({rows, columns}, {columns, 1}, 0), out.as_strided({N}, {1}, K * N));
}

// x [..., K], grads [P, ..., N]: (dW [P, K, N], db [P, N])
SPGT_NATIVE(weight_grad_batched, 2) {
    Call c(args);
    const at::Tensor *x = c.tensor(0), *g = c.tensor(1);
    if (!c.ok || x->dim() < 1 || g->dim() < 2) Py_RETURN_NONE;
    const int64_t K = x->size(-1), N = g->size(-1), P = g->size(0);
    if (K < 1 || N < 1 || P < 1 || P > 64 || K > INT32_MAX || N > INT32_MAX || x->numel() / K * P != g->numel() / N) Py_RETURN_NONE;
    const int64_t T = x->numel() / K;
    const size_t bytes = p_spgt_linear_weight_grad_workspace_bytes(T, (int)K, (int)N, (int)P);
    if (bytes == 0) Py_RETURN_NONE;
    const int64_t E = K * N + N;
    const at::Tensor ws = c.workspace(bytes), out = c.empty({P, E});
    if (launch(p_spgt_linear_weight_grad, data(x), K, (int64_t)0, data(g), N, T * N, out.data_ptr<float>(), ws.data_ptr(),
               (size_t)ws.numel(), T, (int)K, (int)N, (int)P, c.stream))
        Py_RETURN_NONE;
    return wrap_all(out.as_strided({P, K, N}, {E, N, 1}, 0), out.as_strided({P, N}, {E, 1}, K * N));
}

struct Attention {
    const float *q, *k, *v, *pos = nullptr, *ln[4];
    int64_t B = 0, S = 0, H = 0, dp = 0, D = 0;
    float eps = 0.f;
    // arguments: Q, K, V from `first` on, position, four LayerNorm parameters; `tail` holds eps, num_head, dim_position
    Attention(Call& c, int first, int eps_at, int heads_at) {
        H = c.integer(heads_at), dp = c.integer(heads_at + 1);
        eps = (float)c.real(eps_at);
        const at::Tensor* t[3];
        for (int i = 0; i < 3; ++i) t[i] = c.tensor(first + i);
        c.require(H > 0 && H <= 1024 && (dp == 0 || dp == 2));
        if (!c.ok) return;
        c.require(t[0]->dim() == 3 && t[0]->size(2) == H * 32 && t[0]->sizes() == t[1]->sizes() && t[0]->sizes() == t[2]->sizes());
        if (!c.ok) return;
        B = t[0]->size(0), S = t[0]->size(1), D = dp + 32;
        q = data(t[0]), k = data(t[1]), v = data(t[2]);
        for (int i = 0; i < 4; ++i) ln[i] = c.vector(first + 4 + i, H * 32, false);
        if (dp) pos = c.positions(first + 3, B, S, 2, false);
        c.require(B > 0 && S > 0 && B <= INT32_MAX && S <= INT32_MAX);
    }
};

// Q, K, V, position, gK, bK, gV, bV, eps, num_head, dim_position: (out, K^T V / S)
SPGT_NATIVE(attention_forward, 11) {
    Call c(args);
    const Attention a(c, 0, 8, 9);
    if (!c.ok) Py_RETURN_NONE;
    const size_t bytes = p_spgt_galerkin_attention_fused_workspace_bytes((int)a.B, (int)a.S, (int)a.H, (int)a.dp);
    const at::Tensor out = c.empty({a.B, a.S, a.H * a.D}), ktv = c.empty({a.B, a.H, a.D, a.D}), ws = c.workspace(bytes);
    if (launch(p_spgt_galerkin_attention_fused_forward, a.q, a.k, a.v, a.H * 32, a.pos, a.ln[0], a.ln[1], a.ln[2], a.ln[3], a.eps,
               out.data_ptr<float>(), ktv.data_ptr<float>(), ws.data_ptr(), (size_t)ws.numel(), (int)a.B, (int)a.S, (int)a.H,
               (int)a.dp, c.stream))
        Py_RETURN_NONE;
    return wrap_all(out, ktv);
}

// grad_out, Q, K, V, position, gK, bK, gV, bV, eps, ktv, num_head, dim_position: (dQ, dK, dV, dgK, dbK, dgV, dbV)
SPGT_NATIVE(attention_backward, 13) {
    Call c(args);
    const at::Tensor* g = c.tensor(0);
    const Attention a(c, 1, 9, 11);
    const at::Tensor* ktv = c.tensor(10);
    if (!c.ok || g->dim() != 3 || g->size(0) != a.B || g->size(1) != a.S || g->size(2) != a.H * a.D ||
        ktv->sizes() != at::IntArrayRef({a.B, a.H, a.D, a.D}))
        Py_RETURN_NONE;
    const size_t bytes = p_spgt_galerkin_attention_fused_backward_workspace_bytes((int)a.B, (int)a.S, (int)a.H, (int)a.dp);
    if (bytes == 0) Py_RETURN_NONE;
    const int64_t C = a.H * 32, plane = a.B * a.S * C;
    const at::Tensor ws = c.workspace(bytes), grads = c.empty({3, a.B, a.S, C}), ln = c.empty({4, a.H, 32});
    float* d = grads.data_ptr<float>();
    if (launch(p_spgt_galerkin_attention_fused_backward, data(g), a.q, a.k, a.v, C, a.pos, a.ln[0], a.ln[1], a.ln[2], a.ln[3],
               a.eps, data(ktv), d, d + plane, d + 2 * plane, C, ln.data_ptr<float>(), ws.data_ptr(), (size_t)ws.numel(), (int)a.B,
               (int)a.S, (int)a.H, (int)a.dp, c.stream))
        Py_RETURN_NONE;
    auto part = [&](int i) { return grads.as_strided({a.B, a.S, C}, {a.S * C, C, 1}, i * plane); };
    auto row = [&](int i) { return ln.as_strided({a.H, 32}, {32, 1}, i * C); };
    return wrap_all(part(0), part(1), part(2), row(0), row(1), row(2), row(3));
}

// attn_out [..., K1], x [..., D], fc weight [K1, D] and bias, W1 [D, F], b1, W2 [F, D], b2, activation
SPGT_NATIVE(encoder_tail, 9) {
    Call c(args);
    const at::Tensor *a = c.tensor(0), *x = c.tensor(1), *wfc = c.tensor(2), *w1 = c.tensor(4), *w2 = c.tensor(6);
    const int64_t act = c.integer(8);
    if (!c.ok || wfc->dim() != 2 || w1->dim() != 2 || w2->dim() != 2 || a->dim() < 1 || x->dim() < 1) Py_RETURN_NONE;
    const int64_t K1 = wfc->size(0), D = wfc->size(1), F = w1->size(1);
    const float *bfc = c.vector(3, D, false), *b1 = c.vector(5, F, false), *b2 = c.vector(7, D, false);
    c.require(K1 > 0 && D > 0 && w1->size(0) == D && w2->size(0) == F && w2->size(1) == D && a->size(-1) == K1 && x->size(-1) == D);
    if (!c.ok) Py_RETURN_NONE;
    const int64_t T = a->numel() / K1;
    if (T < 1 || x->numel() != T * D) Py_RETURN_NONE;
    const at::Tensor out = c.empty(x->sizes());
    if (launch(p_spgt_encoder_tail_forward, data(a), K1, data(x), data(wfc), bfc, data(w1), b1, data(w2), b2, (int)act,
               out.data_ptr<float>(), T, (int)K1, (int)D, (int)F, c.stream))
        Py_RETURN_NONE;
    return wrap(out);
}

// x [B, S, 128], position or None, a list of the sixteen parameters, eps, activation: None also where it does not pay
SPGT_NATIVE(encoder_layer, 5) {
    Call c(args);
    const at::Tensor* x = c.tensor(0);
    if (!c.ok || x->dim() != 3 || x->size(2) != 128 || x->size(0) < 1 || x->size(0) > 65535) Py_RETURN_NONE;
    const int64_t B = x->size(0), S = x->size(1);
    if (!p_spgt_encoder_layer_pays((int)B, S) || !PyList_CheckExact(args[2]) || PyList_GET_SIZE(args[2]) != 16) Py_RETURN_NONE;
    const float* pos = c.positions(1, B, S, 2, true);
    const int64_t dp = pos ? 2 : 0, F = 256, C = 128;
    const int64_t counts[16] = {C * C, C * C, C * C, C, C, C, C, C, C, C, C * 4 * (32 + dp), C, F * C, F, C * F, C};
    const float* p[16];
    PyObject* parameters[16];
    for (int i = 0; i < 16; ++i) parameters[i] = PyList_GET_ITEM(args[2], i);
    Call q(parameters);
    q.device = c.device, q.ok = c.ok;
    for (int i = 0; i < 16 && q.ok; ++i) p[i] = q.vector(i, counts[i], false);
    const double eps = c.real(3);
    const int64_t act = c.integer(4);
    if (!q.ok || !c.ok) Py_RETURN_NONE;
    const at::Tensor out = c.empty(x->sizes()), ws = c.workspace(p_spgt_encoder_layer_workspace_bytes((int)B, S, (int)dp));
    if (launch(p_spgt_encoder_layer_forward, data(x), pos, p[0], p[1], p[2], p[3], p[4], p[5], p[6], p[7], p[8], p[9], (float)eps,
               p[10], p[11], p[12], p[13], p[14], p[15], (int)act, out.data_ptr<float>(), (int)B, S, (int)dp, 128, 4, 256, nullptr,
               0.f, 0.f, ws.data_ptr(), (size_t)ws.numel(), c.stream))
        Py_RETURN_NONE;
    return wrap(out);
}

// src, padded table, r, 2m, inverse: planar forms only
SPGT_NATIVE(dft_rows_planar, 5) {
    Call c(args);
    const at::Tensor *src = c.tensor(0), *table = c.tensor(1);
    const int64_t r = c.integer(2), m2 = c.integer(3), inverse = c.integer(4);
    if (!c.ok || src->dim() != 4 || src->numel() == 0 || src->size(2) != r || src->size(1) != (inverse ? m2 : r)) Py_RETURN_NONE;
    const int64_t N = src->size(0), C = src->size(3);
    if (N * r > INT32_MAX || C > 65535) Py_RETURN_NONE;
    const at::Tensor out = c.empty({N, inverse ? r : m2, r, C});
    if (launch(inverse ? p_spgt_truncated_dft_rows_inverse : p_spgt_truncated_dft_rows_forward, data(src), data(table),
               out.data_ptr<float>(), N * r, (int)r, (int)C, (int)(m2 / 2), 1, c.stream))
        Py_RETURN_NONE;
    return wrap(out);
}

// Y [N, 2m, r, Cin], the two tables, the two weights [m, m, Cin, Cout, 2]
SPGT_NATIVE(modes_middle, 5) {
    Call c(args);
    const at::Tensor *y = c.tensor(0), *gh = c.tensor(1, at::kComplexFloat), *ghi = c.tensor(2, at::kComplexFloat);
    const at::Tensor *w1 = c.tensor(3), *w2 = c.tensor(4);
    if (!c.ok || y->dim() != 4 || y->numel() == 0 || w1->dim() != 5 || w1->sizes() != w2->sizes()) Py_RETURN_NONE;
    const int64_t N = y->size(0), m = y->size(1) / 2, r = y->size(2), cin = y->size(3), cout = w1->size(3);
    if (y->size(1) != 2 * m || w1->size(0) != m || w1->size(1) != m || w1->size(2) != cin || w1->size(4) != 2 || cout < 1 ||
        gh->dim() != 2 || gh->size(0) != 2 * m || gh->size(1) != r || ghi->dim() != 2 || ghi->size(0) != r ||
        ghi->size(1) != 2 * m || N > INT32_MAX || r > INT32_MAX)
        Py_RETURN_NONE;
    const at::Tensor out = c.empty({N, 2 * m, r, cout});
    const at::Tensor ws = c.workspace(p_spgt_spectral_modes_middle_workspace_bytes((int)N, (int)cout, (int)m));
    auto table = [](const at::Tensor* t) { return static_cast<const float*>(t->const_data_ptr()); };
    if (launch(p_spgt_spectral_modes_middle, data(y), table(gh), table(ghi), data(w1), data(w2), out.data_ptr<float>(),
               ws.data_ptr(), (size_t)ws.numel(), (int)N, (int)r, (int)cin, (int)cout, (int)m, c.stream))
        Py_RETURN_NONE;
    return wrap(out);
}

// U [N, 2m, r, Cout], table operand, X [N, r, r, Cin], weight [Cin, Cout], bias or None, activation
SPGT_NATIVE(inverse_linear, 6) {
    Call c(args);
    const at::Tensor *u = c.tensor(0), *table = c.tensor(1), *x = c.tensor(2), *w = c.tensor(3);
    const int64_t act = c.integer(5);
    if (!c.ok || u->dim() != 4 || x->dim() != 4 || w->dim() != 2 || x->numel() == 0) Py_RETURN_NONE;
    const int64_t N = x->size(0), r = x->size(1), cin = x->size(3), cout = w->size(1), m = u->size(1) / 2;
    const float* bias = c.vector(4, cout, true);
    c.require(x->size(2) == r && w->size(0) == cin && u->size(0) == N && u->size(1) == 2 * m && u->size(2) == r && u->size(3) == cout &&
              table->dim() == 3 && table->size(0) == (r + 31) / 32 && table->size(1) == (m <= 16 ? 16 : 32) && table->size(2) == 64);
    if (!c.ok) Py_RETURN_NONE;
    const at::Tensor out = c.empty({N, r, r, cout});
    if (launch(p_spgt_spectral_inverse_linear, data(u), data(table), data(x), data(w), bias, (int)act, out.data_ptr<float>(), N * r,
               (int)r, (int)cin, (int)cout, (int)m, c.stream))
        Py_RETURN_NONE;
    return wrap(out);
}

// X [N, C, H, W], weight, bias or None, activation, count, turned
SPGT_NATIVE(conv3x3, 6) {
    Call c(args);
    const at::Tensor *x = c.tensor(0), *w = c.tensor(1);
    const int64_t act = c.integer(3), count = c.integer(4), turned = c.integer(5);
    if (!c.ok || x->dim() != 4 || w->dim() != 4 || x->numel() == 0 || w->size(2) != 3 || w->size(3) != 3 ||
        w->size(turned ? 0 : 1) != x->size(1))
        Py_RETURN_NONE;
    const int64_t cout = w->size(turned ? 1 : 0);
    const float* bias = c.vector(2, cout, true);
    for (int d = 0; d < 4; ++d) c.require(x->size(d) <= INT32_MAX);
    if (!c.ok || cout > INT32_MAX) Py_RETURN_NONE;
    const size_t bytes = p_spgt_conv3x3_workspace_bytes((int)x->size(1), (int)cout);
    if (bytes == 0) Py_RETURN_NONE;
    const at::Tensor out = c.empty({x->size(0), cout, x->size(2), x->size(3)}), ws = c.workspace(bytes);
    if (launch(p_spgt_conv3x3_forward, data(x), data(w), bias, out.data_ptr<float>(), (int)x->size(0), (int)x->size(1), (int)cout,
               (int)x->size(2), (int)x->size(3), (int)turned, (int)act, (int)count, ws.data_ptr(), (size_t)ws.numel(),
               c.stream))
        Py_RETURN_NONE;
    return wrap(out);
}

// input [B, S, C], weight [C, C], bias [C], LayerNorm weight and bias or None twice, eps, position, num_head, dim_position:
// heads [B, H, dp + C / H, S], and with LayerNorm (heads, 1 / sigma [B, H, S])
SPGT_NATIVE(projection, 9) {
    Call c(args);
    const at::Tensor *x = c.tensor(0), *w = c.tensor(1);
    const double eps = c.real(5);
    const int64_t H = c.integer(7), dp = c.integer(8);
    if (!c.ok || x->dim() != 3 || x->numel() == 0 || w->dim() != 2 || H < 1 || dp < 0 || dp > 64) Py_RETURN_NONE;
    const int64_t B = x->size(0), S = x->size(1), C = x->size(2);
    const float *b = c.vector(2, C, false), *g = c.vector(3, C, true), *s = c.vector(4, C, true);
    c.require(w->size(0) == C && w->size(1) == C && C % H == 0 && !g == !s && B <= INT32_MAX && S <= INT32_MAX && C <= 65535);
    const float* pos = dp ? c.positions(6, B, S, dp, false) : nullptr;
    if (!c.ok) Py_RETURN_NONE;
    const int64_t d = C / H;
    const at::Tensor out = c.empty({B, H, dp + d, S});
    if (!g) {
        if (launch(p_spgt_multihead_projection_with_position_rrc_forward, data(x), data(w), b, pos, out.data_ptr<float>(), (int)S,
                   (int)C, (int)H, (int)d, (int)dp, (int)B, c.stream))
            Py_RETURN_NONE;
        return wrap(out);
    }
    const at::Tensor inv = c.empty({B, H, S});
    if (launch(p_spgt_multihead_projection_layernorm_with_position_rrc_forward, data(x), data(w), b, g, s, (float)eps, pos,
               out.data_ptr<float>(), inv.data_ptr<float>(), (int)S, (int)C, (int)H, (int)d, (int)dp, (int)B, c.stream))
        Py_RETURN_NONE;
    return wrap_all(out, inv);
}

// Q, K, V [B, H, d, S]: [B, H, S, d]
SPGT_NATIVE(cccr_forward, 3) {
    Call c(args);
    const at::Tensor *q = c.tensor(0), *k = c.tensor(1), *v = c.tensor(2);
    if (!c.ok || q->dim() != 4 || q->numel() == 0 || q->sizes() != k->sizes() || q->sizes() != v->sizes()) Py_RETURN_NONE;
    const int64_t B = q->size(0), H = q->size(1), d = q->size(2), S = q->size(3);
    if (B > INT32_MAX || H > INT32_MAX || d > INT32_MAX || S > INT32_MAX) Py_RETURN_NONE;
    const size_t bytes = p_spgt_galerkin_attention_cccr_workspace_bytes((int)B, (int)H, (int)d, (int)S);
    if (bytes == 0) Py_RETURN_NONE;
    const at::Tensor out = c.empty({B, H, S, d}), ws = c.workspace(bytes);
    if (launch(p_spgt_galerkin_attention_cccr_forward, data(q), data(k), data(v), out.data_ptr<float>(), ws.data_ptr(),
               (size_t)ws.numel(), (int)B, (int)H, (int)d, (int)S, c.stream))
        Py_RETURN_NONE;
    return wrap(out);
}

// grad [B, H, S, d], Q, K, V: (dQ, dK, dV)
SPGT_NATIVE(cccr_backward, 4) {
    Call c(args);
    const at::Tensor *g = c.tensor(0), *q = c.tensor(1), *k = c.tensor(2), *v = c.tensor(3);
    if (!c.ok || q->dim() != 4 || q->numel() == 0 || q->sizes() != k->sizes() || q->sizes() != v->sizes()) Py_RETURN_NONE;
    const int64_t B = q->size(0), H = q->size(1), d = q->size(2), S = q->size(3);
    if (g->dim() != 4 || g->size(0) != B || g->size(1) != H || g->size(2) != S || g->size(3) != d || B > INT32_MAX ||
        H > INT32_MAX || d > INT32_MAX || S > INT32_MAX)
        Py_RETURN_NONE;
    const size_t bytes = p_spgt_galerkin_attention_cccr_backward_workspace_bytes((int)B, (int)H, (int)d, (int)S);
    if (bytes == 0) Py_RETURN_NONE;
    const at::Tensor dq = c.empty(q->sizes()), dk = c.empty(q->sizes()), dv = c.empty(q->sizes()), ws = c.workspace(bytes);
    if (launch(p_spgt_galerkin_attention_cccr_backward, data(g), data(q), data(k), data(v), dq.data_ptr<float>(),
               dk.data_ptr<float>(), dv.data_ptr<float>(), ws.data_ptr(), (size_t)ws.numel(), (int)B, (int)H, (int)d, (int)S,
               c.stream))
        Py_RETURN_NONE;
    return wrap_all(dq, dk, dv);
}

// src [B, H, dp + d, S], dp: [B, S, H d]
SPGT_NATIVE(heads_to_tokens, 2) {
    Call c(args);
    const at::Tensor* src = c.tensor(0);
    const int64_t dp = c.integer(1);
    if (!c.ok || src->dim() != 4 || src->numel() == 0 || dp < 0 || src->size(2) <= dp) Py_RETURN_NONE;
    const int64_t B = src->size(0), H = src->size(1), d = src->size(2) - dp, S = src->size(3);
    if (B > INT32_MAX || H > INT32_MAX || d > INT32_MAX || S > INT32_MAX) Py_RETURN_NONE;
    const at::Tensor out = c.empty({B, S, H * d});
    if (launch(p_spgt_heads_feature_to_token_major, data(src), out.data_ptr<float>(), (int)B, (int)H, (int)dp, (int)d, (int)S,
               c.stream))
        Py_RETURN_NONE;
    return wrap(out);
}

// pre [T, C], grad of T C values, LayerNorm weight, eps, num_head, dim_head: (d pre, d weight, d bias)
SPGT_NATIVE(layernorm_heads_backward, 6) {
    Call c(args);
    const at::Tensor *pre = c.tensor(0), *g = c.tensor(1);
    const double eps = c.real(3);
    const int64_t H = c.integer(4), d = c.integer(5);
    if (!c.ok || pre->dim() != 2 || pre->numel() == 0 || g->numel() != pre->numel() || H < 1 || pre->size(1) != H * d || H > INT32_MAX)
        Py_RETURN_NONE;
    const float* gamma = c.vector(2, H * d, false);
    if (!c.ok) Py_RETURN_NONE;
    const int64_t T = pre->size(0);
    const at::Tensor out = c.empty(pre->sizes()), dg = c.empty({H, d}), db = c.empty({H, d});
    const at::Tensor ws = c.workspace(p_spgt_layernorm_heads_backward_workspace_bytes(T, (int)H));
    if (launch(p_spgt_layernorm_heads_backward, data(pre), data(g), gamma, (float)eps, out.data_ptr<float>(), dg.data_ptr<float>(),
               db.data_ptr<float>(), ws.data_ptr(), (size_t)ws.numel(), T, (int)H, c.stream))
        Py_RETURN_NONE;
    return wrap_all(out, dg, db);
}

// bind(library, {function name: address}): the library whose functions are called from now on
PyObject* bind(PyObject*, PyObject* args) {
    PyObject *lib, *table;
    if (!PyArg_ParseTuple(args, "OO!", &lib, &PyDict_Type, &table)) return nullptr;
#define SPGT_LOOK_UP(name)                                                       \
    {                                                                            \
        PyObject* a = PyDict_GetItemString(table, #name);                        \
        if (!a) return PyErr_Format(PyExc_KeyError, "no address of %s", #name);  \
        p_##name = reinterpret_cast<decltype(&::name)>(PyLong_AsVoidPtr(a));     \
        if (PyErr_Occurred()) return nullptr;                                    \
    }
    SPGT_FUNCTIONS(SPGT_LOOK_UP)
#undef SPGT_LOOK_UP
    g_lib = lib;
    Py_RETURN_NONE;
}

#define SPGT_METHOD(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(name)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {SPGT_METHOD(linear),
                         SPGT_METHOD(input_grad),
                         SPGT_METHOD(projection_input_grad),
                         SPGT_METHOD(packed_input_grad),
                         SPGT_METHOD(weight_grad),
                         SPGT_METHOD(weight_grad_batched),
                         SPGT_METHOD(attention_forward),
                         SPGT_METHOD(attention_backward),
                         SPGT_METHOD(encoder_tail),
                         SPGT_METHOD(encoder_layer),
                         SPGT_METHOD(dft_rows_planar),
                         SPGT_METHOD(modes_middle),
                         SPGT_METHOD(inverse_linear),
                         SPGT_METHOD(conv3x3),
                         SPGT_METHOD(projection),
                         SPGT_METHOD(cccr_forward),
                         SPGT_METHOD(cccr_backward),
                         SPGT_METHOD(heads_to_tokens),
                         SPGT_METHOD(layernorm_heads_backward),
                         {"bind", bind, METH_VARARGS, nullptr},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_native_calls", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__native_calls() { return PyModule_Create(&module); }
