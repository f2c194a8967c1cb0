// Host path of the autograd modules and of the decode ops: argument checks, allocations, autograd node and the
// calls of the C ABI (include/convattn.h) in one native function per op.
//
// A training step of a short sequence runs for 50 us on the GPU; the same host work in Python (ctypes calls, one torch
// call per allocation, an autograd Function) took 107 us.  Every function here takes the ordinary case only
// (plain device tensors the kernels take as they are, a workspace under the cap, nothing beside autograd's backward that
// has to see the call) and returns None for anything else: the Python ops then run, convert, fall back or raise.
#include <torch/extension.h>

#include <ATen/hip/EmptyTensor.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <dlfcn.h>
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/saved_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>

#include <cstdlib>

#include "convattn.h"

namespace {

using at::Tensor;
using torch::autograd::SavedVariable;
using torch::autograd::variable_list;

// ---- the C ABI, from the library Python has loaded ----
#define API_LIST(F)                                                                                                   \
    F(convattn_strerror) F(convattn_kernel_path) F(convattn_fwd) F(convattn_fwd_split_workspace_bytes) F(convattn_fwd_split) F(convattn_bwd_preprocess) F(convattn_bwd_fused_workspace_bytes)              \
    F(convattn_bwd_fused) F(convattn_bwd_split_workspace_bytes) F(convattn_bwd_all) F(convattn_staged_workspace_bytes) F(convattn_staged_fwd) F(convattn_staged_bwd)               \
    F(convattn_decode_strided) F(convattn_decode_splits) F(convattn_decode_step_splits) F(convattn_decode_whole_ok) F(convattn_decode_whole) F(convattn_decode_kv) F(convattn_decode_combine)                 \
    F(convattn_headmix_validate) F(convattn_headmix_fwd_workspace_bytes) F(convattn_headmix_fwd_ws)                   \
    F(convattn_headmix_bwd_fused_workspace_bytes) F(convattn_headmix_bwd_fused_dq_dw_workspace_bytes) F(convattn_headmix_bwd_fused)
struct Api {
#define F(name) decltype(&::name) name = nullptr;
    API_LIST(F)
#undef F
};
Api api;

void init(const std::string &path) {
    void *lib = dlopen(path.c_str(), RTLD_NOW | RTLD_LOCAL);
    TORCH_CHECK(lib, "cannot load ", path, ": ", dlerror());
#define F(name)                                                                            \
    api.name = reinterpret_cast<decltype(api.name)>(dlsym(lib, #name));                    \
    TORCH_CHECK(api.name, path, " has no ", #name);
    API_LIST(F)
#undef F
}

void check(int rc, const char *what) {
    if (rc == 0) return;
    std::string msg = std::string(what) + ": " + api.convattn_strerror(rc);
    if (rc > 0) msg += " (hipError_t " + std::to_string(rc) + ")";
    throw std::runtime_error(msg);
}

void *stream_of(const Tensor &t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

Tensor empty(at::IntArrayRef size, at::ScalarType dt, const Tensor &like) {
    return Tensor(at::detail::empty_cuda(size, dt, like.device(), std::nullopt));
}

// Largest workspace allocated in one piece (CONVATTN_MAX_WORKSPACE_BYTES, 16 GiB)
size_t workspace_cap() {
    const char *e = std::getenv("CONVATTN_MAX_WORKSPACE_BYTES");
    return e ? std::strtoull(e, nullptr, 10) : size_t(16) << 30;
}
// Undefined above the cap or when it cannot be allocated
Tensor workspace(size_t bytes, const Tensor &like) {
    if (bytes == 0 || bytes > workspace_cap()) return Tensor();
    try {
        return empty({(int64_t)bytes}, at::kByte, like);
    } catch (const c10::OutOfMemoryError &) {
        return Tensor();
    }
}

// A device tensor that is nothing but memory: no subclass, no functorch wrapper, no lazy conjugate
bool plain(const Tensor &t) {
    return t.defined() && t.is_cuda() && t.layout() == at::kStrided && !t.is_conj() && !t.is_neg() &&
           !t.key_set().has_any(c10::DispatchKeySet({c10::DispatchKey::Python, c10::DispatchKey::FuncTorchBatched,
                                                     c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::Functionalize}));
}
// The call has to go through torch's own machinery: it is being traced (a native call leaves its result in the trace as a
// constant), or a dispatch mode or a functorch transform (vmap, grad, jvp, functionalize) is active in this thread.
bool watched() {
    return torch::jit::tracer::isTracing() || c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::Python) ||
           c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode);
}
// Forward-mode derivatives: the autograd Functions have none and say so; a native call would drop the tangent
bool has_tangent(const Tensor &t) { return t._fw_grad(/*level=*/0).defined(); }
template <typename... T> bool has_tangents(const T &...t) { return (has_tangent(t) || ...); }
int dt_of(const Tensor &t) { return t.scalar_type() == at::kBFloat16 ? CONVATTN_BF16 : CONVATTN_F32; }
int64_t padded(int64_t n) { return (n + 3) & ~int64_t(3); }   // floats up to the next 16-byte boundary
bool aligned(const Tensor &t) { return (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15) == 0; }

bool same_rows(const Tensor &Q, const Tensor &K, const Tensor &V) {
    const auto st = Q.scalar_type();
    if (!plain(Q) || !plain(K) || !plain(V) || Q.dim() != 4 || K.dim() != 4 || V.dim() != 4) return false;
    if ((st != at::kBFloat16 && st != at::kFloat) || K.scalar_type() != st || V.scalar_type() != st) return false;
    return K.sizes() == V.sizes() && Q.size(0) == K.size(0) && Q.size(3) == K.size(3) && Q.device() == K.device() &&
           Q.device() == V.device();
}

// What the kernels were written to read in the place of a saved tensor: saved-tensor hooks may give back anything
bool as_saved(const Tensor &t, at::IntArrayRef size, at::ScalarType dt, at::Device dev) {
    return plain(t) && t.sizes() == size && t.scalar_type() == dt && t.is_contiguous() && t.device() == dev;
}

// Window weights as the kernels take them, or undefined: [H, c_q, odd c_k] with the pads that belong to them
Tensor window(const Tensor &W, int64_t H, int64_t pad_q, int64_t pad_k, const Tensor &Q) {
    if (!plain(W) || W.dim() != 3 || W.size(0) != H || W.size(2) % 2 == 0 || pad_q != W.size(1) - 1 ||
        pad_k != (W.size(2) - 1) / 2 || W.device() != Q.device() || !at::isFloatingType(W.scalar_type()))
        return Tensor();
    at::AutoDispatchBelowADInplaceOrView guard;
    Tensor w = W.scalar_type() == at::kFloat && W.is_contiguous() ? W : W.to(at::kFloat).contiguous();
    return aligned(w) ? w : w.clone();
}

convattn_desc window_desc(const Tensor &Q, int64_t Nk, const Tensor &W, double scale, bool causal, int out_dt) {
    convattn_desc d{};
    d.B = (int)Q.size(0); d.H = (int)Q.size(1); d.Nq = (int)Q.size(2); d.Nk = (int)Nk; d.d = (int)Q.size(3);
    d.c_q = (int)W.size(1); d.c_k = (int)W.size(2);
    d.scale = (float)scale; d.causal = causal; d.in_dtype = dt_of(Q); d.out_dtype = out_dt; d.n_splits = 1;
    return d;
}

// Python's backward for what the one-pass kernel does not take here (partial gradients, workspace cap)
py::object *window_slow_backward = nullptr, *mix_slow_backward = nullptr;

// ------------------------------------------------------------------ window attention
struct WindowBackward : torch::autograd::Node {
    SavedVariable q, k, v, w, o, ml;   // ml: M then (from the next 16-byte boundary) L, fp32 [B][H][Nq]
    double scale = 1;
    int64_t pad_q = 0, pad_k = 0;
    bool causal = false;

    std::string name() const override { return "FlashConvAttentionCUDAFunctionBackward"; }
    void release_variables() override {
        std::lock_guard<std::mutex> lock(mutex_);
        q.reset_data(); k.reset_data(); v.reset_data(); w.reset_data(); o.reset_data(); ml.reset_data();
    }
    variable_list apply(variable_list &&grads) override {
        std::lock_guard<std::mutex> lock(mutex_);
        variable_list out(4);
        if (!grads[0].defined()) return out;
        const Tensor Q = q.unpack(), K = k.unpack(), V = v.unpack(), W = w.unpack(), O = o.unpack(shared_from_this()), stats = ml.unpack();
        at::AutoDispatchBelowADInplaceOrView guard;
        c10::DeviceGuard dev(Q.device());
        Tensor dO = grads[0];
        if (dO.scalar_type() != Q.scalar_type()) dO = dO.to(Q.scalar_type());
        dO = dO.contiguous();
        const bool all = (task_should_compute_output(0) || task_should_compute_output(3)) &&
                         (task_should_compute_output(1) || task_should_compute_output(2));
        const bool sound = plain(dO) && same_rows(Q, K, V) && K.size(1) == Q.size(1) && Q.is_contiguous() && K.is_contiguous() &&
                           V.is_contiguous() && as_saved(O, Q.sizes(), Q.scalar_type(), Q.device()) &&
                           as_saved(dO, Q.sizes(), Q.scalar_type(), Q.device()) &&
                           as_saved(stats, {2 * padded(Q.size(0) * Q.size(1) * Q.size(2))}, at::kFloat, Q.device());
        const Tensor Wf = all && sound && !watched() ? window(W, Q.size(1), pad_q, pad_k, Q) : Tensor();
        if (Wf.defined()) {
            convattn_desc d = window_desc(Q, K.size(2), Wf, scale, causal, dt_of(Q));
            const size_t rows = (size_t)Q.size(0) * Q.size(1) * Q.size(2), stat = (rows * 4 + 255) / 256 * 256;
            // (D and LSE ahead of the workspace, which counts for the cap alone as in the Python op)
            auto reserve = [&](size_t bytes) { return bytes && bytes <= workspace_cap() ? workspace(bytes + 2 * stat, Q) : Tensor(); };
            Tensor ws = reserve(api.convattn_staged_workspace_bytes(&d, CONVATTN_OP_BWD));
            const bool staged = ws.defined();
            int split = 0;
            if (!staged && api.convattn_kernel_path(&d, CONVATTN_OP_BWD) == 1) {   // (1: the bf16 kernels, which the next two are)
                ws = reserve(api.convattn_bwd_split_workspace_bytes(&d));
                split = ws.defined();
                if (!split) ws = reserve(api.convattn_bwd_fused_workspace_bytes(&d));
            }
            if (ws.defined()) {
                char *base = static_cast<char *>(ws.data_ptr());
                float *D = reinterpret_cast<float *>(base), *lse = reinterpret_cast<float *>(base + stat);
                const float *M = stats.const_data_ptr<float>(), *L = M + padded(rows);
                void *s = stream_of(Q);
                Tensor dQ = empty(Q.sizes(), Q.scalar_type(), Q), dK = empty(K.sizes(), Q.scalar_type(), Q),
                       dV = empty(V.sizes(), Q.scalar_type(), Q), dW = empty(W.sizes(), at::kFloat, Q);
                const float *w = Wf.const_data_ptr<float>();
                if (staged) {
                    convattn_desc pre = d;
                    pre.Nk = pre.Nq; pre.c_q = pre.c_k = 1; pre.scale = 1; pre.causal = 0;
                    check(api.convattn_bwd_preprocess(&pre, O.data_ptr(), dO.data_ptr(), M, L, D, lse, s), "conv_attn.bwd_preprocess");
                    check(api.convattn_staged_bwd(&d, Q.data_ptr(), K.data_ptr(), V.data_ptr(), dO.data_ptr(), D, lse, w, dQ.data_ptr(),
                                                  dK.data_ptr(), dV.data_ptr(), dW.mutable_data_ptr<float>(), base + 2 * stat, s),
                          "conv_attn.backward");
                } else {
                    check(api.convattn_bwd_all(&d, Q.data_ptr(), K.data_ptr(), V.data_ptr(), O.data_ptr(), dO.data_ptr(), M, L, w, D, lse,
                                               dQ.data_ptr(), dK.data_ptr(), dV.data_ptr(), dW.mutable_data_ptr<float>(), split,
                                               base + 2 * stat, s),
                          "conv_attn.backward");
                }
                out[0] = dQ; out[1] = dK; out[2] = dV;
                out[3] = W.scalar_type() == at::kFloat ? dW : dW.to(W.scalar_type());
                return out;
            }
        }
        TORCH_CHECK(Q.dim() == 4, "conv_attn.backward: Q must be [batch, heads, seq_len, d_head]");
        const int64_t rows = Q.size(0) * Q.size(1) * Q.size(2);
        const Tensor M = stats.narrow(0, 0, rows).view({Q.size(0), Q.size(1), Q.size(2)}),
                     L = stats.narrow(0, padded(rows), rows).view({Q.size(0), Q.size(1), Q.size(2)});
        py::gil_scoped_acquire gil;
        auto r = (*window_slow_backward)(Q, K, V, W.detach(), M, L, O.detach(), dO, scale, pad_q, pad_k, causal,
                                         (bool)task_should_compute_output(0), (bool)task_should_compute_output(1),
                                         (bool)task_should_compute_output(2), (bool)task_should_compute_output(3))
                     .cast<std::vector<std::optional<Tensor>>>();
        for (int i = 0; i < 4; ++i)
            if (r[i]) out[i] = *r[i];
        return out;
    }
};

// O = window attention of Q, K, V (with its autograd node where a gradient is wanted), or nothing when the Python path has
// to take the call
std::optional<Tensor> window_attention(const Tensor &Q, const Tensor &K, const Tensor &V, const Tensor &W, double scale,
                                       int64_t pad_q, int64_t pad_k, bool causal) {
    if (watched() || !same_rows(Q, K, V) || K.size(1) != Q.size(1)) return std::nullopt;
    if (has_tangents(Q, K, V, W)) return std::nullopt;
    const Tensor Wf = window(W, Q.size(1), pad_q, pad_k, Q);
    if (!Wf.defined()) return std::nullopt;
    py::gil_scoped_release no_gil;
    c10::DeviceGuard dev(Q.device());
    std::shared_ptr<WindowBackward> node;
    if (torch::autograd::compute_requires_grad(Q, K, V, W)) {
        node = std::shared_ptr<WindowBackward>(new WindowBackward(), torch::autograd::deleteNode);
        node->set_next_edges(torch::autograd::collect_next_edges(Q, K, V, W));
    }
    Tensor Qc = Q, Kc = K, Vc = V, O, stats;
    const int64_t rows = Q.size(0) * Q.size(1) * Q.size(2);
    {
        at::AutoDispatchBelowADInplaceOrView guard;
        if (!Q.is_contiguous()) Qc = Q.contiguous();
        if (!K.is_contiguous()) Kc = K.contiguous();
        if (!V.is_contiguous()) Vc = V.contiguous();
        convattn_desc d = window_desc(Qc, K.size(2), Wf, scale, causal, dt_of(Q));
        const size_t staged = api.convattn_staged_workspace_bytes(&d, CONVATTN_OP_FWD);
        Tensor ws = workspace(staged, Q);
        if (staged && !ws.defined()) return std::nullopt;   // (by groups of heads, or the kernels without that scratch)
        O = empty(Q.sizes(), Q.scalar_type(), Q);
        stats = empty({2 * padded(rows)}, at::kFloat, Q);
        float *M = stats.mutable_data_ptr<float>();
        auto forward = api.convattn_staged_fwd;
        if (!staged) {
            ws = workspace(api.convattn_fwd_split_workspace_bytes(&d), Q);
            forward = api.convattn_fwd_split;
        }
        const float *w = Wf.const_data_ptr<float>();
        check(ws.defined() ? forward(&d, Qc.data_ptr(), Kc.data_ptr(), Vc.data_ptr(), w, ws.data_ptr(), O.data_ptr(), M, M + padded(rows),
                                     stream_of(Q))
                           : api.convattn_fwd(&d, Qc.data_ptr(), Kc.data_ptr(), Vc.data_ptr(), w, O.data_ptr(), M, M + padded(rows), stream_of(Q)),
              "conv_attn.forward");
    }
    if (node) {
        node->scale = scale; node->pad_q = pad_q; node->pad_k = pad_k; node->causal = causal;
        node->q = SavedVariable(Qc, false); node->k = SavedVariable(Kc, false); node->v = SavedVariable(Vc, false);
        node->w = SavedVariable(W, false);
        node->ml = SavedVariable(stats, false);
        torch::autograd::set_history(O, node);
        node->o = SavedVariable(O, true);
    }
    return O;
}

// ------------------------------------------------------------------ head-mixing attention
convattn_headmix_desc mix_desc(const Tensor &Q, double scale, bool causal) {
    return convattn_headmix_desc{(int)Q.size(0), (int)Q.size(1), (int)Q.size(2), (int)Q.size(3), (float)scale, causal,
                                 CONVATTN_BF16, CONVATTN_BF16};
}

struct MixBackward : torch::autograd::Node {
    SavedVariable q, k, v, w, o, lm;   // lm: L then M, fp32 [B][H][N]
    double scale = 1;
    bool causal = false;

    std::string name() const override { return "HeadConvAttentionFunctionBackward"; }
    void release_variables() override {
        std::lock_guard<std::mutex> lock(mutex_);
        q.reset_data(); k.reset_data(); v.reset_data(); w.reset_data(); o.reset_data(); lm.reset_data();
    }
    variable_list apply(variable_list &&grads) override {
        std::lock_guard<std::mutex> lock(mutex_);
        variable_list out(4);
        if (!grads[0].defined()) return out;
        const Tensor Q = q.unpack(), K = k.unpack(), V = v.unpack(), W = w.unpack(), O = o.unpack(shared_from_this()), stats = lm.unpack();
        at::AutoDispatchBelowADInplaceOrView guard;
        c10::DeviceGuard dev(Q.device());
        Tensor dO = grads[0];
        if (dO.scalar_type() != at::kBFloat16) dO = dO.to(at::kBFloat16);
        dO = dO.contiguous();
        TORCH_CHECK(Q.dim() == 4, "head_conv_attention_bwd: q must be [batch, heads, seq_len, d_model]");
        const int64_t rows = Q.size(0) * Q.size(1) * Q.size(2);
        const auto bf16 = at::kBFloat16;
        const bool sound = as_saved(Q, Q.sizes(), bf16, Q.device()) && as_saved(K, Q.sizes(), bf16, Q.device()) &&
                           as_saved(V, Q.sizes(), bf16, Q.device()) && as_saved(O, Q.sizes(), bf16, Q.device()) &&
                           as_saved(dO, Q.sizes(), bf16, Q.device()) && as_saved(stats, {2 * rows}, at::kFloat, Q.device()) &&
                           plain(W) && W.dim() == 2 && W.size(0) == Q.size(1) && W.size(1) == Q.size(1) && W.device() == Q.device() &&
                           at::isFloatingType(W.scalar_type());
        const bool want_q = task_should_compute_output(0) || task_should_compute_output(3),
                   want_kv = task_should_compute_output(1) || task_should_compute_output(2);
        convattn_headmix_desc d = mix_desc(Q, scale, causal);
        Tensor ws = sound && !watched() ? workspace((want_kv ? api.convattn_headmix_bwd_fused_workspace_bytes
                                                         : api.convattn_headmix_bwd_fused_dq_dw_workspace_bytes)(&d), Q) : Tensor();
        if (ws.defined()) {
            const Tensor Wf = W.scalar_type() == at::kFloat && W.is_contiguous() ? W : W.to(at::kFloat).contiguous();
            if (want_q) { out[0] = empty(Q.sizes(), at::kBFloat16, Q); out[3] = empty(W.sizes(), at::kFloat, Q); }
            if (want_kv) { out[1] = empty(Q.sizes(), at::kBFloat16, Q); out[2] = empty(Q.sizes(), at::kBFloat16, Q); }
            const float *L = stats.const_data_ptr<float>();
            auto ptr = [](const Tensor &t) { return t.defined() ? t.data_ptr() : nullptr; };
            check(api.convattn_headmix_bwd_fused(&d, CONVATTN_BF16, Q.data_ptr(), K.data_ptr(), V.data_ptr(),
                                                 Wf.const_data_ptr<float>(), O.data_ptr(), dO.data_ptr(), L, L + rows, ws.data_ptr(),
                                                 ptr(out[0]), ptr(out[1]), ptr(out[2]), static_cast<float *>(ptr(out[3])), stream_of(Q)),
                  "head_conv_attention_bwd");
            if (want_q && W.scalar_type() != at::kFloat) out[3] = out[3].to(W.scalar_type());
            return out;
        }
        const Tensor L = stats.narrow(0, 0, rows).view({Q.size(0), Q.size(1), Q.size(2)}),
                     M = stats.narrow(0, rows, rows).view({Q.size(0), Q.size(1), Q.size(2)});
        py::gil_scoped_acquire gil;
        auto r = (*mix_slow_backward)(Q, K, V, W.detach(), O.detach(), dO, L, M, causal, scale, want_q, want_kv)
                     .cast<std::vector<std::optional<Tensor>>>();
        for (int i = 0; i < 4; ++i)
            if (r[i]) out[i] = *r[i];
        return out;
    }
};

std::optional<Tensor> mix_attention(const Tensor &Q, const Tensor &K, const Tensor &V, const Tensor &W, bool causal, double scale) {
    if (watched() || !same_rows(Q, K, V) || Q.scalar_type() != at::kBFloat16 || Q.sizes() != K.sizes()) return std::nullopt;
    if (has_tangents(Q, K, V, W)) return std::nullopt;
    if (!plain(W) || W.dim() != 2 || W.size(0) != Q.size(1) || W.size(1) != Q.size(1) || W.device() != Q.device() ||
        !at::isFloatingType(W.scalar_type()))
        return std::nullopt;
    convattn_headmix_desc d = mix_desc(Q, scale, causal);
    if (api.convattn_headmix_validate(&d)) return std::nullopt;
    py::gil_scoped_release no_gil;
    c10::DeviceGuard dev(Q.device());
    std::shared_ptr<MixBackward> node;
    if (torch::autograd::compute_requires_grad(Q, K, V, W)) {
        node = std::shared_ptr<MixBackward>(new MixBackward(), torch::autograd::deleteNode);
        node->set_next_edges(torch::autograd::collect_next_edges(Q, K, V, W));
    }
    Tensor Qc = Q, Kc = K, Vc = V, O, stats;
    const int64_t rows = Q.size(0) * Q.size(1) * Q.size(2);
    {
        at::AutoDispatchBelowADInplaceOrView guard;
        Tensor ws = workspace(api.convattn_headmix_fwd_workspace_bytes(&d), Q);
        if (!ws.defined()) return std::nullopt;
        if (!Q.is_contiguous()) Qc = Q.contiguous();
        if (!K.is_contiguous()) Kc = K.contiguous();
        if (!V.is_contiguous()) Vc = V.contiguous();
        const Tensor Wf = W.scalar_type() == at::kFloat && W.is_contiguous() ? W : W.to(at::kFloat).contiguous();
        O = empty(Q.sizes(), at::kBFloat16, Q);
        stats = empty({2 * rows}, at::kFloat, Q);
        float *L = stats.mutable_data_ptr<float>();
        check(api.convattn_headmix_fwd_ws(&d, Qc.data_ptr(), Kc.data_ptr(), Vc.data_ptr(), Wf.const_data_ptr<float>(), ws.data_ptr(),
                                          O.data_ptr(), L, L + rows, stream_of(Q)),
              "head_conv_attention_forward");
    }
    if (node) {
        node->scale = scale; node->causal = causal;
        node->q = SavedVariable(Qc, false); node->k = SavedVariable(Kc, false); node->v = SavedVariable(Vc, false);
        node->w = SavedVariable(W, false);
        node->lm = SavedVariable(stats, false);
        torch::autograd::set_history(O, node);
        node->o = SavedVariable(O, true);
    }
    return O;
}

// ------------------------------------------------------------------ decode
// [B,H,N,d] as it lies, or a view of a longer cache: rows of a head dense, heads and batches strided
bool cache_rows(const Tensor &t) {
    if (t.is_contiguous()) return true;
    const auto N = t.size(2), d = t.size(3);
    return t.stride(3) == 1 && t.stride(2) == d && t.stride(1) >= N * d && t.stride(1) % 8 == 0 && t.stride(0) % 8 == 0 &&
           (t.size(0) == 1 || t.stride(0) >= N * d);
}
int64_t head_stride(const Tensor &t) { return t.is_contiguous() ? t.size(2) * t.size(3) : t.stride(1); }
int64_t batch_stride(const Tensor &t) { return t.is_contiguous() ? t.size(1) * t.size(2) * t.size(3) : t.stride(0); }

using Decoded = std::tuple<Tensor, Tensor, Tensor, Tensor, Tensor, Tensor>;   // O, M, L and the partials

template <typename Launch>
Decoded run_decode(const convattn_desc &d, const Tensor &Q, at::ScalarType out, const char *what, const Launch &launch) {
    py::gil_scoped_release no_gil;
    c10::DeviceGuard dev(Q.device());
    at::AutoDispatchBelowADInplaceOrView guard;
    const int64_t B = d.B, H = d.H, n = d.n_splits, D = d.d;
    Tensor Op = empty({B, H, n, D}, at::kFloat, Q), Mp = empty({B, H, n}, at::kFloat, Q), Lp = empty({B, H, n}, at::kFloat, Q);
    Tensor O = empty({B, H, 1, D}, out, Q), M = empty({B, H, 1}, at::kFloat, Q), L = empty({B, H, 1}, at::kFloat, Q);
    float *op = Op.mutable_data_ptr<float>(), *mp = Mp.mutable_data_ptr<float>(), *lp = Lp.mutable_data_ptr<float>();
    void *s = stream_of(Q);
    check(launch(op, mp, lp, s), what);
    check(api.convattn_decode_combine(&d, op, mp, lp, O.data_ptr(), M.mutable_data_ptr<float>(), L.mutable_data_ptr<float>(), s), what);
    return {O, M, L, Op, Mp, Lp};
}

std::optional<at::ScalarType> out_type(const py::object &dtype) {
    const auto t = dtype.cast<at::ScalarType>();
    if (t != at::kBFloat16 && t != at::kFloat) return std::nullopt;
    return t;
}

// k_splits > 0, or 0: the library's choice.  Without `partials` k_splits is a most, and they may be missing from the result.
std::optional<Decoded> decode_dense(const Tensor &Q, const Tensor &K, const Tensor &V, const Tensor &W, int64_t k_splits, double scale,
                                    bool causal, const py::object &out_dtype, bool partials) {
    const auto out = out_type(out_dtype);
    if (!out || watched() || !same_rows(Q, K, V) || K.size(1) != Q.size(1) || !Q.is_contiguous() || !cache_rows(K) || K.strides() != V.strides() ||
        Q.size(2) > 16 || k_splits < 0 || k_splits > 1024 || k_splits > K.size(2) || W.dim() != 3)
        return std::nullopt;
    const Tensor Wf = window(W, Q.size(1), W.size(1) - 1, (W.size(2) - 1) / 2, Q);
    if (!Wf.defined()) return std::nullopt;
    convattn_desc d = window_desc(Q, K.size(2), Wf, scale, causal, *out == at::kFloat ? CONVATTN_F32 : CONVATTN_BF16);
    d.n_splits = k_splits > 0 ? (int)k_splits : 1;
    if (!partials && api.convattn_kernel_path(&d, CONVATTN_OP_DECODE) == 1) {
        d.n_splits = api.convattn_decode_step_splits(d.B, d.H, d.Nk, d.d, (int)k_splits);
        const bool whole = api.convattn_decode_whole_ok(&d) != 0;
        const char *what = "conv_attn.forward_inference";
        py::gil_scoped_release no_gil;
        c10::DeviceGuard dev(Q.device());
        at::AutoDispatchBelowADInplaceOrView guard;
        Tensor O = empty({d.B, d.H, 1, d.d}, *out, Q), M = empty({d.B, d.H, 1}, at::kFloat, Q), L = empty({d.B, d.H, 1}, at::kFloat, Q);
        const int64_t slots = (int64_t)d.B * d.H * d.n_splits;
        const Tensor part = whole ? Tensor() : empty({slots * d.d + 2 * padded(slots)}, at::kFloat, Q);
        const void *q = Q.data_ptr(), *k = K.data_ptr(), *v = V.data_ptr();
        const float *w = Wf.const_data_ptr<float>();
        float *m = M.mutable_data_ptr<float>(), *l = L.mutable_data_ptr<float>();
        void *s = stream_of(Q);
        if (whole) {
            check(api.convattn_decode_whole(&d, q, k, v, w, batch_stride(K), head_stride(K), O.data_ptr(), m, l, s), what);
        } else {
            float *op = part.mutable_data_ptr<float>(), *mp = op + slots * d.d, *lp = mp + padded(slots);
            check(api.convattn_decode_strided(&d, q, k, v, w, batch_stride(K), head_stride(K), op, mp, lp, s), what);
            check(api.convattn_decode_combine(&d, op, mp, lp, O.data_ptr(), m, l, s), what);
        }
        return Decoded{O, M, L, Tensor(), Tensor(), Tensor()};
    }
    if (k_splits == 0) d.n_splits = api.convattn_decode_splits(d.B, d.H, d.Nk, 0, d.d);
    return run_decode(d, Q, *out, "conv_attn.forward_inference", [&](float *o, float *m, float *l, void *s) {
        return api.convattn_decode_strided(&d, Q.data_ptr(), K.data_ptr(), V.data_ptr(), Wf.const_data_ptr<float>(), batch_stride(K),
                                           head_stride(K), o, m, l, s);
    });
}

// Shared KV heads, dense rows (no table) or pages; checks beyond these stay with the Python op
std::optional<Decoded> decode_kv(const Tensor &Q, const Tensor &K, const Tensor &V, const std::optional<Tensor> &table,
                                 const std::optional<Tensor> &lens, int64_t Nk, const Tensor &W, int64_t k_splits, double scale, bool causal,
                                 const py::object &out_dtype, const std::string &what) {
    const auto out = out_type(out_dtype);
    if (!out || watched() || !plain(Q) || !plain(K) || !plain(V) || Q.dim() != 4 || K.dim() != 4 || K.sizes() != V.sizes() ||
        K.strides() != V.strides() || !Q.is_contiguous() || Q.scalar_type() != at::kBFloat16 || K.scalar_type() != at::kBFloat16 ||
        V.scalar_type() != at::kBFloat16 || K.size(3) != Q.size(3) || Q.size(1) % K.size(1) != 0 || Q.size(2) > 16 || k_splits < 1 ||
        k_splits > 1024 || k_splits > Nk || W.dim() != 3 || K.device() != Q.device() || V.device() != Q.device())
        return std::nullopt;
    if (lens && (!plain(*lens) || lens->scalar_type() != at::kInt || lens->dim() != 1 || lens->size(0) != Q.size(0) || !lens->is_contiguous()))
        return std::nullopt;
    convattn_kv_layout lay{};
    lay.H_kv = (int)K.size(1);
    lay.seq_lens = lens ? lens->const_data_ptr<int>() : nullptr;
    if (table) {
        if (!plain(*table) || table->scalar_type() != at::kInt || table->dim() != 2 || table->size(0) != Q.size(0) ||
            !table->is_contiguous() || !K.is_contiguous() || table->size(1) * K.size(2) < Nk)
            return std::nullopt;
        lay.page_size = (int)K.size(2);
        lay.head_stride = K.size(2) * K.size(3);
        lay.page_stride = K.size(1) * lay.head_stride;
        lay.block_table = table->const_data_ptr<int>();
        lay.table_stride = (int)table->size(1);
    } else {
        if (K.size(0) != Q.size(0) || K.size(2) != Nk || !cache_rows(K)) return std::nullopt;
        lay.batch_stride = batch_stride(K);
        lay.head_stride = head_stride(K);
    }
    const Tensor Wf = window(W, Q.size(1), W.size(1) - 1, (W.size(2) - 1) / 2, Q);
    if (!Wf.defined()) return std::nullopt;
    convattn_desc d = window_desc(Q, Nk, Wf, scale, causal, *out == at::kFloat ? CONVATTN_F32 : CONVATTN_BF16);
    d.n_splits = (int)k_splits;
    return run_decode(d, Q, *out, what.c_str(), [&](float *o, float *m, float *l, void *s) {
        return api.convattn_decode_kv(&d, Q.data_ptr(), K.data_ptr(), V.data_ptr(), &lay, Wf.const_data_ptr<float>(), o, m, l, s);
    });
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
    m.def("init", &init);
    m.def("set_slow_backward", [](const std::string &which, py::object fn) {
        (which == "window" ? window_slow_backward : mix_slow_backward) = new py::object(std::move(fn));
    });
    m.def("window_attention", &window_attention);
    m.def("mix_attention", &mix_attention);
    m.def("decode_dense", &decode_dense);
    m.def("decode_kv", &decode_kv);
}
