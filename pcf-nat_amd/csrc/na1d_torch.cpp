// The attention operators' autograd nodes for torch in C++: what fused.py, dense.py and nattn.py do per call, without the
// interpreter.  A windowed layer's forward and backward at a training batch are 45 us of kernels; the same host path in
// Python took 115 us (allocations, context managers, ctypes, and the engine's thread waiting for the interpreter lock).
//
// Every function here returns nothing (None) for calls it does not take as they are - other devices, types, layouts,
// tensor subclasses, transforms, tracers, forward-mode gradients - and for those that the library refuses (the kernels are
// launched before a node is built).  The Python implementation then serves or refuses them as before.
#include <torch/extension.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/jit/frontend/tracer.h>

#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPGraphsC10Utils.h>

#include "na1d.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;
using MaybeTensor = std::optional<Tensor>;

PyObject *error_class = PyExc_RuntimeError;             // the package's exception, which lives as long as this module

// In a backward, on a thread of torch's: its engine carries a Python error to the caller.
void check(int status, const char *name) {
    if (status == NA1D_OK) return;
    const pybind11::gil_scoped_acquire gil;
    PyErr_Format(error_class, "%s failed: %s (status %d)", name, na1d_status_string(status), status);
    python_error error;
    error.persist();
    throw error;
}
void *stream_of(const Tensor &t) { return c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(t.device().index()).stream(); }
void *ptr(const Tensor &t) { return t.defined() ? t.data_ptr() : nullptr; }
int tag(const Tensor &t) { return t.scalar_type() == at::kBFloat16 ? NA1D_BF16 : NA1D_FP16; }

// A plain GPU tensor that nothing but autograd looks at.
bool plain(const Tensor &t) {
    const auto keys = t.key_set();
    return t.defined() && t.is_cuda() && t.layout() == at::kStrided && !t.is_conj() && !t.is_neg() &&
           !keys.has_any(c10::DispatchKeySet({c10::DispatchKey::Python, c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper,
                                              c10::DispatchKey::Functionalize, c10::DispatchKey::Batched, c10::DispatchKey::FuncTorchVmapMode})) &&
           !t._fw_grad(0).defined();
}
bool plain_call() {
    const auto tls = c10::impl::tls_local_dispatch_key_set().included_;
    return !torch::jit::tracer::isTracing() && !c10::impl::dispatch_mode_enabled() &&
           !tls.has_any(c10::DispatchKeySet({c10::DispatchKey::FuncTorchDynamicLayerFrontMode, c10::DispatchKey::FuncTorchDynamicLayerBackMode,
                                             c10::DispatchKey::FuncTorchVmapMode, c10::DispatchKey::Functionalize, c10::DispatchKey::Python}));
}
bool half_type(const Tensor &t) { return t.scalar_type() == at::kBFloat16 || t.scalar_type() == at::kHalf; }
// [B, T, C] operands of one kind.
bool same_operands(const Tensor &q, const Tensor &k, const Tensor &v) {
    for (const Tensor &t : {q, k, v})
        if (!plain(t) || t.dim() != 3 || !t.is_contiguous() || t.scalar_type() != q.scalar_type() || t.sizes() != q.sizes() || t.device() != q.device())
            return false;
    return half_type(q) && q.numel() > 0;
}
struct Dropout {
    double p;
    uint64_t seed;
};

// ------------------------------------------------------------------------------------------------ the fused operator
struct Geometry {
    int64_t N, H, T, C, W, left, dilation;
    double scale;
    Dropout drop;
    bool in_place;                                    // q, k, v inside a projection's output [N, T, 3, H, C]
};
struct Strides {
    int64_t in[3], out[3];
};
Strides strides_of(const Geometry &g) {
    if (g.in_place) return Strides{{g.T * 3 * g.H * g.C, g.C, 3 * g.H * g.C}, {g.T * g.H * g.C, g.C, g.H * g.C}};
    return Strides{{g.H * g.T * g.C, g.T * g.C, g.C}, {g.H * g.T * g.C, g.T * g.C, g.C}};
}
bool capturing() { return c10::hip::currentStreamCaptureStatusMayInitCtx() != c10::hip::CaptureStatus::None; }

int forward_kernel(const Geometry &g, const Tensor &out, const Tensor &lse, const Tensor &clear, const void *q, const void *k, const void *v, const Tensor &rpb, const Tensor &t_valid,
                   int dtype, void *stream) {
    const float *bias = (const float *)ptr(rpb);
    const int32_t *valid = (const int32_t *)ptr(t_valid);
    if (clear.defined()) {
        const Strides s = strides_of(g);
        return na1d_fused_forward_clear(ptr(out), (float *)ptr(lse), (float *)ptr(clear), q, k, v, bias, valid, g.N, g.H, g.T, g.C, g.W, g.left, g.dilation, (float)g.scale,
                                        dtype, s.in, s.out, (float)g.drop.p, g.drop.seed, stream);
    }
    if (g.dilation == 1 && !g.in_place) {
        if (g.drop.p > 0)
            return na1d_fused_forward_dropout(ptr(out), (float *)ptr(lse), q, k, v, bias, valid, g.N * g.H, g.H, g.T, g.C, g.W, g.left, (float)g.scale, dtype,
                                              (float)g.drop.p, g.drop.seed, stream);
        return na1d_fused_forward(ptr(out), (float *)ptr(lse), q, k, v, bias, valid, g.N * g.H, g.H, g.T, g.C, g.W, g.left, (float)g.scale, dtype, stream);
    }
    const Strides s = strides_of(g);
    return na1d_fused_forward_dilated(ptr(out), (float *)ptr(lse), q, k, v, bias, valid, g.N, g.H, g.T, g.C, g.W, g.left, g.dilation, (float)g.scale, dtype, s.in, s.out,
                                      (float)g.drop.p, g.drop.seed, stream);
}
int backward_kernel(const Geometry &g, void *dq, void *dk, void *dv, const Tensor &drpb, const void *q, const void *k, const void *v, const Tensor &out,
                    const Tensor &dout, const Tensor &lse, const Tensor &rpb, const Tensor &t_valid, int dtype, void *stream) {
    const float *bias = (const float *)ptr(rpb);
    const int32_t *valid = (const int32_t *)ptr(t_valid);
    if (g.dilation == 1 && !g.in_place) {
        if (g.drop.p > 0)
            return na1d_fused_backward_dropout(dq, dk, dv, (float *)ptr(drpb), q, k, v, ptr(out), ptr(dout), (const float *)ptr(lse), bias, valid, g.N * g.H, g.H, g.T,
                                               g.C, g.W, g.left, (float)g.scale, dtype, (float)g.drop.p, g.drop.seed, nullptr, 0, stream);
        return na1d_fused_backward(dq, dk, dv, (float *)ptr(drpb), q, k, v, ptr(out), ptr(dout), (const float *)ptr(lse), bias, valid, g.N * g.H, g.H, g.T, g.C, g.W,
                                   g.left, (float)g.scale, dtype, nullptr, 0, stream);
    }
    const Strides s = strides_of(g);
    return na1d_fused_backward_dilated(dq, dk, dv, (float *)ptr(drpb), q, k, v, ptr(dout), (const float *)ptr(lse), bias, valid, g.N, g.H, g.T, g.C, g.W, g.left,
                                       g.dilation, (float)g.scale, dtype, s.in, s.out, (float)g.drop.p, g.drop.seed, nullptr, 0, stream);
}
void remember(AutogradContext *ctx, const Geometry &g, const MaybeTensor &rpb, const Tensor &cleared) {
    ctx->saved_data["geometry"] = std::vector<int64_t>{g.N, g.H, g.T, g.C, g.W, g.left, g.dilation, (int64_t)g.drop.seed, g.in_place};
    ctx->saved_data["scale"] = g.scale;
    ctx->saved_data["p"] = g.drop.p;
    ctx->saved_data["bias"] = rpb && rpb->requires_grad();
    ctx->saved_data["bias_shape"] = rpb ? rpb->sizes().vec() : std::vector<int64_t>{};
    if (cleared.defined()) ctx->saved_data["cleared"] = cleared;
}
Geometry recall(AutogradContext *ctx) {
    const auto v = ctx->saved_data["geometry"].toIntVector();
    return Geometry{v[0], v[1], v[2], v[3], v[4], v[5], v[6], ctx->saved_data["scale"].toDouble(), {ctx->saved_data["p"].toDouble(), (uint64_t)v[7]}, v[8] != 0};
}
// The gradient of the bias, all zeros, which the backward's kernel adds to; undefined where none is asked for.  The forward's kernel has
// cleared it on the way, for the first backward of a node; any further one, on whatever thread, clears its own.  (The tensor's version
// says that it is taken, also to a copy of the node's data as compiled autograd makes them.)  A graph may hold the forward and not the
// backward, or replay them unevenly, so under capture every backward clears its own too.
Tensor begin_bias_gradient(AutogradContext *ctx, const Tensor &like) {
    if (!ctx->saved_data["bias"].toBool()) return Tensor();
    const auto held = ctx->saved_data.find("cleared");
    if (held != ctx->saved_data.end() && !capturing()) {
        static std::mutex mutex;
        const std::lock_guard<std::mutex> lock(mutex);
        if (held->second.isTensor()) {
            Tensor t = std::move(held->second).toTensor();
            held->second = c10::IValue();
            if (t.defined() && t._version() == 0) {
                t.unsafeGetTensorImpl()->bump_version();
                return t;
            }
        }
    }
    return at::zeros(ctx->saved_data["bias_shape"].toIntVector(), like.options().dtype(at::kFloat));
}
Tensor bias_of(const MaybeTensor &rpb, const Geometry &g, bool node) {
    if (rpb && !node && rpb->scalar_type() == at::kFloat && rpb->is_contiguous()) return *rpb;
    return rpb ? rpb->detach().reshape({g.H, g.W}).to(at::kFloat).contiguous() : Tensor();
}
Tensor lengths_of(const MaybeTensor &t_valid, const Tensor &like) { return t_valid ? t_valid->to(like.device(), at::kInt).contiguous() : Tensor(); }

// A forward whose kernels are launched: what its node is built around.
struct Done {
    Tensor out, lse, bias, valid, cleared;
};
Tensor to_be_cleared(const MaybeTensor &rpb, const Tensor &like, bool node) {
    return node && rpb && rpb->requires_grad() && !capturing() ? at::empty(rpb->sizes(), like.options().dtype(at::kFloat)) : Tensor();
}

struct Fused : torch::autograd::Function<Fused> {
    static Tensor forward(AutogradContext *ctx, const Tensor &q, const Tensor &k, const Tensor &v, const MaybeTensor &rpb, const MaybeTensor &,
                          const Geometry &g, const Done &done) {
        ctx->save_for_backward({q, k, v, done.out, done.bias, done.valid, done.lse});
        remember(ctx, g, rpb, done.cleared);
        return done.out;
    }
    static variable_list backward(AutogradContext *ctx, const variable_list &grads) {
        const variable_list s = ctx->get_saved_variables();
        const Geometry g = recall(ctx);
        const Tensor &q = s[0];
        const c10::DeviceGuard guard(q.device());
        const Tensor dout = grads[0].contiguous(), dq = at::empty_like(q), dk = at::empty_like(q), dv = at::empty_like(q);
        const Tensor drpb = begin_bias_gradient(ctx, q);
        check(backward_kernel(g, ptr(dq), ptr(dk), ptr(dv), drpb, ptr(q), ptr(s[1]), ptr(s[2]), s[3], dout, s[6], s[4], s[5], tag(q), stream_of(q)),
              "na1d_fused_backward");
        return {dq, dk, dv, drpb, Tensor(), Tensor(), Tensor()};
    }
};
struct FusedQKV : torch::autograd::Function<FusedQKV> {
    static Tensor forward(AutogradContext *ctx, const Tensor &qkv, const MaybeTensor &rpb, const MaybeTensor &, const Geometry &g, const Done &done) {
        ctx->save_for_backward({qkv, done.bias, done.valid, done.lse});
        remember(ctx, g, rpb, done.cleared);
        return done.out;
    }
    static variable_list backward(AutogradContext *ctx, const variable_list &grads) {
        const variable_list s = ctx->get_saved_variables();
        const Geometry g = recall(ctx);
        const Tensor &qkv = s[0];
        const c10::DeviceGuard guard(qkv.device());
        const Tensor dout = grads[0].contiguous(), dqkv = at::empty_like(qkv);
        const Tensor drpb = begin_bias_gradient(ctx, qkv);
        const int64_t step = 2 * g.H * g.C;
        char *dq = (char *)ptr(dqkv);
        const char *q = (const char *)ptr(qkv);
        check(backward_kernel(g, dq, dq + step, dq + 2 * step, drpb, q, q + step, q + 2 * step, Tensor(), dout, s[3], s[1], s[2], tag(qkv), stream_of(qkv)),
              "na1d_fused_backward");
        return {dqkv, drpb, Tensor(), Tensor(), Tensor()};
    }
};
// Whether bias and lengths are what the Python path takes without complaint, and the sizes what the one-launch kernels cover.
bool covered(const Geometry &g, const Tensor &like, const MaybeTensor &rpb, const MaybeTensor &t_valid) {
    if (g.H < 1 || g.W < 1 || g.W > NA1D_MAX_WINDOW || g.left < 0 || g.left >= g.W || g.dilation < 1 || g.C % 8 || g.C > 128 || !(g.drop.p >= 0 && g.drop.p < 1))
        return false;
    if (rpb && (!plain(*rpb) || rpb->device() != like.device() || rpb->numel() != g.H * g.W || !rpb->is_floating_point())) return false;
    if (t_valid && (!plain(*t_valid) || t_valid->numel() != g.N || t_valid->device() != like.device())) return false;
    return na1d_fused_backward_dilated_workspace_bytes(g.N, g.H, g.T, g.C, g.W, g.left, g.dilation, tag(like)) > 0;
}

bool needs_grad(std::initializer_list<Tensor> operands, const MaybeTensor &rpb) {
    if (!at::GradMode::is_enabled()) return false;
    for (const Tensor &t : operands)
        if (t.requires_grad()) return true;
    return rpb && rpb->requires_grad();
}

MaybeTensor fused(const Tensor &q, const Tensor &k, const Tensor &v, const MaybeTensor &rpb, const MaybeTensor &t_valid, int64_t H, int64_t W, int64_t left,
                  double scale, int64_t dilation, double p, uint64_t seed) {
    if (!plain_call() || !same_operands(q, k, v) || H < 1 || q.size(0) % H) return std::nullopt;
    const Geometry g{q.size(0) / H, H, q.size(1), q.size(2), W, left, dilation, scale, {p, seed}, false};
    if (!covered(g, q, rpb, t_valid)) return std::nullopt;
    const c10::DeviceGuard guard(q.device());
    const bool node = needs_grad({q, k, v}, rpb);      // otherwise no log-sum-exp either
    const Done done{at::empty_like(q), node ? at::empty({g.N * g.H, g.T}, q.options().dtype(at::kFloat)) : Tensor(), bias_of(rpb, g, node),
                    lengths_of(t_valid, q), to_be_cleared(rpb, q, node)};
    if (forward_kernel(g, done.out, done.lse, done.cleared, ptr(q), ptr(k), ptr(v), done.bias, done.valid, tag(q), stream_of(q)) != NA1D_OK) return std::nullopt;
    return node ? Fused::apply(q, k, v, rpb, t_valid, g, done) : done.out;
}
MaybeTensor fused_qkv(const Tensor &qkv, const MaybeTensor &rpb, const MaybeTensor &t_valid, int64_t W, int64_t left, double scale, int64_t dilation, double p,
                      uint64_t seed) {
    if (!plain_call() || !plain(qkv) || qkv.dim() != 5 || qkv.size(2) != 3 || !qkv.is_contiguous() || !half_type(qkv) || !qkv.numel()) return std::nullopt;
    const Geometry g{qkv.size(0), qkv.size(3), qkv.size(1), qkv.size(4), W, left, dilation, scale, {p, seed}, true};
    if (!covered(g, qkv, rpb, t_valid)) return std::nullopt;
    const c10::DeviceGuard guard(qkv.device());
    const bool node = needs_grad({qkv}, rpb);
    const Done done{at::empty({g.N, g.T, g.H * g.C}, qkv.options()), node ? at::empty({g.N * g.H, g.T}, qkv.options().dtype(at::kFloat)) : Tensor(),
                    bias_of(rpb, g, node), lengths_of(t_valid, qkv), to_be_cleared(rpb, qkv, node)};
    const char *q = (const char *)ptr(qkv);
    const int64_t step = 2 * g.H * g.C;
    if (forward_kernel(g, done.out, done.lse, done.cleared, q, q + step, q + 2 * step, done.bias, done.valid, tag(qkv), stream_of(qkv)) != NA1D_OK) return std::nullopt;
    return node ? FusedQKV::apply(qkv, rpb, t_valid, g, done) : done.out;
}

// ------------------------------------------------------------------------------------------------ dense attention
struct Dense : torch::autograd::Function<Dense> {
    static Tensor forward(AutogradContext *ctx, const Tensor &q, const Tensor &k, const Tensor &v, int64_t H, double scale, double p, uint64_t seed,
                          const Done &done) {
        ctx->save_for_backward({q, k, v, done.out, done.lse, done.valid});
        ctx->saved_data["heads"] = H;
        ctx->saved_data["scale"] = scale;
        ctx->saved_data["p"] = p;
        ctx->saved_data["seed"] = (int64_t)seed;
        return done.out;
    }
    static variable_list backward(AutogradContext *ctx, const variable_list &grads) {
        const variable_list s = ctx->get_saved_variables();
        const Tensor &q = s[0];
        const c10::DeviceGuard guard(q.device());
        const int64_t B = q.size(0), T = q.size(1), C = q.size(2), H = ctx->saved_data["heads"].toInt();
        const Tensor dout = grads[0].contiguous(), dq = at::empty_like(q), dk = at::empty_like(q), dv = at::empty_like(q);
        const int64_t nbytes = na1d_global_backward_workspace_bytes(B, H, T, C, tag(q));
        check((int)std::min<int64_t>(nbytes, 0), "na1d_global_backward_workspace_bytes");
        const Tensor ws = at::empty({nbytes}, q.options().dtype(at::kByte));
        check(na1d_global_backward(ptr(dq), ptr(dk), ptr(dv), ptr(q), ptr(s[1]), ptr(s[2]), ptr(s[3]), ptr(dout), (const float *)ptr(s[4]), (const int32_t *)ptr(s[5]),
                                   B, H, T, C, (float)ctx->saved_data["scale"].toDouble(), tag(q), (float)ctx->saved_data["p"].toDouble(),
                                   (uint64_t)ctx->saved_data["seed"].toInt(), ptr(ws), nbytes, stream_of(q)),
              "na1d_global_backward");
        return {dq, dk, dv, Tensor(), Tensor(), Tensor(), Tensor(), Tensor()};
    }
};
MaybeTensor dense(const Tensor &q, const Tensor &k, const Tensor &v, const MaybeTensor &t_valid, int64_t H, double scale, double p, uint64_t seed) {
    if (!plain_call() || !same_operands(q, k, v) || H < 1 || q.size(0) % H || q.size(2) % 8 || q.size(2) > 128) return std::nullopt;
    if (t_valid && (!plain(*t_valid) || t_valid->scalar_type() != at::kInt || t_valid->numel() != q.size(0) / H || !t_valid->is_contiguous() ||
                    t_valid->device() != q.device()))
        return std::nullopt;
    const c10::DeviceGuard guard(q.device());
    const Done done{at::empty_like(q), at::empty({q.size(0), q.size(1)}, q.options().dtype(at::kFloat)), Tensor(), t_valid ? *t_valid : Tensor()};
    if (na1d_global_forward(ptr(done.out), (float *)ptr(done.lse), ptr(q), ptr(k), ptr(v), (const int32_t *)ptr(done.valid), q.size(0), H, q.size(1), q.size(2),
                            (float)scale, tag(q), (float)p, seed, stream_of(q)) != NA1D_OK)
        return std::nullopt;
    return Dense::apply(q, k, v, H, scale, p, seed, done);
}

// ------------------------------------------------------------------------------------------------ the two-call operator
using Band = int(void *, const void *, const void *, int64_t, int64_t, int64_t, int64_t, int64_t, int, void *);
int band(Band *f, const Tensor &out, const Tensor &a, const Tensor &b, const Tensor &like, int64_t W, int64_t left) {
    return f(ptr(out), ptr(a), ptr(b), like.size(0), like.size(1), like.size(2), W, left, tag(like), stream_of(like));
}
struct QK : torch::autograd::Function<QK> {
    static Tensor forward(AutogradContext *ctx, const Tensor &q, const Tensor &k, int64_t W, int64_t left, const Done &done) {
        ctx->save_for_backward({q, k});
        ctx->saved_data["W"] = W;
        ctx->saved_data["left"] = left;
        return done.out;
    }
    static variable_list backward(AutogradContext *ctx, const variable_list &grads) {
        const variable_list s = ctx->get_saved_variables();
        const int64_t W = ctx->saved_data["W"].toInt(), left = ctx->saved_data["left"].toInt();
        const c10::DeviceGuard guard(s[0].device());
        const Tensor g = grads[0].contiguous(), dq = at::empty_like(s[0]), dk = at::empty_like(s[0]);
        check(band(na1d_q_backward, dq, g, s[1], s[0], W, left), "na1d_q_backward");
        check(band(na1d_k_backward, dk, g, s[0], s[0], W, left), "na1d_k_backward");
        return {dq, dk, Tensor(), Tensor(), Tensor()};
    }
};
struct AV : torch::autograd::Function<AV> {
    static Tensor forward(AutogradContext *ctx, const Tensor &attn, const Tensor &v, int64_t W, int64_t left, const Done &done) {
        ctx->save_for_backward({attn, v});
        ctx->saved_data["W"] = W;
        ctx->saved_data["left"] = left;
        return done.out;
    }
    static variable_list backward(AutogradContext *ctx, const variable_list &grads) {
        const variable_list s = ctx->get_saved_variables();
        const int64_t W = ctx->saved_data["W"].toInt(), left = ctx->saved_data["left"].toInt();
        const c10::DeviceGuard guard(s[1].device());
        const Tensor g = grads[0].contiguous(), dattn = at::empty_like(s[0]), dv = at::empty_like(s[1]);
        check(band(na1d_a_backward, dattn, g, s[1], s[1], W, left), "na1d_a_backward");
        check(band(na1d_v_backward, dv, s[0], g, s[1], W, left), "na1d_v_backward");
        return {dattn, dv, Tensor(), Tensor(), Tensor()};
    }
};
bool band_window(int64_t W, int64_t left) { return W >= 1 && W <= NA1D_MAX_WINDOW && left >= 0 && left < W; }
MaybeTensor qk(const Tensor &q, const Tensor &k, int64_t W, int64_t left) {
    if (!plain_call() || !same_operands(q, k, k) || q.size(2) % 8 || !band_window(W, left)) return std::nullopt;
    const c10::DeviceGuard guard(q.device());
    const Done done{at::empty({q.size(0), q.size(1), W}, q.options().dtype(at::kFloat)), Tensor(), Tensor(), Tensor()};
    if (band(na1d_qk_forward, done.out, q, k, q, W, left) != NA1D_OK) return std::nullopt;
    return QK::apply(q, k, W, left, done);
}
MaybeTensor av(const Tensor &attn, const Tensor &v, int64_t W, int64_t left) {
    if (!plain_call() || !same_operands(v, v, v) || v.size(2) % 8 || !band_window(W, left)) return std::nullopt;
    if (!plain(attn) || attn.scalar_type() != at::kFloat || !attn.is_contiguous() || attn.device() != v.device() || attn.dim() != 3 || attn.size(0) != v.size(0) ||
        attn.size(1) != v.size(1) || attn.size(2) != W)
        return std::nullopt;
    const c10::DeviceGuard guard(v.device());
    const Done done{at::empty_like(v), Tensor(), Tensor(), Tensor()};
    if (band(na1d_av_forward, done.out, attn, v, v, W, left) != NA1D_OK) return std::nullopt;
    return AV::apply(attn, v, W, left, done);
}

// ------------------------------------------------------------------------------------------------ an encoder layer in training
// What train.py's node does between its checks and its bookkeeping.  A layer is some two dozen allocations and a dozen
// launches each way: through the interpreter they took longer than the kernels of a small batch.
void refuse(int64_t status, const char *name) {             // called by Python
    if (status >= 0) return;
    PyErr_Format(error_class, "%s failed: %s (status %d)", name, na1d_status_string((int)status), (int)status);
    throw pybind11::error_already_set();
}
// (dtype, dim, hidden, heads, window, left, dilation, groups, ordered, scale, late), as the struct has them
na1d_train_layer layer_of(const pybind11::tuple &geom) {
    na1d_train_layer l{};
    int32_t *const numbers[] = {&l.dtype, &l.dim, &l.hidden, &l.heads, &l.window, &l.left, &l.dilation, &l.groups, &l.ordered};
    for (int i = 0; i < 9; ++i) *numbers[i] = geom[i].cast<int32_t>();
    l.scale = geom[9].cast<float>();
    l.late = geom[10].cast<int32_t>();
    return l;
}
const float *floats(const Tensor &t) { return static_cast<const float *>(t.data_ptr()); }
const float *floats(const MaybeTensor &t) { return t ? floats(*t) : nullptr; }

// params: rpb or linear_pos' weight, weight and bias of the norms, of qkv, proj, fc1, fc2; state: running mean, running
// variance and batches of the norms; numbers: their momentum and eps.  Returns the output and what a backward reads.
std::pair<Tensor, Tensor> train_forward(const Tensor &x, const MaybeTensor &by_channel, const pybind11::tuple &geom, const std::vector<Tensor> &state,
                                        const std::vector<double> &numbers, const MaybeTensor &scale_attn, const MaybeTensor &scale_mlp, const MaybeTensor &pos,
                                        const std::vector<Tensor> &params) {
    na1d_train_layer l = layer_of(geom);
    const int64_t N = x.size(0), T = x.size(1), dim = x.size(2);
    for (int i = 0; i < 2; ++i) {
        l.norm[i].weight = floats(params[1 + 2 * i]);
        l.norm[i].bias = floats(params[2 + 2 * i]);
        l.norm[i].batches = static_cast<int64_t *>(state[3 * i + 2].data_ptr());
        l.norm[i].eps = (float)numbers[2 * i + 1];
    }
    for (int i = 0; i < 4; ++i) l.w[i] = floats(params[5 + 2 * i]), l.b[i] = floats(params[6 + 2 * i]);
    (pos ? l.w[4] : l.rpb) = floats(params[0]);
    l.pos = pos ? pos->data_ptr() : nullptr;
    l.scale_attn = floats(scale_attn), l.scale_mlp = floats(scale_mlp);
    const c10::DeviceGuard guard(x.device());
    void *const stream = stream_of(x);
    const int64_t saved_bytes = na1d_train_layer_saved_bytes(&l, N, T), ws_bytes = na1d_train_layer_workspace_bytes(&l, N, T, 0);
    refuse(std::min(saved_bytes, ws_bytes), "na1d_train_layer_saved_bytes");
    const auto bytes = x.options().dtype(at::kByte);
    const Tensor out = at::empty_like(x), saved = at::empty({saved_bytes}, bytes), ws = at::empty({ws_bytes}, bytes);
    Tensor of = by_channel ? *by_channel : at::empty({N, dim, T}, x.options());
    if (!by_channel) refuse(na1d_train_to_channels(&l, of.data_ptr(), x.data_ptr(), N, T, stream), "na1d_train_to_channels");
    const Tensor x1 = at::empty({N, dim, T}, x.options());
    std::tuple<Tensor, Tensor> stats[2];                    // until the kernels that read them are launched
    for (int part = 0; part < 2; ++part) {
        stats[part] = at::batch_norm_update_stats(part ? x1 : of, state[3 * part], state[3 * part + 1], numbers[2 * part]);
        l.norm[part].batch_mean = floats(std::get<0>(stats[part])), l.norm[part].batch_var = floats(std::get<1>(stats[part]));
        refuse(na1d_train_layer_forward(&l, part, (part ? out : x1).data_ptr(), x.data_ptr(), saved.data_ptr(), saved_bytes, ws.data_ptr(), ws_bytes, N, T, stream),
               "na1d_train_layer_forward");
    }
    for (const Tensor &t : state) t.unsafeGetTensorImpl()->bump_version();
    return {out, saved};
}
// The gradients of x and of the parameters, in train_forward's order.
std::vector<Tensor> train_backward(const Tensor &given, const Tensor &x, const Tensor &saved, const pybind11::tuple &geom, const MaybeTensor &rpb, const Tensor &n1w,
                                   const Tensor &n2w, const MaybeTensor &scale_attn, const MaybeTensor &scale_mlp, const MaybeTensor &pos,
                                   const std::vector<std::vector<int64_t>> &shapes) {
    na1d_train_layer l = layer_of(geom);
    const int64_t N = x.size(0), T = x.size(1);
    const c10::DeviceGuard guard(x.device());
    Tensor dout = given.contiguous();
    if ((uintptr_t)dout.data_ptr() % 16) dout = dout.clone();
    const auto fp32 = x.options().dtype(at::kFloat);
    std::vector<Tensor> grads{at::empty_like(x), pos ? at::empty(shapes[0], fp32) : at::zeros(shapes[0], fp32)};      // the scores' bias gradient is added to
    for (size_t i = 1; i < shapes.size(); ++i) grads.push_back(at::empty(shapes[i], fp32));
    auto grad = [&](int i) { return static_cast<float *>(grads[1 + i].data_ptr()); };
    for (int i = 0; i < 4; ++i) l.dw[i] = grad(5 + 2 * i), l.db[i] = grad(6 + 2 * i);
    (pos ? l.dw[4] : l.drpb) = grad(0);
    l.norm[0].weight = floats(n1w), l.norm[1].weight = floats(n2w);
    for (int i = 0; i < 2; ++i) l.norm[i].dweight = grad(1 + 2 * i), l.norm[i].dbias = grad(2 + 2 * i);
    l.rpb = floats(rpb), l.pos = pos ? pos->data_ptr() : nullptr;
    l.scale_attn = floats(scale_attn), l.scale_mlp = floats(scale_mlp);
    const int64_t ws_bytes = na1d_train_layer_workspace_bytes(&l, N, T, 1);
    refuse(ws_bytes, "na1d_train_layer_workspace_bytes");
    const Tensor ws = at::empty({ws_bytes}, x.options().dtype(at::kByte));
    refuse(na1d_train_layer_backward(&l, grads[0].data_ptr(), dout.data_ptr(), x.data_ptr(), saved.data_ptr(), saved.numel(), ws.data_ptr(), ws_bytes, N, T, stream_of(x)),
           "na1d_train_layer_backward");
    return grads;
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
    m.def("raise_as", [](pybind11::object c) { error_class = c.inc_ref().ptr(); });
    m.def("fused", &fused);
    m.def("fused_qkv", &fused_qkv);
    m.def("dense", &dense);
    m.def("qk", &qk);
    m.def("av", &av);
    m.def("train_forward", &train_forward);
    m.def("train_backward", &train_backward);
}
